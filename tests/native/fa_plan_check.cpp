// The score route of FLASH_ATTN_EXT on the host: where fa_score_tiles takes a work list to the matrix-core
// score kernel, every (item, 256-cell tile) has to appear once in the list's map, at the tile of its cells, and
// every index that the kernel forms from the map has to stay inside its item's scores and tile maxima. Prints
// what it saw; exit status 1 and the first failure otherwise.
#include "fa_plan.hpp"

#include <cstdio>
#include <cstdlib>

using namespace tsr;

static const char * check(const FaWork & w, uint32_t T, uint32_t n_head, uint32_t n_map, uint32_t lo, const uint32_t * msum) {
    std::vector<uint32_t> list(fa_list_bytes(w.items.size(), T, n_map) / 4u);
    fa_pack_list(w, T, n_map, lo, msum, (uint8_t *)list.data());
    const uint32_t * map = list.data() + w.items.size() * (sizeof(FaItem) / 4u) + 2u * T, * hi = map + (size_t)n_map * T;
    std::vector<uint8_t> seen(w.n_tiles, 0);
    for (uint32_t at = 0; at < n_map; ++at)
        for (uint32_t t = 0; t < T; ++t) {
            const uint32_t idx = map[(size_t)at * T + t], cell0 = 16u * (lo / 16u + 16u * at);
            if (idx == 0xFFFFFFFFu) continue;
            if (idx >= w.items.size()) return "an item that there is not";
            const FaItem & it = w.items[idx];
            if (it.t != t || hi[t] != msum[9u + 4u * t]) return "another row's item or run end";
            const uint32_t c0 = 16u * it.u0, n16 = 16u * it.n;
            if (cell0 < c0 || cell0 >= c0 + n16) return "a tile outside its item";
            if ((cell0 - c0) % 256u != 0u) return "a tile that is not one of its item's";
            const uint32_t tile = it.tile0 + (cell0 - c0) / 256u;
            if (tile >= it.tile0 + it.ntiles || tile >= w.n_tiles) return "a tile maximum outside the item's";
            if (seen[tile]++) return "a tile twice";
            // the kernel's first and last score of the tile: head h, cells cell0 .. min(cell0 + 256, end) - 1
            const uint64_t last = std::min(cell0 + 256u, c0 + n16) - 1u - c0;
            const uint64_t s_hi = (uint64_t)it.s_off * n_head + (uint64_t)(n_head - 1u) * n16 + last;
            if (s_hi >= w.cells * n_head || 4u * s_hi >= (1ull << 32)) return "a score outside the array";
        }
    for (uint32_t k = 0; k < w.n_tiles; ++k)
        if (!seen[k]) return "a tile of an item that no workgroup scores";
    return nullptr;
}

// The scratch: no more than the other route's, and nothing that is alive together overlaps.
static const char * check_layout(const FaWork & w, uint32_t T, uint32_t n_head, uint32_t D, uint32_t n_map) {
    const size_t n = w.items.size(), K = (size_t)n_head * D;
    const FaLayout l = fa_layout(n, w.cells, w.n_tiles, T, n_head, D, false, n_map);
    if (l.bytes > fa_layout(n, w.cells, w.n_tiles, T, n_head, D, false, 0u).bytes) return "more scratch than the one-row route";
    struct Part { size_t at, bytes; };
    const Part S = { l.S, 4u * (size_t)w.cells * n_head }, Mp = { l.Mp, 4u * (size_t)w.n_tiles * n_head },
               LP = { l.LP, 16u * n * n_head }, OP = { l.OP, 16u * n * K }, items = { l.items, fa_list_bytes(n, T, 0u) },
               list = { l.items, (fa_list_bytes(n, T, n_map) + 15u) / 16u * 16u }, xq = { l.xq, T * K }, xd = { l.xd, T * K / 8u };
    auto apart = [&](std::vector<Part> p) {
        for (size_t i = 0; i < p.size(); ++i) {
            if (p[i].at % 256u != 0u || p[i].at + p[i].bytes > l.bytes) return false;
            for (size_t j = 0; j < i; ++j)
                if (p[i].at < p[j].at + p[j].bytes && p[j].at < p[i].at + p[i].bytes) return false;
        }
        return true;
    };
    std::vector<Part> scores = { S, Mp, list }, rest = { S, Mp, LP, OP, items };   // up to the scores; from P.V on
    if (n_map != 0u) scores.insert(scores.end(), { xq, xd });
    return apart(scores) && apart(rest) ? nullptr : "overlapping scratch";
}

// k_fa_pv has one wave per segment of the longest item: every channel of every item has to fit.
static const char * check_segments(const FaWork & w) {
    const uint32_t nw = fa_segments(w.max_groups);
    if (nw > kMaxSegments) return "more segments than waves of a workgroup";
    for (const FaItem & it : w.items)
        for (uint32_t c = 0; c < kC; ++c) {                       // as PvBlock counts them
            const uint32_t first = it.u0 + ((c + 4u - (it.u0 & 3u)) & 3u), end = it.u0 + it.n;
            const uint32_t nu = first < end ? (end - 1u - first) / 4u + 1u : 0u;
            if ((nu + 3u) / 4u > nw) return "a segment without a wave";
        }
    return nullptr;
}

int main() {
    size_t taken = 0, refused = 0, cut = 0, sparse = 0;
    for (uint32_t nkv = 1; nkv <= 64; ++nkv)
        for (uint32_t D : { 64u, 128u })
            for (uint32_t G : { 1u, 4u, 8u })
                for (uint32_t lo : { 0u, 37u, 4096u })
                    for (uint32_t hist : { 300u, 1500u, 2048u, 2100u, 3600u, 9300u })
                        for (uint32_t shape : { 9u, 20u, 23u, 33u, 62u, 256u, 1256u }) {
                            const uint32_t T = shape % 1000u;     // 1256: one row in four long, the others of 40 cells
                            const uint32_t E = nkv * D, n_head = nkv * G;
                            if (n_head * D > 32768u || G * E > 32768u || E / 64u > 511u) continue;   // not shapes of the library
                            std::vector<uint32_t> msum(8u + 4u * T, 0u);
                            msum[1] = T;
                            msum[2] = lo + hist + T;
                            for (uint32_t t = 0; t < T; ++t) {
                                msum[8u + 4u * t] = lo;
                                msum[9u + 4u * t] = lo + (shape > 1000u && t % 4u ? 40u : hist + 1u + t);
                            }
                            const uint32_t runs[1][2] = { { lo + hist, lo + hist + T } };
                            FaWork w;
                            if (fa_plan_rows(E, D, T, msum.data(), runs, 1u, false, w) != 0) return 2;
                            uint32_t first = 0;
                            const uint32_t n_map = fa_score_tiles(w, D, n_head, T, msum.data(), first);
                            bool aligned = true;                  // the chunk length of every row in whole tiles
                            for (uint32_t t = 0; t < T; ++t) {
                                const uint32_t n = (msum[9u + 4u * t] + 15u) / 16u - lo / 16u, ncg = ncg_of(E, D, n);
                                aligned = aligned && (ncg % 16u == 0u || n <= ncg);
                            }
                            uint64_t formed = 0;                  // cells of the tiles that a workgroup of 32 rows forms
                            for (uint32_t b = 0; b < T; b += 32u) {
                                uint32_t top = 0;
                                for (uint32_t t = b; t < std::min(b + 32u, T); ++t) top = std::max(top, (msum[9u + 4u * t] + 15u) / 16u - lo / 16u);
                                formed += 32u * 256u * (uint64_t)((top + 15u) / 16u);
                            }
                            const bool dense = 3u * w.cells >= 2u * formed;
                            const bool enough = w.cells * n_head * (D / 64u) >= (10ull << 20) && 4u * w.cells * n_head < (1ull << 31);
                            const char * bad = n_map ? check(w, T, n_head, n_map, first, msum.data()) : nullptr;
                            if (bad == nullptr) bad = check_layout(w, T, n_head, D, n_map);
                            if (bad == nullptr) bad = check_segments(w);
                            if (bad == nullptr && (n_map != 0u) != (aligned && enough && dense)) bad = "the route's rule";
                            if (bad != nullptr) {
                                printf("%s: %u of %u heads, D %u, %u rows behind %u cells from %u\n", bad, nkv, n_head, D, T, hist, lo);
                                return 1;
                            }
                            taken += n_map != 0u;
                            refused += n_map == 0u;
                            cut += enough && dense && !aligned;
                            sparse += enough && aligned && !dense;
                        }
    printf("%zu work lists on the matrix cores, %zu not, %zu of them for their chunk cuts, %zu as too sparse\n", taken, refused, cut, sparse);
    return taken != 0u && cut != 0u && sparse != 0u ? 0 : 3;
}
