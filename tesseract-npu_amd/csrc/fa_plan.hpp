// fa_plan.hpp -- the host planner of FLASH_ATTN_EXT: the chunks of every query row, the flat work list and the
// score route. Plain C++ without the HIP runtime, so that it is checked on the CPU.
#pragma once

#include <cstdint>
#include <cstring>

#include <algorithm>
#include <vector>

#include "fa_item.hpp"
#include "tsr_hip.h"

namespace tsr {

constexpr uint32_t kC = 4u, kPcap = 9344u;

struct Chunk {
    uint32_t u0, n, c_lo, c_hi, general;
};

// NCG = min(128, C floor(PCAP / (16 E / D)), max(4C, roundup_4C(ceil(n_total / 2))))
// (sw/sim/include/tsr_fa_plan.h:130-156).
inline uint32_t ncg_of(uint32_t E, uint32_t D, uint32_t n_total) {
    const uint64_t pc = (uint64_t)kC * (kPcap / (16u * (E / D)));
    const uint64_t half = ((uint64_t)n_total + 1u) / 2u, c4 = 4u * kC;
    const uint64_t m = half <= c4 ? c4 : (half + c4 - 1u) / c4 * c4;
    return (uint32_t)std::min<uint64_t>(std::min<uint64_t>(128u, pc), m);
}

// A fixed-capacity stand-in for std::vector in the planner of the entry point that allocates nothing:
// push_back past the capacity records an overflow instead of growing.
template <class T, size_t N>
struct FixedVec {
    T v[N];
    size_t n = 0;
    bool overflow = false;
    void clear() { n = 0; overflow = false; }
    void push_back(const T & x) {
        if (n < N) v[n++] = x;
        else overflow = true;
    }
    void assign(size_t k, const T & x) {
        if (k > N) { overflow = true; k = N; }
        n = k;
        for (size_t i = 0; i < k; ++i) v[i] = x;
    }
    size_t size() const { return n; }
    T & operator[](size_t i) { return v[i]; }
    const T & operator[](size_t i) const { return v[i]; }
    T * data() { return v; }
    const T * begin() const { return v; }
    const T * end() const { return v + n; }
};
template <class V> bool overflowed(const V &) { return false; }
template <class T, size_t N> bool overflowed(const FixedVec<T, N> & v) { return v.overflow; }

// The chunks of one query row in execution order (one-row tiles: rules 1, 2, 4, 7, 8 of the planner,
// sw/sim/include/tsr_fa_plan.h:16-42). Returns false for a malformed MSUM row.
template <class Out>
bool plan_row(uint32_t E, uint32_t D, const uint32_t * words, uint32_t q, const uint32_t (*new_runs)[2],
              uint32_t n_new, Out & out) {
    const uint32_t n_kv = words[2];
    const bool general = (words[3] & 1u) != 0u;
    struct Sub { uint32_t ulo, uhi; uint64_t lo, hi; } sub[2];
    uint32_t nsub = 0;
    if (general) {
        if (n_kv > 0u) sub[nsub++] = { 0u, (n_kv + 15u) / 16u, 0u, 0u };
    } else {
        const uint32_t * w = words + 8u + 4u * q;
        if (w[0] > w[1] || w[2] > w[3] || w[1] > n_kv || w[3] > n_kv) return false;
        if (w[1] > w[0] && w[3] > w[2] && !(w[1] <= w[2] || w[3] <= w[0])) return false;
        uint32_t r[2][2], nr = 0;
        if (w[1] > w[0]) { r[nr][0] = w[0]; r[nr][1] = w[1]; ++nr; }
        if (w[3] > w[2]) { r[nr][0] = w[2]; r[nr][1] = w[3]; ++nr; }
        if (nr == 2u && r[1][0] < r[0][0]) { std::swap(r[0][0], r[1][0]); std::swap(r[0][1], r[1][1]); }
        for (uint32_t k = 0; k < nr; ++k) sub[nsub++] = { r[k][0] / 16u, (r[k][1] + 15u) / 16u, r[k][0], r[k][1] };
    }
    if (nsub == 0u) {                                      // no visible cell: one empty chunk
        out.push_back({ 0u, 1u, 0u, 0u, 0u });
        return true;
    }
    uint32_t n_total = 0;
    for (uint32_t k = 0; k < nsub; ++k) n_total += sub[k].uhi - sub[k].ulo;
    const uint32_t ncg = ncg_of(E, D, n_total);
    if (ncg == 0u) return false;
    for (int pass = 0; pass < 2; ++pass)                   // chunks holding a new cell go last
        for (uint32_t k = 0; k < nsub; ++k)
            for (uint32_t a = sub[k].ulo; a < sub[k].uhi; a += ncg) {
                const uint32_t b = std::min(a + ncg, sub[k].uhi);
                bool has_new = false;
                for (uint32_t i = 0; i < n_new; ++i)
                    has_new |= new_runs[i][1] > new_runs[i][0] && (uint64_t)new_runs[i][0] < 16ull * b &&
                                (uint64_t)new_runs[i][1] > 16ull * a;
                if ((int)has_new != pass) continue;
                Chunk c{ a, b - a, 0u, 16u * (b - a), general ? 1u : 0u };
                if (!general) {
                    const int64_t A = 16 * (int64_t)a, n16 = 16 * (int64_t)(b - a);
                    c.c_lo = (uint32_t)std::max<int64_t>((int64_t)sub[k].lo - A, 0);
                    c.c_hi = (uint32_t)std::min<int64_t>((int64_t)sub[k].hi - A, n16);
                }
                out.push_back(c);
            }
    return true;
}

// The work list of one call: every token row planned, flattened into items (chunks) with their
// 256-cell score tiles; tok = tok_first[T] | tok_count[T]. FaWorkFixed holds at most the inline list
// (kFaInlItems items of at most kFaInlTok tokens) in fixed arrays: planning it allocates nothing.
template <class Items, class Tok, class Chunks>
struct FaWorkT {
    Items items;
    Tok tok;
    Chunks ch;               // one row's chunks (planner temporary)
    uint64_t cells = 0;
    uint32_t n_tiles = 0, maxtiles = 1, max_groups = 0;
};
using FaWork = FaWorkT<std::vector<FaItem>, std::vector<uint32_t>, std::vector<Chunk>>;
using FaWorkFixed = FaWorkT<FixedVec<FaItem, kFaInlItems>, FixedVec<uint32_t, 2u * kFaInlTok>,
                            FixedVec<Chunk, kFaInlItems>>;

// Returns TSR_HIP_E_RANGE when a fixed-capacity work list overflows.
template <class W>
int fa_plan_rows(uint32_t E, uint32_t D, uint32_t T, const uint32_t * msum, const uint32_t (*new_runs)[2], uint32_t n_new,
                 bool have_mask, W & w) {
    w.items.clear();
    w.tok.assign(2u * (size_t)T, 0u);
    if (overflowed(w.tok)) return TSR_HIP_E_RANGE;
    w.cells = 0;
    w.n_tiles = 0;
    w.maxtiles = 1;
    w.max_groups = 0;
    auto & ch = w.ch;
    for (uint32_t t = 0; t < T; ++t) {
        ch.clear();
        if (!plan_row(E, D, msum, t, new_runs, n_new, ch)) return TSR_HIP_E_MASK;
        if (overflowed(ch)) return TSR_HIP_E_RANGE;
        w.tok[t] = (uint32_t)w.items.size();
        w.tok[T + t] = (uint32_t)ch.size();
        for (const Chunk & c : ch) {
            if (c.general && !have_mask) return TSR_HIP_E_MASK;
            FaItem it{};
            it.t = t;
            it.u0 = c.u0;
            it.n = c.n;
            it.c_lo = c.c_lo;
            it.c_hi = c.c_hi;
            it.general = c.general;
            it.s_off = (uint32_t)w.cells;
            it.tile0 = w.n_tiles;
            it.ntiles = (16u * c.n + 255u) / 256u;
            w.n_tiles += it.ntiles;
            w.maxtiles = std::max(w.maxtiles, it.ntiles);
            w.max_groups = std::max(w.max_groups, c.n);
            w.cells += 16u * c.n;
            w.items.push_back(it);
        }
        if (overflowed(w.items)) return TSR_HIP_E_RANGE;
    }
    return TSR_HIP_OK;
}

// The scores of many rows on the matrix cores (k_fa_qk_mm), or 0: the one-row kernel (k_fa_qk). Returns the
// number of 256-cell score tiles from group lo / 16 on and in lo the first visible cell of the rows.
// - One FAST run per row, all from one cell, and every item on a tile boundary from there: a tile then lies in
//   one item of each row. The chunk cuts are on such boundaries while NCG is a multiple of 16 groups, which the
//   planner's cap of 4 floor(9344 / (16 n_head_kv)) is not for every n_head_kv (72 groups for 32 KV heads, 116
//   for 20), so the items themselves are looked at.
// - Enough scores: it needs the queries' quantization as a launch of its own (3-6 us), and pays from ~4 M scores
//   of D 128 on. Measured, one-row kernel -> QACT + this one: 512 rows behind 1536 cells (29 M scores) 110 -> 56
//   us, 300 rows behind 700 (8 M) 38 -> 30, D 64: 256 rows from cell 0 (1.3 M) 9.4 -> 13.7.
// - At least two thirds of the scores that it forms in use: a workgroup forms a tile for 32 rows when one of them
//   reaches it. Whole calls, one-row kernel -> this one, 64 query heads of D 128: 1 row of 103 K cells 115 ->
//   407 us, 8 rows of 22 K 123 -> 162, 512 rows, 16 of them of 6000 cells and the others of 40, 365 -> 582; behind
//   12 K cells 17 rows 134 -> 144, 20 rows 150 -> 156, 22 rows (0.69 in use) 162 -> 164, 28 rows 198 -> 193, 32 rows
//   221 -> 199; with 32 heads 20 rows 91 -> 93, 22 rows 98.3 -> 97.9, 28 rows 117 -> 111.
template <class W>
uint32_t fa_score_tiles(const W & w, uint32_t D, uint32_t n_head, uint32_t T, const uint32_t * msum, uint32_t & lo) {
    lo = msum[8];
    if (D > 128u || (msum[3] & 1u) != 0u || w.cells * n_head * (D / 64u) < (10ull << 20) ||
        4u * w.cells * n_head >= (1ull << 31) || (uint64_t)T * n_head * D >= (1ull << 31))
        return 0u;
    uint32_t n_map = 0, n_blk = 0;                                // tiles of the longest row, of the 32 rows so far
    uint64_t formed = 0;                                          // cells
    for (uint32_t t = 0; t < T; ++t) {
        const uint32_t * r = msum + 8u + 4u * t;
        if (r[0] != lo || r[1] <= r[0] || r[2] < r[3]) return 0u;
        n_blk = std::max(n_blk, ((r[1] + 15u) / 16u - lo / 16u + 15u) / 16u);
        if (t % 32u != 31u && t + 1u < T) continue;
        n_map = std::max(n_map, n_blk);
        formed += 32u * 256u * (uint64_t)n_blk;
        n_blk = 0;
    }
    if (3u * w.cells < 2u * formed) return 0u;
    for (const FaItem & it : w.items)
        if (((it.u0 - lo / 16u) & 15u) != 0u) return 0u;
    return n_map;
}

// The device form of a work list: items | tok_first | tok_count and, with n_map != 0 (fa_score_tiles), the
// item of every (tile, row) [n_map][T], ~0u none, and the rows' run ends [T].
inline size_t fa_list_bytes(size_t n_items, uint32_t T, uint32_t n_map) {
    return n_items * sizeof(FaItem) + 8u * (size_t)T + (n_map ? 4u * ((size_t)n_map * T + T) : 0u);
}
template <class W>
void fa_pack_list(const W & w, uint32_t T, uint32_t n_map, uint32_t lo, const uint32_t * msum, uint8_t * list) {
    const size_t n_items = w.items.size();
    memcpy(list, &w.items[0], n_items * sizeof(FaItem));
    memcpy(list + n_items * sizeof(FaItem), &w.tok[0], 8u * (size_t)T);
    if (n_map == 0u) return;
    uint32_t * m = (uint32_t *)(list + n_items * sizeof(FaItem) + 8u * (size_t)T);
    std::fill(m, m + (size_t)n_map * T, 0xFFFFFFFFu);
    for (size_t i = 0; i < n_items; ++i) {
        const FaItem & it = w.items[i];
        for (uint32_t k = 0, a0 = (it.u0 - lo / 16u) / 16u; k < it.ntiles; ++k) m[(size_t)(a0 + k) * T + it.t] = (uint32_t)i;
    }
    for (uint32_t t = 0; t < T; ++t) m[(size_t)n_map * T + t] = msum[8u + 4u * t + 1u];
}

// The scratch of one unplanned call (byte offsets). With n_map != 0 the tail of the list (tile map, run ends) and
// the quantized queries lie where the P.V kernel later writes the channel partials: the score kernel, which runs
// before it, is their only reader, and the call needs no more scratch than on the other route.
struct FaLayout {
    size_t S, Mp, LP, items, OP, xq, xd, bytes;
};
inline FaLayout fa_layout(size_t n_items, uint64_t cells, uint32_t n_tiles, uint32_t T, uint32_t n_head, uint32_t D,
                          bool inl, uint32_t n_map) {
    auto up256 = [](size_t x) { return (x + 255u) & ~(size_t)255u; };
    const size_t K = (size_t)n_head * D;
    FaLayout l{};
    l.Mp = up256(4u * (size_t)cells * n_head);
    l.LP = l.Mp + up256(4u * (size_t)n_tiles * n_head);
    l.items = l.LP + up256(4u * n_items * kC * n_head);
    l.OP = l.items + (inl ? 0u : up256(fa_list_bytes(n_items, T, 0u)));
    l.bytes = l.OP + up256(4u * n_items * kC * K);
    if (n_map != 0u) {
        l.xq = up256(l.items + fa_list_bytes(n_items, T, n_map));
        l.xd = l.xq + up256(T * K);
        l.bytes = std::max(l.bytes, l.xd + up256(T * K / 8u));
    }
    return l;
}

}  // namespace tsr
