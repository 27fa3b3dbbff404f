// The partials that the waves of the Q4_K prefill kernel form (mm_route.hpp: mm_split, mm_partial), for rows of
// 1 .. 128 super-blocks: every partial of the row in exactly one wave, a wave's partials in ascending order and each
// half's beside each other, and even shares. Exit status 1 and the first row length that breaks one.
#include "mm_route.hpp"
#include "wlayout.hpp"

#include <cstdio>

int main() {
    for (uint32_t nb = 1; nb <= 128u; ++nb)
        for (uint32_t W : { 4u, 8u }) {
            const tsr::WGeom g = tsr::wgeom(32u, nb, 32u, true);
            const tsr::MmSplit m = tsr::mm_split(nb, W);
            uint32_t seen[16] = {}, share[8] = {}, simd = 0;
            for (uint32_t j = 0; j < W; ++j)
                for (uint32_t pi = 0; pi < m.halves * m.per; ++pi) {
                    const uint32_t p = tsr::mm_partial(m, j, pi);
                    const bool beside = pi % m.per == 0u || p == tsr::mm_partial(m, j, pi - 1u) + 1u;
                    const bool half = m.halves == 1u || p / 8u == pi / m.per;
                    if (p >= 16u || !beside || !half) return printf("%u super-blocks, %u waves: wave %u, partial %u\n", nb, W, j, p), 1;
                    seen[p]++;
                    share[j] += tsr::wl_count(g, p);
                }
            for (uint32_t p = 0; p < 16u; ++p)
                if (tsr::wl_count(g, p) != 0u ? seen[p] != 1u : seen[p] > 1u)
                    return printf("%u super-blocks, %u waves: partial %u in %u waves\n", nb, W, p, seen[p]), 1;
            for (uint32_t j = 0; j < W; ++j) {
                const uint32_t both = share[j] + (W == 8u ? share[(j + 4u) % 8u] : 0u);   // waves j, j + 4: one SIMD
                simd = both > simd ? both : simd;
            }
            // eight waves share the SIMDs evenly; the fullest of four has at most one super-block too many
            if (nb > 4u && simd > (nb + 3u) / 4u + (W == 8u ? 0u : 1u))
                return printf("%u super-blocks, %u waves: %u on one SIMD\n", nb, W, simd), 1;
        }
    printf("128 row lengths\n");
    return 0;
}
