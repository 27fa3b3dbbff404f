// The rule of mm_route.hpp at measured shapes (256 CUs): each line is a call whose other kernels took at least
// 5 % longer. Exit status 1 and the first one that goes the other way.
#include "mm_route.hpp"

#include <cstdio>

struct Call { bool q4k; uint32_t N, K, T; char opt; bool few; };   // opt: - plain, n norm, g GLU

static const Call calls[] = {
    // the matvec: one round of workgroups; few row blocks and long rows; two rows of large weights of short rows
    { true, 1024, 2048, 4, '-', false },  { false, 512, 512, 15, '-', false },   { false, 300, 1024, 15, '-', false },
    { false, 512, 4096, 9, '-', false },  { false, 512, 4096, 15, 'n', false },  { false, 512, 8192, 15, 'n', false },
    { false, 1024, 4864, 8, 'n', false }, { false, 1024, 8192, 12, 'n', false }, { false, 512, 14336, 9, '-', false },
    { true, 512, 4096, 9, 'n', false },   { true, 512, 8192, 9, '-', false },    { true, 512, 8192, 15, 'n', false },
    { true, 1024, 8192, 8, 'n', false },  { true, 1024, 8192, 14, 'n', false },  { true, 512, 14336, 12, '-', false },
    { true, 28672, 2048, 2, '-', false }, { true, 28672, 2048, 2, 'g', false },  { false, 14336, 512, 2, '-', false },
    { false, 4864, 896, 2, 'g', false },  { false, 4096, 2048, 2, 'g', false },  { false, 28672, 896, 2, 'g', false },
    { false, 1024, 2048, 7, '-', false }, { false, 4864, 1536, 2, '-', false }, { false, 1024, 3072, 8, '-', false },
    // the few-row kernels
    { true, 6144, 4096, 8, 'n', true },   { true, 2048, 2048, 3, '-', true },    { true, 1024, 2048, 5, '-', true },
    { true, 1024, 4096, 5, '-', true },   { true, 1024, 4096, 15, '-', true },   { true, 4096, 14336, 15, '-', true },
    { true, 28672, 4096, 3, '-', true },  { true, 28672, 4096, 8, 'n', true },   { true, 5000, 1024, 31, 'n', true },
    { true, 2048, 8192, 3, '-', true },   { false, 4864, 896, 3, '-', true },    { false, 4096, 4096, 2, 'n', true },
    { false, 14336, 4096, 2, '-', true }, { false, 1024, 2048, 5, 'n', true },   { false, 896, 4864, 15, '-', true },
    { false, 1024, 2048, 15, '-', true }, { false, 14336, 2048, 2, '-', true }, { false, 4096, 4096, 5, 'g', true },   { false, 14336, 2048, 2, 'g', true },
};

int main() {
    for (const Call & c : calls) {
        uint32_t rb = (c.N + 255u) / 256u;                        // tsr_wl_rows_per_block (no shape here meets its LDS limit)
        rb = rb < 16u ? 16u : rb + (rb & 1u);
        if (tsr::few_rows_pay(c.q4k, c.K, rb, (c.N + rb - 1u) / rb, c.T, c.opt == 'n', 256u) != c.few) {
            printf("%s %ux%u, %u rows, %c: not %s\n", c.q4k ? "Q4_K" : "Q8_0", c.N, c.K, c.T, c.opt, c.few ? "the few-row kernels" : "the matvec");
            return 1;
        }
    }
    printf("%zu calls\n", sizeof calls / sizeof calls[0]);
    return 0;
}
