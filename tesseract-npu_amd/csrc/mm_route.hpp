// mm_route.hpp -- which kernels a MUL_MAT of several token rows runs on, and which partials a wave of the Q4_K
// prefill kernel forms. Plain C++ without the HIP runtime, so that it is checked on the CPU.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace tsr {

// The few-row kernels (k_matrows.hip: the weights once per 15 rows) instead of the matvec once per row, for T > 1.
// The matvec has a workgroup per row block (rb weight rows) and row, and its time is its rounds of n_cu workgroups; a
// few-row workgroup quantizes all its rows itself, up to 8 at a time, which takes the time of a number s of matvec
// rounds. Measured over 4661 calls of N 200 .. 50000, K 512 .. 14336 and 2 .. 15 rows, plain, with the norm and with
// GLU, this rule takes the slower one by more than 6 % in 8 of them (at most 10 %). Where the lines lie, matvec ->
// few rows in us:
// - one round of matvecs: Q4_K 768x2048, 5 rows 5.5 -> 6.1, with the norm 7.2 -> 9.9;
// - s = 1 up to 4 rows, 2 up to 8, 3 up to 15 where a row takes several steps to quantize (Q8_0 from K 2048 on, Q4_K
//   from 6144, with the norm from 4096). Two rounds: Q8_0 1024x4864 with norm, 8 rows 17.3 -> 19.5, Q4_K 1024x8192
//   with norm, 8 rows 15.1 -> 20.1, 512x8192 with norm, 15 rows 15.2 -> 32.1. Three: Q8_0 1024x4864, 12 rows 14.3 ->
//   15.7. Four: Q8_0 896x4864, 15 rows 19.8 -> 15.5;
// - one less where one step is enough: Q8_0 1024x2048 with norm, 8 rows, two rounds 12.4 -> 10.8; Q4_K 1024x2048 with
//   norm, 12 rows, three 16.4 -> 11.5; but 512x4096 with norm, 12 rows, two 12.4 -> 16.1;
// - Q4_K without the norm up to K 2048: always 1 (768x512, 10 rows, two rounds 8.0 -> 6.7);
// - Q8_0 without the norm has two workgroups a CU: at least 2 where one step is enough (1024x2048, 7 rows, two rounds
//   6.6 -> 6.9, 11 rows, three 8.2 -> 8.6), and 2 for small weights of larger row blocks (4864x1536, 2 rows 6.7 -> 8.4;
//   14336x2048 14.1 -> 10.7);
// - two rows of large Q4_K weights (the few-row kernels form the results of 16): 28672x2048 14.1 -> 15.6;
// - the norm of long rows, more than 8: 4 (Q4_K 1024x8192, 14 rows, four rounds 27.4 -> 32.6).
inline bool few_rows_pay(bool q4k, uint32_t K, uint32_t rb, uint32_t blocks, uint32_t T, bool norm, uint32_t n_cu) {
    auto rounds = [n_cu](uint64_t workgroups) { return (workgroups + n_cu - 1u) / n_cu; };
    const uint32_t shares = (T + 14u) / 15u, rows = (T + shares - 1u) / shares;   // as tsr_launch_mr splits them
    uint32_t s = rows <= 4u ? 1u : (rows <= 8u ? 2u : 3u);
    if (q4k) {
        if (T == 2u && rb > 96u && K >= 1024u) s = 2u;
        else if (!norm && K <= 2048u) s = 1u;
        else if (K <= (norm ? 4096u : 6144u)) s = std::max(s, 2u) - 1u;
    } else {
        if (norm) s = K <= 2048u ? std::max(s, 2u) - 1u : s;
        else if (rb > 16u && (K < 1024u || rb * K < 65536u)) s = 2u;
        else if (rb <= 16u && K <= 2048u) s = std::max(s, 2u);
    }
    if (norm && rows > 8u && K > (q4k ? 7168u : 6144u)) s = 4u;
    return rounds((uint64_t)blocks * T) > s * rounds((uint64_t)blocks * shares);
}

// k_mm_q4k: the partials of wave j of W (4 or 8) for rows of nb super-blocks. The first nb mod 16 partials have one
// super-block more than the others. A wave takes `per` neighbours from partials 0 .. 7 and the same ones of 8 .. 15,
// subtrees of the 16-partial tree, or (halves 1) neighbours only.
// Four waves, one a SIMD: two and two; four neighbours gave the first wave up to twice the others' work (2048x5632,
// 160 rows 20.8 -> 18.4 us). Eight waves, j and j + 4 on one SIMD: one and one where that leaves the fullest SIMD a
// super-block less (GLU 896x4864, 64 rows 11.6 -> 10.6 us), else two neighbours, whose sum goes through LDS once
// (2048x5632, 64 rows 12.2 -> 11.4).
struct MmSplit {
    uint32_t halves, per;                                         // 2: both halves; partials in each
};
constexpr MmSplit mm_split(uint32_t nb, uint32_t W) {
    const uint32_t np = nb > 4u ? 8u : (nb > 2u ? 4u : nb), rem = nb & 15u;   // partials in use in a half, a power of two
    if (W == 8u && nb > 8u && !((rem >= 2u && rem <= 4u) || (rem >= 10u && rem <= 12u))) return { 1u, 2u };
    return { nb > 8u ? 2u : 1u, np > W ? np / W : 1u };
}
// The wave's partial pi < halves * per, in the order it forms them.
constexpr uint32_t mm_partial(const MmSplit & m, uint32_t j, uint32_t pi) {
    return m.per * j + pi + (pi < m.per ? 0u : 8u - m.per);
}

}  // namespace tsr
