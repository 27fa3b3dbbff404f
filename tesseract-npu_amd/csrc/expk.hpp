// expk.hpp -- EXPK on the device (VU 6.3; sw/sim/tsr_ref_math.c:78-159), shared by the flash
// attention and the SILU of the glue kernels.
#pragma once

#include "kernels.hpp"
#include "tsr_dev.hpp"

namespace tsr {

// EXPK(v, P1) (VU 6.3; sw/sim/tsr_ref_math.c:78-159), constants from the host (ExpkTab). The
// 2^(j/64) table is read from LDS (t64): an index into the kernel arguments that differs per lane
// would be a vector load from the argument segment on every call. Straight-line, with no special-case
// selects but the NaN one: |v| log2(e) 2^32 = Mv LK 2^(ev - 156) is formed exactly (Mv < 2^24, LK <
// 2^39: 63 bits) and shifted right by min(156 - ev, 63), so a zero gives T = 0 and the result 1 like any
// tiny v, and ev >= 156 (Inf included) keeps the whole product, whose integer part (>= 2^29) drives the
// exponent past 255 (Inf) or below 1 (+0 for negative v) as the saturation cases of the reference do.
// The rounding of the 2^frac significand M (in [2^30, 2^31 + 2^25)) to 24 bits, ties to even, is its
// f32 conversion. Checked against the restatement of the reference over all 2^32 inputs.
template <typename Lookup>
__device__ __forceinline__ float expk_with(float v, const ExpkTab & e, Lookup t64) {
    const uint32_t u = fb(daz(v));
    const uint32_t a = u & 0x7FFFFFFFu;
    const bool neg = (u >> 31) != 0u;
    const uint32_t ev = a >> 23;
    const uint32_t mv = 0x00800000u | (a & 0x007FFFFFu);
    const uint32_t sh = min(156u - min(ev, 156u), 63u);
    const uint32_t lk_lo = (uint32_t)e.lk, lk_hi = (uint32_t)(e.lk >> 32);
    const uint64_t prod = ((uint64_t)(__umulhi(mv, lk_lo) + mv * lk_hi) << 32) | (uint64_t)(mv * lk_lo);
    const uint64_t T = prod >> sh;
    // +-T in fixed point: the integer part n0 (floor, |n0| < 2^31) and the fraction F
    const uint64_t Ts = neg ? 0ull - T : T;
    const int32_t n0 = (int32_t)(uint32_t)(Ts >> 32);
    const uint32_t F = (uint32_t)Ts;
    // the cubic in fixed point: G < 2^26 and c1, c2, c3 < 2^32 (ln2^k / k! 2^32), and every sum below stays
    // under 2^32, so each (G x) >> 32 is the high word of one 32-bit product; likewise t < 2^31, pf < 2^26
    const uint32_t G = F & 0x03FFFFFFu;
    const uint32_t pf = __umulhi(G, (uint32_t)e.c1 + __umulhi(G, (uint32_t)e.c2 + __umulhi(G, (uint32_t)e.c3)));
    const uint32_t t = t64(F >> 26);
    const uint32_t M = t + __umulhi(t, pf);
    const uint32_t fm = fb((float)M);                             // exponent field 157 or 158
    const int32_t be = (int32_t)(fm >> 23) - 30 + n0;
    const uint32_t r = be >= 255 ? 0x7F800000u : (be <= 0 ? 0u : (((uint32_t)be << 23) | (fm & 0x007FFFFFu)));
    return bf(a > 0x7F800000u ? kNaN : r);
}
__device__ __forceinline__ float expk(float v, const ExpkTab & e, const uint32_t * t64) {
    return expk_with(v, e, [t64](uint32_t j) { return t64[j]; });
}
// EXPK(FM(FS(s, m), scale)) by the f32 rules, for operands s and m that are never subnormal (scores
// and maxima): only the difference's FTZ is kept. The rule ops' NaN canonicalization is dropped since
// EXPK maps every NaN to the canonical one, and the product's FTZ since EXPK's own DAZ flushes a
// subnormal input to the same signed zero.
template <typename Lookup>
__device__ __forceinline__ float expk_diff_with(float s, float m, float scale, const ExpkTab & e, Lookup t64) {
    const float d = s - m;
    const float dz = __builtin_amdgcn_classf(d, 0x90) ? bf(fb(d) & 0x80000000u) : d;
    return expk_with(dz * scale, e, t64);
}
__device__ __forceinline__ float expk_diff(float s, float m, float scale, const ExpkTab & e, const uint32_t * t64) {
    return expk_diff_with(s, m, scale, e, [t64](uint32_t j) { return t64[j]; });
}
// EXPK(FM(FS(s, m), scale)) for s <= m in MAXT's order (every ASMAX exponent: m is the maximum, so the
// argument v is <= 0 or NaN), in f64 arithmetic: EXPK's integers are products of up to 64 bits truncated to
// integers, and with the f64 rounding mode set to truncation (f64_round_to_zero) fma(a, b, 2^52) holds
// floor(a b) exactly in its low word. A step is a full-rate fma and add where the 32-bit form takes quarter-
// rate integer products (~33 issue slots a value instead of ~60). v is cut off at -180, whose result is +0 as
// that of everything below. Equal to the oracle's EXPK on all 2^31 negative floats (tests/test_rounding.py, on the
// CPU in the truncating mode). td: t64[j] 2^-32 as f64, in LDS.
// The wave's f64 (and f16) operations truncate from here on (MODE.FP_ROUND[3:2] = toward zero); f32 keeps
// rounding to nearest even. In asm, because the compiler takes a mode set by its builtin back in front of
// the next f64 operation. x: a value on which every f64 operation meant depends (the only order that the
// compiler keeps between them and the asm).
__device__ __forceinline__ void f64_round_to_zero(float & x) {
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3\n\ts_nop 7" : "+v"(x));
}
__device__ __forceinline__ float expk_neg_diff(float s, float m, float scale, const ExpkNeg & e, const double * td) {
    constexpr double k52 = 4503599627370496.0;
    const float d = s - m;
    const float dz = __builtin_amdgcn_classf(d, 0x90) ? bf(fb(d) & 0x80000000u) : d;
    const float v = dz * scale;
    const double T = __builtin_fma((double)__builtin_fmaxf(v, -180.0f), -e.lk, k52);   // 2^52 + |v| log2(e) 2^32
    const uint64_t r = __builtin_bit_cast(uint64_t, (9007199254740992.0 + 2251799813685248.0) - T);   // 2^52 + 2^51 - T
    const uint32_t F = (uint32_t)r;
    const double G = __builtin_bit_cast(double, 0x4130000000000000ull | (F & 0x03FFFFFFu)) - 1048576.0;   // G 2^-32
    const double m1 = __builtin_fma(G, e.c3, k52);
    const double m2 = __builtin_fma(G, m1 + e.c2, k52);
    const double m3 = __builtin_fma(G, m2 + e.c1, k52);
    const double M = __builtin_fma(td[F >> 26], m3 + (4294967296.0 - k52), k52);
    const uint32_t fm = fb((float)(uint32_t)__builtin_bit_cast(uint64_t, M));
    const uint32_t x = fm + (((uint32_t)(r >> 32) - (0x43380000u + 30u)) << 23);   // the exponent moved by n0 - 30
    const uint32_t q = (int32_t)x < 0x00800000 ? 0u : x;
    return bf(v != v ? kNaN : q);
}
// EXPK with the table in a register: lane j of the wave holds t64[j] (read by ds_bpermute, no
// LDS table and no barrier).
__device__ __forceinline__ float expk_reg(float v, const ExpkTab & e, uint32_t t64_lane) {
    return expk_with(v, e, [t64_lane](uint32_t j) {
        return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(j << 2), (int)t64_lane);
    });
}

// SILU(x) = FM(x, RC(FA(1, EXPK(x, N1)))) with EXPK(x, N1) = EXPK(-x, P1), and SWIGLU(g, u) =
// FM(SILU(g), u) (sw/sim/tsr_ref_vu.c:102-133; sw/sim/tsr_ref_math.c:165-172).
__device__ __forceinline__ float swiglu_reg(float g, float u, const ExpkTab & e, uint32_t t64_lane) {
    const float ng = bf(fb(g) ^ 0x80000000u);
    const float sig = srcp(sadd(1.0f, expk_reg(ng, e, t64_lane)));
    return smul(smul(g, sig), u);
}

// TANH (VU 6.5; sw/sim/tsr_ref_math.c:182-199): canonical NaN for NaN; for |x| < 2^-6 (DAZ'd)
// |x| (3 - x^2) THIRD with THIRD = f32(1/3); else (1 - e) RC(1 + e), e = EXPK(|x|, N2); the sign of x.
// LK(N2) = 2 LK(P1) with a negative sign (tsr_ref_math.c:53-59), so EXPK(a, N2) = EXPK(-(a + a), P1):
// a + a only moves the exponent (a is DAZ'd and normal here), or overflows to Inf, which EXPK
// saturates to 0 as N2 does for its Ev > 156.
// Both forms run on every lane and one is selected (a table lookup that reads another lane's register
// must not sit in a branch).
template <typename Lookup>
__device__ __forceinline__ float tanh_with(float x, const ExpkTab & e, Lookup t64) {
    const uint32_t u = fb(x);
    const uint32_t axb = fb(daz(x)) & 0x7FFFFFFFu;
    const float ax = bf(axb);
    const float q = smul(ax, ax);
    const float small = smul(smul(ssub(3.0f, q), ax), bf(0x3EAAAAABu));
    const float ee = expk_with(-(ax + ax), e, t64);
    const float big = smul(ssub(1.0f, ee), srcp(sadd(1.0f, ee)));
    float t = axb < 0x3C800000u ? small : big;
    t = (u >> 31) ? bf(fb(t) ^ 0x80000000u) : t;
    return (u & 0x7FFFFFFFu) > 0x7F800000u ? bf(kNaN) : t;
}

}  // namespace tsr
