// glue.hpp -- device helpers of the decode-layer glue ops, shared by their own kernels and by the
// kernels that fuse them (the matvec's x preparation, ROPE + SET_ROWS_KV): the RMS_NORM scale,
// SIN / COS and the ROPE angle recurrence, on the f32 rules of tsr_dev.hpp.
#pragma once

#include "kernels.hpp"
#include "tsr_dev.hpp"

namespace tsr {

__device__ __forceinline__ float ssqrt(float a) { return fin(sqrtf(daz(a))); }   // correctly rounded sqrtf
__device__ __forceinline__ float fneg(float x) { return bf(fb(x) ^ 0x80000000u); }

// ---- RMS_NORM scale (sw/sim/tsr_ref_vu.c:171-263; sw/ctrl/ref/rmsnorm_ref.hpp:11-14) ---------------
// The RED sum of x^2 is 128 partials, p_i = FA(... FA(+0, FM(x_i, x_i)) ..., FM(x_(i+128k), ...)) in
// order of k, then a 7-level tree of adjacent pairs. Every square FM(x, x) is +0, a positive normal,
// +Inf or a NaN, so every partial and tree sum is one of those too (a sum of non-negative normals is
// at least its larger addend): the plain IEEE addition never rounds into the subnormal range, keeps a
// NaN a NaN, and equals FA on these operands up to the NaN payload, which the last sum (FA of the two
// halves, rms_scale) makes canonical. sq_rule(x) is FM(x, x) but for that payload: a subnormal x squares
// to a subnormal or zero and a tiny normal x to a subnormal, each flushed to +0. rms_tree64 runs the tree on
// the 128 threads holding p_0 .. p_127 (threads 0 .. 127 of the workgroup, p_i on thread i): levels
// 1-6 on DPP and swizzles within each wave (f32 addition is commutative, so the exchange partners xor
// 1, xor 2, half mirror, mirror, xor 16, xor 32 form exactly the tree's pairs); it returns the sum of
// the wave's 64 partials in every lane. The caller adds the two halves (level 7): sum = FA(lo, hi).
__device__ __forceinline__ float sq_rule(float x) { return ftz(x * x); }
__device__ __forceinline__ float rms_tree64(float p) {
    p = p + dpp_f<kDppXor1>(p);
    p = p + dpp_f<kDppXor2>(p);
    p = p + dpp_f<kDppRowHalfMirror>(p);
    p = p + dpp_f<kDppRowMirror>(p);
    p = p + xor16_f(p);
    p = p + xor32_f(p);
    return p;
}
// s = RC(SQ(FA(FM(sum, inv_n), eps))) from the two wave sums of the tree.
__device__ __forceinline__ float rms_scale(float lo, float hi, float inv_n, float eps) {
    return srcp(ssqrt(sadd(smul(sadd_n(lo, hi), inv_n), eps)));
}

// ---- SIN / COS (VU 6.6; sw/sim/tsr_ref_math.c:232-416) -------------------------------------------
// t 2/pi = M round(2/pi 2^64) 2^(E - 214) in 128-bit integers: the integer part mod 4 is the
// quadrant, the fraction (units of 2^-62) is rounded to the nearest quadrant; the remainder
// r = RNE24(F round(pi/2 2^62) 2^-124) enters the Cephes sinf / cosf polynomials on the f32 rules
// (r, z = r r and the polynomial values are never subnormal except r = 0).
typedef unsigned __int128 u128;
constexpr uint64_t kTwoOverPi64 = 0xA2F9836E4E44152Aull;        // 2/pi = 0.A2F9836E4E441529FC27... (hex)
constexpr uint64_t kPiOver2_62 = 0x6487ED5110B4611Aull;         // pi/2 = 1.921FB54442D18469898C... (hex)

__device__ __forceinline__ float u128_to_f32(u128 R, bool neg) {  // RNE24(R 2^-124), 0 < R < 2^124
    const uint64_t hi = (uint64_t)(R >> 64), lo = (uint64_t)R;
    const int b = hi ? 64 + (63 - __builtin_clzll(hi)) : 63 - __builtin_clzll(lo);
    const int shift = b - 23;
    uint64_t sig = (uint64_t)(R >> shift);
    const u128 rem = R & ((((u128)1) << shift) - 1u), half = ((u128)1) << (shift - 1);
    uint32_t be = (uint32_t)(b + 3);
    if (rem > half || (rem == half && (sig & 1u))) {
        if (++sig == (1ull << 24)) { sig >>= 1; ++be; }
    }
    return bf((neg ? 0x80000000u : 0u) | (be << 23) | ((uint32_t)sig & 0x007FFFFFu));
}

__device__ inline void dsincos(float t, float * so, float * co) {
    const uint32_t u = fb(daz(t)), a = u & 0x7FFFFFFFu;
    if (a >= 0x7F800000u) { *so = *co = bf(kNaN); return; }
    const uint32_t E = a >> 23;
    if (E < 115u) { *so = bf(u); *co = 1.0f; return; }         // zero and |t| < 2^-12
    const uint64_t M = 0x00800000u | (a & 0x007FFFFFu);
    const u128 P = (u128)M * kTwoOverPi64;
    const int sh = 214 - (int)E;                                  // -40 .. 99
    const uint64_t mask62 = (1ull << 62) - 1u;
    uint32_t k4;
    uint64_t F;
    if (sh >= 62) { k4 = (uint32_t)(P >> sh) & 3u; F = (uint64_t)(P >> (sh - 62)) & mask62; }
    else if (sh >= 0) { k4 = (uint32_t)(P >> sh) & 3u; F = (uint64_t)(P << (62 - sh)) & mask62; }
    else { k4 = (uint32_t)(P << -sh) & 3u; F = 0; }
    bool rneg = false;
    uint64_t Fm = F;
    if (F >= (1ull << 61)) { k4 = (k4 + 1u) & 3u; rneg = true; Fm = (1ull << 62) - F; }
    const float r = Fm ? u128_to_f32((u128)Fm * kPiOver2_62, rneg) : 0.0f;
    const float z = smul(r, r);
    float p = smul(-1.9515295891e-4f, z);
    p = sadd(p, 8.3321608736e-3f);
    p = smul(p, z);
    p = sadd(p, -1.6666654611e-1f);
    p = smul(p, z);
    p = smul(p, r);
    const float sn = sadd(p, r);
    p = smul(2.443315711809948e-5f, z);
    p = sadd(p, -1.388731625493765e-3f);
    p = smul(p, z);
    p = sadd(p, 4.166664568298827e-2f);
    p = smul(p, z);
    p = smul(p, z);
    const float cs = sadd(ssub(p, smul(0.5f, z)), 1.0f);
    float S, C;
    switch (k4) {
        case 0: S = sn; C = cs; break;
        case 1: S = cs; C = fneg(sn); break;
        case 2: S = fneg(sn); C = fneg(cs); break;
        default: S = fneg(cs); C = sn; break;
    }
    *so = (u >> 31) ? fneg(S) : S;
    *co = C;
}


// ---- ROPE angles (sw/sim/tsr_ref_vu.c:308-376) -------------------------------------------------------
// theta_0 = i2f(pos), phi_i = theta_i (divided by the freq factor FD, times freq_scale FM, when
// given), theta_(i+1) = FM(theta_i, TS), i < half, written to phi[]. Without factors the chain is
// run with plain multiplies: theta_0 is an integer and TS a normal number, so each plain product
// equals the rule's FM unless it is subnormal (FTZ) -- the chain is then run again with FM.
__device__ __forceinline__ void rope_angles(int32_t pos, uint32_t half, float ts, const float * ff, float freq_scale,
                                            bool fs, float * phi) {
    if (ff == nullptr && !fs) {
        float theta = i2f(pos);
        bool sub = false;
        for (uint32_t i = 0; i < half; ++i) {
            phi[i] = theta;
            theta = theta * ts;
            sub |= __builtin_amdgcn_classf(theta, 0x90) != 0;   // -/+ subnormal
        }
        if (!sub) return;
    }
    float theta = i2f(pos);
    for (uint32_t i = 0; i < half; ++i) {
        float f = ff ? sdiv(theta, ff[i]) : theta;
        if (fs) f = smul(freq_scale, f);
        phi[i] = f;
        theta = smul(theta, ts);
    }
}

// The same recurrence with one angle per lane: every lane runs the whole chain (the same operations
// in the same order, so the same values) and lane l keeps phi_l (l < half <= 64, all of them active; no freq
// factors, freq_scale 1). Returns c_l = FM(M, cos phi_l) and s_l = FM(M, sin phi_l); lanes from half on hold
// unused values.
__device__ __forceinline__ void rope_cs_lane(int32_t pos, uint32_t half, float ts, float m, uint32_t lane, float * c,
                                             float * s) {
    float theta = i2f(pos), mine = 0.0f;
    for (uint32_t i = 0; i < half; ++i) {
        mine = i == lane ? theta : mine;
        theta = theta * ts;
    }
    // -/+ subnormal: run the rule instead (one test of the kept angles; a test of every step of the chain, 0.7 us at
    // 64 angles, was what the chain's lanes waited for)
    if (__ballot(lane < half && __builtin_amdgcn_classf(mine, 0x90)) != 0ull) {
        theta = i2f(pos);
        for (uint32_t i = 0; i < half; ++i) {
            mine = i == lane ? theta : mine;
            theta = smul(theta, ts);
        }
    }
    float sn, cs;
    dsincos(mine, &sn, &cs);
    *c = smul(m, cs);
    *s = smul(m, sn);
}

// ROPE of 4 consecutive values of one head (value jh0 .. jh0 + 3 of the head, jh0 % 4 == 0) from the
// per-lane tables of rope_cs_lane (every lane of the wave active: the entries are read by bpermute).
// NORMAL pairs (2i, 2i + 1) lie inside the 4 values; NEOX pairs (i, i + half) take the partner from
// `part` (the 4 values half away). y0 = FS(FM(x0, c), FM(x1, s)), y1 = FA(FM(x0, s), FM(x1, c));
// values from n_dims on are kept.
// rope4 when the lane's angles come from the table in registers -- csa: (cos, sin) of angles i, i + 1,
// csb: of angles i + 2, i + 3, with i the lane's first angle (NORM: jh0 / 2, NEOX: jh0 mod n_dims / 2)
// -- and the wave qualifies (wave-uniform result): every x, partner, cos and sin a normal number or a
// zero. DAZ is then the identity; a product can be subnormal (FTZ) or overflow, never NaN; the sum or
// difference of two such products can be subnormal or NaN (Inf - Inf); each case is one class test.
// The result equals rope4's. Returns false when the wave does not qualify.
__device__ __forceinline__ bool rope4_tab_fast(float4 & out, float4 v, float4 part, uint32_t jh0, uint32_t n_dims,
                                               bool neox, float4 csa, float4 csb) {
    const uint32_t half = n_dims / 2u;
    const float x[4] = { v.x, v.y, v.z, v.w }, pr[4] = { part.x, part.y, part.z, part.w };
    const float c[4] = { csa.x, neox ? csa.z : csa.x, neox ? csb.x : csa.z, neox ? csb.z : csa.z };
    const float sn[4] = { csa.y, neox ? csa.w : csa.y, neox ? csb.y : csa.w, neox ? csb.w : csa.w };
    constexpr int kBad = 0x297;                                   // NaN, +-Inf, +-subnormal
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        bad |= __builtin_amdgcn_classf(x[k], kBad) | __builtin_amdgcn_classf(c[k], kBad) | __builtin_amdgcn_classf(sn[k], kBad);
        if (neox) bad |= __builtin_amdgcn_classf(pr[k], kBad);
    }
    if (__ballot(bad) != 0ull) return false;
    auto ftz = [](float r) { return __builtin_amdgcn_classf(r, 0x90) ? bf(fb(r) & 0x80000000u) : r; };
    float y[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        const uint32_t jh = jh0 + k;
        const bool first = neox ? jh < half : (jh & 1u) == 0u;
        const float x0 = first ? x[k] : (neox ? pr[k] : x[k ^ 1u]);
        const float x1 = first ? (neox ? pr[k] : x[k ^ 1u]) : x[k];
        const float p1 = ftz(x0 * (first ? c[k] : sn[k])), p2 = ftz(x1 * (first ? sn[k] : c[k]));
        float r = ftz(first ? p1 - p2 : p1 + p2);
        r = __builtin_amdgcn_classf(r, 0x3) ? bf(kNaN) : r;
        y[k] = jh < n_dims ? r : x[k];
    }
    out = make_float4(y[0], y[1], y[2], y[3]);
    return true;
}

__device__ __forceinline__ float4 rope4(float4 v, float4 part, uint32_t jh0, uint32_t n_dims, bool neox, float c_l,
                                        float s_l) {
    const uint32_t half = n_dims / 2u;
    float x[4] = { v.x, v.y, v.z, v.w }, pr[4] = { part.x, part.y, part.z, part.w }, y[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        const uint32_t jh = jh0 + k;
        const uint32_t ip = neox ? (jh < half ? jh : jh - half) : (jh >> 1);
        const float c = __int_as_float(__builtin_amdgcn_ds_bpermute((int)(min(ip, 63u) << 2), __float_as_int(c_l)));
        const float s = __int_as_float(__builtin_amdgcn_ds_bpermute((int)(min(ip, 63u) << 2), __float_as_int(s_l)));
        const bool first = neox ? jh < half : (jh & 1u) == 0u;
        const float x0 = first ? x[k] : (neox ? pr[k] : x[k ^ 1u]);
        const float x1 = first ? (neox ? pr[k] : x[k ^ 1u]) : x[k];
        const float r = first ? ssub(smul(x0, c), smul(x1, s)) : sadd(smul(x0, s), smul(x1, c));
        y[k] = jh < n_dims ? r : x[k];
    }
    return make_float4(y[0], y[1], y[2], y[3]);
}

}  // namespace tsr
