// k_matrows.hip -- MUL_MAT of a few token rows (2 .. 15 a workgroup) on gfx950: short ubatches, several sequences
// decoded together, and the fused norm form at any T. Same numerics as the matvec (k_matvec.hip): the term of
// block s goes to partial s mod 16 in order of s, then the 16-partial tree; the fused RMS_NORM, the GLU
// epilogue, addend and accumulation as there.
//
// Work split. As in the matvec a workgroup of 16 waves owns one row block of the weight layout and wave w
// computes partial p[w], but for all tokens at once: the weights are read once instead of once per token. A
// wave multiplies tiles of 16 weight rows (columns of the result) by up to 16 tokens (rows) on the int8
// matrix core: a lane unpacks 32 weight bytes of its own row, whose scales it decoded itself, and holds the
// results of that row for 4 tokens. Each wave quantizes the blocks of x that its partial needs into its own
// LDS area, so the waves meet only for the fused norm's scales and for the tree.
//
// What bounds it: a chain of latencies (x for the norm, x again, the first weights, the tree: ~1 us each) up to
// about one tile a workgroup; then ~140 VALU instructions per tile and Q4_K super-block (2304 bytes), and the
// quantization of every row in every workgroup (A32 ~8, A256 ~6, the norm ~7 instructions a value).
// Against the matvec run once per row (the same box, us):
//   Q4_K norm 6144x4096, 8 rows 40.7 -> 13.3; 4096x14336, 15 rows 93 -> 26; GLU norm 28672x4096, 8 rows 86 -> 28
//   Q8_0 4864x896, 8 rows 14.3 -> 6.1; 14336x4096, 8 rows 84 -> 15; 4096x14336, 15 rows 176 -> 34
// Registers decide it: with 128 a wave, weights requested ahead of the quantization, or addresses kept over
// the phases, spilled 20 to 60 of them and cost 5 to 20 us (mr_again; the rare paths in small steps).
#include "expk.hpp"
#include "glue.hpp"
#include "kernels.hpp"
#include "mv_q4k.hpp"
#include "qact.hpp"
#include "tsr_hip.h"
#include "wlayout.hpp"

#include <algorithm>

namespace tsr {

typedef int v4i_r __attribute__((ext_vector_type(4)));
typedef float v4f_r __attribute__((ext_vector_type(4)));
typedef _Float16 v2h_r __attribute__((ext_vector_type(2)));
typedef _Float16 v8h_r __attribute__((ext_vector_type(8)));
typedef unsigned short v2u_r __attribute__((ext_vector_type(2)));

constexpr uint32_t kMrWaves = 16;

// A lane index whose derived addresses are formed again where it is used: kept over the phases of the kernel
// they would take half of the 128 registers.
__device__ __forceinline__ uint32_t mr_again(uint32_t lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

// The wave's own LDS writes before its own reads (the LDS runs one wave's operations in order).
__device__ __forceinline__ void mr_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float mr_bcast(float v, uint32_t l) {  // lane l's v
    return __int_as_float(__builtin_amdgcn_ds_bpermute((int)(4u * l), __float_as_int(v)));
}

// kPrepNorm: the RMS scale of token t in lane t of every wave. The two halves (lane i: partials i and i + 64) of
// a token's 128-partial chain are summed by two waves (T <= 8) or by one (K % 32 == 0, K <= 8192; missing
// terms of the last round are not added).
__device__ __forceinline__ float mr_norm_scales(const MvArgs & a, uint32_t t0, uint32_t T, uint32_t w, uint32_t lane, float * s_half) {
    const bool two = T <= 8u;
    const uint32_t t = two ? w >> 1 : w, h = two ? w & 1u : 0u;
    if (t < T) {
        const float * x = a.x + (size_t)(t0 + t) * a.x_stride;
        float p[2] = { 0.0f, 0.0f };                              // plain additions: see rms_tree64
        const uint32_t st = two ? 128u : 64u;
        for (uint32_t j0 = 64u * h; j0 < a.K; j0 += 32u * st) {
            float v[32];
#pragma unroll
            for (uint32_t k = 0; k < 32u; ++k) v[k] = x[min(j0 + st * k + lane, a.K - 1u)];
#pragma unroll
            for (uint32_t k = 0; k < 32u; ++k) {
                float & pk = p[k & 1u];
                const float o = two ? p[0] : pk, n = o + sq_rule(v[k]), r = j0 + st * k + lane < a.K ? n : o;
                if (two) p[0] = r;
                else pk = r;
            }
        }
        p[0] = rms_tree64(p[0]);
        p[1] = rms_tree64(p[1]);
        if (lane == 0u) {
            s_half[two ? w : 2u * w] = p[0];
            if (!two) s_half[2u * w + 1u] = p[1];
        }
    }
    lds_barrier();
    return rms_scale(s_half[2u * min(lane, T - 1u)], s_half[2u * min(lane, T - 1u) + 1u], a.inv_n, a.eps);
}

// The partials of NTL tiles (p: row lane % 16, tokens 4 (lane / 16) + r) -> the tree -> y, in rounds of RT
// tiles through LDS (s_p: [wave][tile][token][row]). r0: the first row of the tiles in the row block. Every
// wave of the workgroup calls it; the LDS is free at entry (a barrier inside) and at exit.
template <int NTL>
__device__ __forceinline__ void mr_tree_store(const MvArgs & a, const float (&p)[NTL][4], float * s_p, const int * s_slow,
                                              uint32_t t0, uint32_t T, uint32_t row_lo, uint32_t nrow, uint32_t r0, uint32_t w) {
    const uint32_t lane = mr_again(__lane_id());
    constexpr int RT = NTL < 4 ? NTL : 4;
    const uint32_t c16 = lane & 15u, q = lane >> 4;
    uint32_t t64 = 0;
    if (a.glu) t64 = a.ex.t64[lane];
#pragma unroll
    for (int i0 = 0; i0 < NTL; i0 += RT) {
        lds_barrier();                                            // the last reads of this LDS are done
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (uint32_t r = 0; r < 4u; ++r) s_p[((w * RT + i) * 16u + 4u * q + r) * 16u + c16] = p[i0 + i][r];
        lds_barrier();
        const uint32_t o = 64u * w + lane;                        // whole waves: 64 consecutive outputs
        if (o < 256u * RT) {
            bool slow = false;
#pragma unroll
            for (uint32_t k = 0; k < kMrWaves; ++k) slow |= s_slow[k] != 0;
            float v[16];
#pragma unroll
            for (uint32_t k = 0; k < 16u; ++k) v[k] = s_p[k * RT * 256u + o];
            if (__builtin_expect(!slow, 1)) {
#pragma unroll
                for (int m = 16; m > 1; m >>= 1)
#pragma unroll
                    for (int k = 0; k < m / 2; ++k) v[k] = v[2 * k] + v[2 * k + 1];
            } else {
#pragma unroll
                for (int m = 16; m > 1; m >>= 1)
#pragma unroll
                    for (int k = 0; k < m / 2; ++k) v[k] = sadd(v[2 * k], v[2 * k + 1]);
            }
            float y = canon(v[0]);
            const uint32_t t = (o >> 4) & 15u, r = r0 + 16u * (i0 + (o >> 8)) + (o & 15u);
            if (a.glu) {                                          // every lane: the table is read by bpermute
                y = swiglu_reg(y, dpp_f<kDppXor1>(y), a.ex, t64);
                if ((o & 1u) == 0u && t < T && r < nrow) a.y[(size_t)(t0 + t) * a.y_stride + ((row_lo + r) >> 1)] = y;
            } else if (t < T && r < nrow) {
                float * yp = a.y + (size_t)(t0 + t) * a.y_stride + row_lo + r;
                if (a.add) y = sadd(a.add[(size_t)(t0 + t) * a.add_stride + row_lo + r], y);
                else if (a.acc) y = sadd(*yp, y);
                *yp = y;
            }
        }
    }
    lds_barrier();
}

// ---- Q4_K -----------------------------------------------------------------------------------------
// One super-block and tile: lane quarter q = lane / 16 holds the row's pieces q and q + 4 (piece p: low
// nibbles sub-block 2 (p / 2), high nibbles the next one, values 16 (p mod 2) ..), so the products of set s
// (pieces 4 s + q) and nibble n take the activations of sub-block 4 s + 2 (q / 2) + n, half q mod 2. As in
// k_mm_q4k: sc = 8 a + b scales the quants bytewise for two exact int32 accumulators, the mins meet the
// sub-block sums 64 h + l in one f16 product of integers.
template <int TP>
struct MrX4 {                                                     // LDS of one quantized super-block of 4 TP tokens
    static constexpr uint32_t TT = 4u * TP, kQ = kXq4Stride * TT, kS = 32u * TT, kBytes = kQ + kS + 4u * TT;
    static constexpr uint32_t kSlots = TP == 2 ? 4u : 2u;         // super-blocks a wave holds at once (157.7 KB in all)
};

template <int TP, int NTL>
__global__ __launch_bounds__(1024) void k_mr_q4k(MvArgs a, uint32_t tsh, uint32_t sp_off) {
    const uint32_t t0 = blockIdx.y * tsh, T = min(a.T - t0, tsh);  // the workgroup's tokens
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ float s_half[32];
    __shared__ int s_slow[kMrWaves];
    using X = MrX4<TP>;
    constexpr uint32_t TT = X::TT;
    constexpr int RD = NTL >= 2 ? 2 : 1;                          // tiles requested ahead
    const WGeom g = wgeom(a.N, a.K >> 8, a.rb, true);
    const uint32_t lane = __lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cnt = wl_count(g, w);
    const uint32_t B = blockIdx.x, row_lo = B * g.rb, R = wl_rows(g, B);
    const uint32_t SG = min(g.q + (g.rem ? 1u : 0u), X::kSlots);  // as the launcher's LDS
    uint8_t * s_x = lds + (size_t)w * SG * X::kBytes;
    const uint8_t * wb = a.w + (size_t)B * g.bstride;
    const uint32_t R16 = 16u * R;
    const bool norm = a.prep == kPrepNorm;
    const bool keep = sp_off != 0u;                               // one group, and the tree's LDS lies behind it
    const float scale = norm ? mr_norm_scales(a, t0, T, w, lane, s_half) : 0.0f;
    bool slow = false;

    for (uint32_t r0 = 0; r0 < R; r0 += 16u * NTL) {              // row chunks
    const uint32_t lc = mr_again(lane), c16 = lc & 15u, q = lc >> 4;
    float p[NTL][4];
#pragma unroll
    for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) p[i][r] = 0.0f;
    if (cnt > 0u) {
    const uint32_t oq = q * g.nb * R16, o4 = 4u * g.nb * R16, om = 8u * g.nb * R16;
    uint4 w0[RD], w1[RD], wm[RD];
    auto load_w = [&](int slot, uint32_t i, uint32_t k) {         // ring slot <- tile i of the wave's super-block k
        const uint32_t o = wl_slot(g, w, k) * R16 + 16u * min(r0 + 16u * i + c16, R - 1u);
        w0[slot] = *(const uint4 *)(wb + (oq + o));
        w1[slot] = *(const uint4 *)(wb + (oq + o4 + o));
        wm[slot] = *(const uint4 *)(wb + (om + o));
    };
    for (uint32_t k0 = 0; k0 < cnt; k0 += SG) {
        const uint32_t ng = min(SG, cnt - k0);
        // quantize the group's super-blocks: pass ps: token 4 ps + q, lane c16 its values 16 c16 ..; the loads of
        // two passes at a time, or of two super-blocks where one pass holds every token
        const uint32_t two = T <= 4u && !norm ? 1u : 0u;
        for (uint32_t kk = 0; kk < ng && (r0 == 0u || !keep); kk += 1u + two) {
            const uint32_t ln = mr_again(lane), c16 = ln & 15u, q = ln >> 4;
            const uint32_t xo = 256u * (w + 16u * (k0 + kk)) + 16u * c16;
            float4 pv[4];
            if (norm) {
                const float * pl = a.pw ? a.pw : a.x;             // without MUL: a valid address, unused
#pragma unroll
                for (int e = 0; e < 4; ++e) pv[e] = *(const float4 *)(pl + xo + 4 * e);
            }
            for (uint32_t p0 = 0; p0 < TP && 4u * p0 < T; p0 += 2u) {
                float4 xv[2][4];
#pragma unroll
                for (uint32_t e2 = 0; e2 < 2u; ++e2) {
                    const uint32_t t = min(4u * (p0 + (two ? 0u : e2)) + q, T - 1u);
                    const float * xp = a.x + (size_t)(t0 + t) * a.x_stride + xo + (two ? 4096u * min(e2, ng - 1u - kk) : 0u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) xv[e2][e] = *(const float4 *)(xp + 4 * e);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (uint32_t e2 = 0; e2 < 2u; ++e2) {
                    const uint32_t t = 4u * (p0 + (two ? 0u : e2)) + q;
                    if (two ? kk + e2 >= ng : 4u * (p0 + e2) >= T) break;   // uniform
                    uint8_t * sx = s_x + (kk + (two ? e2 : 0u)) * X::kBytes;
                    if (norm) {
                        const float sc = mr_bcast(scale, min(t, T - 1u));
                        if (!prep_norm_apply_fast(xv[e2], sc, pv, a.pw != nullptr)) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                xv[e2][e] = prep_norm_apply(xv[e2][e], sc, pv[e], a.pw != nullptr);
                                __builtin_amdgcn_sched_barrier(0);   // fewer registers in the rare path
                            }
                        }
                    }
                    float d;
                    int s16;
                    bool tiny;
                    const uint4 qq = qact_a256_row(xv[e2], &d, &s16, &tiny);
                    const int s32 = s16 + dpp_i<kDppXor1>(s16);   // sum of the 32 quants of a sub-block
                    *(uint4 *)(sx + kXq4Stride * t + 16u * c16) = qq;
                    if ((c16 & 1u) == 0u) {
                        const int bh = (s32 + 32) >> 6;
                        const v2h_r hl = { (_Float16)bh, (_Float16)(s32 - 64 * bh) };
                        *(uint32_t *)(sx + X::kQ + 32u * t + 2u * c16) = __builtin_bit_cast(uint32_t, hl);
                    }
                    if (c16 == 0u) *(float *)(sx + X::kQ + X::kS + 4u * t) = d;
                    slow = slow || __ballot(tiny) != 0ull;        // wave-uniform, sticky
                }
            }
        }
        mr_wave_sync();
#pragma unroll
        for (int i = 0; i < RD; ++i) load_w(i, i, k0);
        for (uint32_t kk = 0; kk < ng; ++kk) {
            const uint8_t * sx = s_x + kk * X::kBytes;
            const uint32_t t = c16 & (TT - 1u);                   // tokens beyond 4 TP: a copy, not stored
            const uint8_t * xr = sx + kXq4Stride * t + 64u * (q >> 1) + 16u * (q & 1u);
            v4i_r A[2][2];
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int n = 0; n < 2; ++n) A[s][n] = *(const v4i_r *)(xr + 128 * s + 32 * n);
            const uint2 bs = *(const uint2 *)(sx + X::kQ + 32u * t + 8u * q);
            const uint4 bs4 = make_uint4(bs.x, bs.y, 0u, 0u);
            const v8h_r Ab = __builtin_bit_cast(v8h_r, bs4);
            const float4 dx = *(const float4 *)(sx + X::kQ + X::kS + 16u * (q & (TT / 4u - 1u)));
            const float dxs[4] = { dx.x, dx.y, dx.z, dx.w };
            const uint32_t k = k0 + kk, kn = k0 + min(kk + 1u, ng - 1u);
#pragma unroll
            for (int i = 0; i < NTL; ++i) {
                constexpr uint32_t m4 = 0x0F0F0F0Fu;
                auto bmul = [](uint32_t v, uint32_t f) -> int {   // bytewise q f <= 105
                    return (int)__builtin_bit_cast(uint32_t, __builtin_bit_cast(v2u_r, v) * (v2u_r){ (unsigned short)f, (unsigned short)f });
                };
                const int sl = i % RD;
                const uint4 mt = wm[sl];
                v4i_r ia = {}, ib = {};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const uint4 v = s ? w1[sl] : w0[sl];
                    const uint32_t ws[4] = { v.x, v.y, v.z, v.w };
                    const uint32_t wd = s ? mt.z : mt.y;
                    const uint32_t sc0 = __builtin_amdgcn_ubfe(wd, 16u * (q >> 1), 6), sc1 = __builtin_amdgcn_ubfe(wd, 16u * (q >> 1) + 8u, 6);
                    v4i_r la, lb, ha, hb;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t lo = ws[e] & m4, hi = (ws[e] >> 4) & m4;
                        la[e] = bmul(lo, sc0 >> 3);
                        lb[e] = bmul(lo, sc0 & 7u);
                        ha[e] = bmul(hi, sc1 >> 3);
                        hb[e] = bmul(hi, sc1 & 7u);
                    }
                    ia = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[s][0], la, ia, 0, 0, 0);
                    ib = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[s][0], lb, ib, 0, 0, 0);
                    ia = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[s][1], ha, ia, 0, 0, 0);
                    ib = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[s][1], hb, ib, 0, 0, 0);
                }
                // the mins of sub-blocks 2 q and 2 q + 1
                const uint32_t wd = q < 2u ? mt.y : mt.z;
                const uint32_t m0 = __builtin_amdgcn_ubfe(wd, 16u * (q & 1u) + 6u, 2) | (__builtin_amdgcn_ubfe(mt.w, 8u * q, 4) << 2);
                const uint32_t m1 = __builtin_amdgcn_ubfe(wd, 16u * (q & 1u) + 14u, 2) | (__builtin_amdgcn_ubfe(mt.w, 8u * q + 4u, 4) << 2);
                v8h_r mb = {};
                mb[0] = (_Float16)(unsigned short)(m0 << 6);
                mb[1] = (_Float16)(unsigned short)m0;
                mb[2] = (_Float16)(unsigned short)(m1 << 6);
                mb[3] = (_Float16)(unsigned short)m1;
                v4f_r ms = {};
                ms = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ab, mb, ms, 0, 0, 0);
                const float d = h2f_fast(mt.x & 0xFFFFu), dm = h2f_fast(mt.x >> 16);
                if (__builtin_expect(!slow, 1)) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float tt = (d * dxs[r]) * (float)((ia[r] << 3) + ib[r]) - (dm * dxs[r]) * ms[r];
                        p[i][r] = p[i][r] + tt;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float tt = ssub(smul(smul(d, dxs[r]), i2f((ia[r] << 3) + ib[r])), smul(smul(dm, dxs[r]), ms[r]));
                        p[i][r] = sadd(p[i][r], tt);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                load_w(sl, (uint32_t)(i + RD < NTL ? i + RD : i + RD - NTL), i + RD < NTL ? k : kn);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    }
    if (lane == 0u) s_slow[w] = slow ? 1 : 0;
    mr_tree_store<NTL>(a, p, (float *)(lds + sp_off), s_slow, t0, T, row_lo, R, r0, w);
    }
}

// ---- Q8_0 -----------------------------------------------------------------------------------------
// Two blocks of the partial and a tile at a time: lane quarter q holds the row's half q mod 2 of block
// k + q / 2; the activations of the one block with zeros in the other's quarters give each block's sums. The
// A32 scales are fp16 values, so the plain operations are the rule's.
template <int TP>
struct MrX8 {                                                     // LDS of one quantized block of 4 TP tokens: [half][token][16 B], scales
    static constexpr uint32_t TT = 4u * TP, kH = 16u * TT, kBytes = 2u * kH + 4u * TT;
    static constexpr uint32_t kBlocks = TP == 2 ? 32u : 16u;      // blocks a wave holds at once (9216 bytes)
};

template <int TP, int NTL>
__global__ __launch_bounds__(1024) void k_mr_q80(MvArgs a, uint32_t tsh, uint32_t sp_off) {
    const uint32_t t0 = blockIdx.y * tsh, T = min(a.T - t0, tsh);  // the workgroup's tokens
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ float s_half[32];
    __shared__ int s_slow[kMrWaves];
    using X = MrX8<TP>;
    constexpr uint32_t TT = X::TT;
    constexpr int RD = NTL >= 2 ? 2 : 1;
    const WGeom g = wgeom(a.N, a.K >> 5, a.rb, false);
    const uint32_t lane = __lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cnt = wl_count(g, w);
    const uint32_t B = blockIdx.x, row_lo = B * g.rb, R = wl_rows(g, B);
    const uint32_t SG = min(g.q + (g.rem ? 1u : 0u), X::kBlocks);
    uint8_t * s_x = lds + (size_t)w * SG * X::kBytes;
    const uint8_t * wb = a.w + (size_t)B * g.bstride;
    const uint32_t R16 = 16u * R;
    const bool norm = a.prep == kPrepNorm;
    const bool keep = sp_off != 0u;
    const uint32_t lt = T <= 2u ? 1u : (T <= 4u ? 2u : 3u);
    if (lane == 0u) s_slow[w] = 0;
    const float scale = norm ? mr_norm_scales(a, t0, T, w, lane, s_half) : 0.0f;

    for (uint32_t r0 = 0; r0 < R; r0 += 16u * NTL) {
    const uint32_t lc = mr_again(lane), c16 = lc & 15u, q = lc >> 4;
    float p[NTL][4];
#pragma unroll
    for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) p[i][r] = 0.0f;
    if (cnt > 0u) {
    const uint32_t oh = (q & 1u) * g.nb * R16, om = 2u * g.nb * R16;
    uint4 wq[RD];
    uint32_t wd0[RD], wd1[RD];
    auto load_w = [&](int slot, uint32_t i, uint32_t k) {         // ring slot <- tile i of blocks k, k + 1 (clamped)
        const uint32_t s0 = wl_slot(g, w, k), s1 = wl_slot(g, w, min(k + 1u, cnt - 1u)), row = min(r0 + 16u * i + c16, R - 1u);
        wq[slot] = *(const uint4 *)(wb + (oh + (q < 2u ? s0 : s1) * R16 + 16u * row));
        wd0[slot] = *(const uint16_t *)(wb + (om + 2u * (s0 * R + row)));
        wd1[slot] = *(const uint16_t *)(wb + (om + 2u * (s1 * R + row)));
    };
    for (uint32_t k0 = 0; k0 < cnt; k0 += SG) {                   // SG is even or covers every block of the wave
        const uint32_t ng = min(SG, cnt - k0);
        // quantize: 8 lanes per (token, block): 1 << lt tokens of 8 >> lt blocks at a time, four times; then the tokens from 8 on
        const uint32_t nb8 = 8u >> lt;
        for (uint32_t kk = 0; kk < ng && (r0 == 0u || !keep); kk += 4u * nb8) {
            for (uint32_t p0 = 0; p0 < T; p0 += 8u) {
                const uint32_t ln = mr_again(lane), l8 = ln & 7u, b8 = (ln >> 3) >> lt, t = p0 + ((ln >> 3) & ((1u << lt) - 1u));
                const float * xt = a.x + (size_t)(t0 + min(t, T - 1u)) * a.x_stride + 4u * l8, * pt = (a.pw ? a.pw : a.x) + 4u * l8;
                const float sc = norm ? mr_bcast(scale, min(t, T - 1u)) : 0.0f;
                uint8_t * st = s_x + (l8 >> 2) * X::kH + 16u * t + 4u * (l8 & 3u), * sd = s_x + 2u * X::kH + 4u * t;
                // step b's block of this lane; the last blocks of a group store the same bytes again
                auto blk = [&](uint32_t b) { return min(kk + b * nb8 + b8, ng - 1u); };
                float4 xv[4], pv[4];
#pragma unroll
                for (uint32_t b = 0; b < 4u; ++b) {
                    const uint32_t xo = 32u * (w + 16u * (k0 + blk(b)));
                    xv[b] = *(const float4 *)(xt + xo);
                    if (norm) pv[b] = *(const float4 *)(pt + xo);
                }
                __builtin_amdgcn_sched_barrier(0);
                uint32_t qq[4];
                float D;
                if (__builtin_expect((!norm || prep_norm_apply_fast(xv, sc, pv, a.pw != nullptr)) && qact_a32_lane4_fast(xv, qq, &D), 1)) {
#pragma unroll
                    for (uint32_t b = 0; b < 4u; ++b) {
                        *(uint32_t *)(st + blk(b) * X::kBytes) = qq[b];
                        if (l8 == b) *(float *)(sd + blk(b) * X::kBytes) = D;
                    }
                } else {                                          // one block at a time, x read again
#pragma unroll 1
                    for (uint32_t b = 0; b < 4u; ++b) {
                        const uint32_t xo = 32u * (w + 16u * (k0 + blk(b)));
                        float4 v = *(const float4 *)(xt + xo);
                        if (norm) v = prep_norm_apply(v, sc, *(const float4 *)(pt + xo), a.pw != nullptr);
                        const uint32_t qb = qact_a32_lane(v, &D);
                        *(uint32_t *)(st + blk(b) * X::kBytes) = qb;
                        if (l8 == 0u) *(float *)(sd + blk(b) * X::kBytes) = D;
                    }
                }
            }
        }
        mr_wave_sync();
#pragma unroll
        for (int i = 0; i < RD; ++i) load_w(i, i, k0);
        for (uint32_t kk = 0; kk < ng; kk += 2u) {
            const bool two = kk + 1u < ng;                        // wave-uniform
            const uint8_t * x0 = s_x + kk * X::kBytes, * x1 = s_x + min(kk + 1u, ng - 1u) * X::kBytes;
            const uint32_t t = c16 & (TT - 1u);
            const v4i_r v = *(const v4i_r *)((q < 2u ? x0 : x1) + (q & 1u) * X::kH + 16u * t);
            v4i_r A0, A1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                A0[e] = q < 2u ? v[e] : 0;
                A1[e] = q < 2u ? 0 : v[e];
            }
            const uint32_t dxo = 2u * X::kH + 16u * (q & (TT / 4u - 1u));
            const float4 d0 = *(const float4 *)(x0 + dxo), d1 = *(const float4 *)(x1 + dxo);
            const float dx0[4] = { d0.x, d0.y, d0.z, d0.w }, dx1[4] = { d1.x, d1.y, d1.z, d1.w };
            const uint32_t k = k0 + kk, kn = kk + 2u < ng ? k + 2u : k;
#pragma unroll
            for (int i = 0; i < NTL; ++i) {
                const int sl = i % RD;
                const v4i_r W = { (int)wq[sl].x, (int)wq[sl].y, (int)wq[sl].z, (int)wq[sl].w };
                v4i_r i0 = {}, i1 = {};
                i0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A0, W, i0, 0, 0, 0);
                i1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A1, W, i1, 0, 0, 0);
                const float e0 = h2f_fast(wd0[sl]), e1 = h2f_fast(wd1[sl]);
                __builtin_amdgcn_sched_barrier(0);
                load_w(sl, (uint32_t)(i + RD < NTL ? i + RD : i + RD - NTL), i + RD < NTL ? k : kn);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < 4; ++r) p[i][r] = p[i][r] + (e0 * dx0[r]) * (float)i0[r];
                if (two) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) p[i][r] = p[i][r] + (e1 * dx1[r]) * (float)i1[r];
                }
            }
        }
    }
    }
    mr_tree_store<NTL>(a, p, (float *)(lds + sp_off), s_slow, t0, T, row_lo, R, r0, w);
    }
}

}  // namespace tsr

// One workgroup per row block and share of at most 15 tokens (even shares). A wave holds the results of at most
// 4 tiles of 16 rows (Q4_K: 2, its unpacked weights need the registers; with 4 the 28672x4096 GLU takes 36 us
// instead of 28); a row block of more rows runs in chunks. The quantized x stays in LDS for all of them
// (keep: sp_off, the offset of the tree's LDS behind it) when the wave's blocks fit at once and the tree's LDS
// beside them; otherwise the two share the LDS and every chunk quantizes again. Up to 8 tokens, or up to 15
// (twice the LDS per block).
template <int TP, int NTL>
static void launch_mr(const tsr::MvArgs & a, bool q4k, uint32_t tsh, uint32_t sp_off, dim3 grid, size_t lds, hipStream_t s) {
    if (q4k) {
        if constexpr (NTL <= 2) hipLaunchKernelGGL((tsr::k_mr_q4k<TP, NTL>), grid, dim3(1024), lds, s, a, tsh, sp_off);
    } else {
        hipLaunchKernelGGL((tsr::k_mr_q80<TP, NTL>), grid, dim3(1024), lds, s, a, tsh, sp_off);
    }
}
template <int TP>
static void launch_mr_t(const tsr::MvArgs & a, bool q4k, uint32_t tsh, hipStream_t s) {
    const uint32_t nb = a.K / (q4k ? 256u : 32u), kx = (nb + 15u) / 16u;
    const uint32_t tiles = (std::min(a.rb, a.N) + 15u) / 16u, ntl = tiles <= 1u ? 1u : (tiles <= 2u || q4k ? 2u : 4u);
    const uint32_t most = q4k ? tsr::MrX4<TP>::kSlots : tsr::MrX8<TP>::kBlocks;
    const size_t x = (size_t)tsr::kMrWaves * std::min(kx, most) * (q4k ? tsr::MrX4<TP>::kBytes : tsr::MrX8<TP>::kBytes);
    const size_t tree = (size_t)16384u * ntl;
    const bool keep = tiles > ntl && kx <= most && x + tree <= 159u * 1024u;
    const uint32_t sp_off = keep ? (uint32_t)x : 0u;
    const size_t lds = keep ? x + tree : std::max(x, tree);
    const dim3 grid((a.N + a.rb - 1u) / a.rb, (a.T + tsh - 1u) / tsh);
    switch (ntl) {
        case 1: launch_mr<TP, 1>(a, q4k, tsh, sp_off, grid, lds, s); break;
        case 2: launch_mr<TP, 2>(a, q4k, tsh, sp_off, grid, lds, s); break;
        default: launch_mr<TP, 4>(a, q4k, tsh, sp_off, grid, lds, s); break;
    }
}

int tsr_launch_mr(const tsr::MvArgs & a, bool q4k, hipStream_t s) {
    if (a.T < 2u || a.isums != nullptr || (a.prep != tsr::kPrepNone && a.K > 8192u)) return -2;
    if (a.glu && ((a.rb & 1u) || (a.N & 1u) || a.add != nullptr || a.acc)) return -2;
    const uint32_t n = (a.T + 14u) / 15u, tsh = (a.T + n - 1u) / n;
    if (tsh <= 8u) launch_mr_t<2>(a, q4k, tsh, s);
    else launch_mr_t<4>(a, q4k, tsh, s);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}
