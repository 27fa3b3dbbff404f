// k_attn.hip -- FLASH_ATTN_EXT over the q8_0 KV cache on gfx950, bit-exact to the reference's
// composite flash attention (tsr_ref_fa, sw/sim/tsr_ref_at.c:774-860; AT section 6.6) in its fixed
// configuration C = 4 channels, PCAP = 9344, T_MAX = 1 (one query row per tile).
//
// The host planner cuts every token's visible cells into chunks of NCG groups (16 cells each); the
// reference processes chunk after chunk: scores (ATTQK, MAXOUT), p = EXP((s - m) scale) with the
// chunk maximum m (ASMAX), per channel c (groups u = c mod 4) the block-float P.V over segments of
// 4 of its groups (ATTPV with LSUM), then CTREE over the 4 channel partials and the online merge
// (AMERGE), and finally O / l (ANORM). On the GPU the chunks of a token and the channels of a chunk
// are independent until the merge, so they run as parallel workgroups (split-K); only the f32 steps
// that the reference orders are kept in its order:
//   k_fa_qk     QACT of the query heads, scores of a 256-cell tile of one chunk for the query heads
//               of one KV head, and the tile's maxima (MAXT is an order-free total-order maximum)
//   k_fa_pv     one (chunk, channel, KV head, 64-value slice): EXP, block float per segment, the f32
//               segment sums in segment order, the segment row-sums (LSUM)
//   k_fa_merge  one (token, KV head, slice): CTREE of the channels, the online merge in chunk order,
//               ANORM
//
// Block float (AT 6.4; sw/sim/tsr_ref_at.c:380-488): in a segment every weight w = p dV is scaled
// to an integer W = RNE(w 2^(23 - E_S)) (|W| <= 2^24) and A = sum W q is exact. W is split into four
// balanced base-256 digits d_k in [-128, 127] (W = sum d_k 256^k), so A = sum_k 256^k (sum d_k q)
// runs on the int8 matrix core with exact int32 digit sums (|sum| <= 64 * 128 * 128).
//
// Subnormal operands. A score is a tree sum of terms (dK Dx) f32(isum) with fp16 dK and Dx: every
// term is 0 or a multiple of 2^-48 in magnitude, so is every sum, and a GENERAL mask is added with
// the full f32 rule: no score is subnormal. Maxima are scores or the floor; EXPK values,
// block-float values and the results of rule operations are never subnormal either. The f32 steps
// after the scores therefore use the rule without the input DAZ (sadd_n / smul_n).
#include "expk.hpp"
#include "glue.hpp"
#include "kernels.hpp"
#include "kvstore.hpp"
#include "qact.hpp"
#include "fa_common.hpp"

#include <algorithm>

namespace tsr {

// ---------------------------------------------------------------------------------------------
// P.V: block (item * 4 + channel c, KV head g, group hg of 4 query heads x value part vh of VS); one
// wave per segment of the channel (4 of its groups = 64 cells). Each segment's results go to LDS; the f32 segment chain then runs in segment order.
// A block covers D / VS values of its heads (VS > 1 when the grid would not fill the chip: the
// value-independent EXP and LSUM work is then repeated per part, the value work is split).
//
// Phase A (lane = head row hr = lane / 16, 4 consecutive cells of the segment: group kk = (lane /
// 4) % 4, cells 4 (lane % 4) .. + 3): EXP of the scores, the weights w = p dV of the value blocks,
// and, over the 16 lanes of a head row (DPP), the segment's block-float exponent E_S per 64-value
// slice, the non-finite flags per block and LSUM. The block-float integers W = RNE(w 2^(23 - E_S))
// (|W| <= 2^24) are split into four balanced base-256 digits d_k in [-128, 127]: the bytes of
// (W + 0x80808080) ^ 0x80808080 (the offset makes every byte d_k + 128, the xor subtracts 128).
// The digits go to LDS as [block][head][digit][group][16 cells].
// Phase B (matrix core): A[h][v] = sum_cells W[h][cell] q[cell][v] = sum_k 256^k sum_cells d_k q is
// v_mfma_i32_16x16x64_i8 with rows (head, digit), columns 16 values and K the 64 cells; lane l then
// holds the four digit sums of head l / 16 and value l % 16 and forms RNE24(A) (digits_rne24).
// Every global load of the first batch is issued before the EXP work, so that a block waits for
// memory once.
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kPvWaves = kMaxSegments;                       // one a segment

// The P.V work of one block (chunk item, channel c, KV head g, head group hg, value part vh), shared by
// k_fa_pv (the item's scores in global memory). Lane = (head row hr, group kk of the segment, cell quad);
// one wave per segment.
template <int D, int VS>
struct PvBlock {
    static constexpr uint32_t DV = D / VS;                        // values of the block (>= 64)
    static constexpr uint32_t NBV = DV / 32;                      // their value blocks
    static constexpr uint32_t BB = 2;                             // blocks per batch: one 64-value slice (fewer registers: more waves per SIMD)
    static constexpr uint32_t NBT = NBV / BB;                     // batches
    static_assert(DV >= 64 && NBV % BB == 0, "value part");
    // the loads of one segment: scores, value scales and the value quants of a batch
    struct Loads {
        float4 sv;
        uint32_t mb[BB][2];                                       // block e: scales of cells 0, 1 | 2, 3
        int4 bq[2 * BB];
    };
    const FaArgs & a;
    const float * S;                                              // the scores of head h, cell j at S[j - s_off]
    uint32_t g, c, vh, lane, hr, kk, quad, u0, u_first, nu, nseg, vb0, nbk, s_off;
    bool head_ok;
    const uint16_t * vmeta;
    const uint8_t * vq;

    __device__ __forceinline__ PvBlock(const FaArgs & a_, const FaItem & it, uint32_t c_, uint32_t g_, uint32_t hg,
                                       uint32_t vh_, const float * S_, uint32_t s_off_ = 0u)
        : a(a_), S(S_), g(g_), c(c_), vh(vh_), s_off(s_off_) {
        lane = __lane_id();
        hr = lane >> 4;
        kk = (lane >> 2) & 3u;
        quad = lane & 3u;
        head_ok = 4u * hg + hr < a.G;
        u0 = it.u0;
        u_first = it.u0 + ((c + 4u - (it.u0 & 3u)) & 3u);
        const uint32_t u_end = it.u0 + it.n;
        nu = u_first < u_end ? (u_end - 1u - u_first) / 4u + 1u : 0u;
        nseg = (nu + 3u) / 4u;
        vb0 = vh * NBV;                                           // first value block of the part (in the head)
        nbk = a.E / 32u;                                          // value blocks of a cell
        vmeta = (const uint16_t *)a.vc.base;
        vq = a.vc.base + a.vc.quant_off;
    }

    __device__ __forceinline__ void load_scores(uint32_t seg, Loads & L) const {
        const uint32_t u = u_first + 4u * min(4u * seg + kk, nu - 1u);
        L.sv = *(const float4 *)(S + 16u * (u - u0) + 4u * quad - s_off);
    }

    __device__ __forceinline__ void loads(uint32_t seg, uint32_t vb, Loads & L, bool scores) const {
        const uint32_t gi = 4u * seg + kk;
        const uint32_t u = u_first + 4u * min(gi, nu - 1u);        // clamped: loads stay in the item
        if (scores) load_scores(seg, L);
        const uint16_t * vm = vmeta + ((size_t)u * nbk + (size_t)g * (D / 32u) + vb) * 16u + 4u * quad;
#pragma unroll
        for (uint32_t e = 0; e < BB; ++e) {                       // the 4 cells' scales of block e: 8 bytes
            const uint2 m2 = *(const uint2 *)(vm + (size_t)e * 16u);
            L.mb[e][0] = m2.x;
            L.mb[e][1] = m2.y;
        }
        const uint32_t uB = u_first + 4u * min(4u * seg + (lane >> 4), nu - 1u);
        const uint8_t * vqB = vq + ((size_t)uB * a.E + (size_t)g * D + 32u * vb + (lane & 15u)) * 16u;
#pragma unroll
        for (uint32_t t8 = 0; t8 < 2 * BB; ++t8) L.bq[t8] = *(const int4 *)(vqB + 256u * t8);
    }

    // The digits of the weights' integers W = RNE_int(w 2^(23 - es)) of the lane's 4 cells to LDS, for block e
    // and digit k in one word; the fences keep the wave's own LDS accesses in order.
    __device__ __forceinline__ void digits(const float (&w)[4][BB], int32_t es, uint8_t * dg) const {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (uint32_t e = 0; e < BB; ++e) {
            uint32_t P[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) P[i] = ((uint32_t)bf_int_n(w[i][e], es) + 0x80808080u) ^ 0x80808080u;   // byte k = digit k
            // transpose the 4 x 4 bytes: word k = digit k of cells 0..3
            const uint32_t lo01 = __builtin_amdgcn_perm(P[1], P[0], 0x05010400u);   // d0c0 d0c1 d1c0 d1c1
            const uint32_t lo23 = __builtin_amdgcn_perm(P[3], P[2], 0x05010400u);
            const uint32_t hi01 = __builtin_amdgcn_perm(P[1], P[0], 0x07030602u);   // d2c0 d2c1 d3c0 d3c1
            const uint32_t hi23 = __builtin_amdgcn_perm(P[3], P[2], 0x07030602u);
            const uint32_t q[4] = { __builtin_amdgcn_perm(lo23, lo01, 0x05040100u), __builtin_amdgcn_perm(lo23, lo01, 0x07060302u),
                                    __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), __builtin_amdgcn_perm(hi23, hi01, 0x07060302u) };
#pragma unroll
            for (int k = 0; k < 4; ++k)
                *(uint32_t *)(dg + (((e * 4u + hr) * 4u + (uint32_t)k) * 4u + kk) * 16u + 4u * quad) = q[k];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // One segment (L holds its loads): EXP, LSUM, the block-float weights, their digits and the
    // matrix-core digit sums; the segment's results go to s_c [seg][4 heads][DV] and s_l [seg][4 heads].
    // The common case of a batch (wave-uniform: every p and value scale finite, every head row's largest
    // weight 0 or in [2^-102, 2^106)) needs no flag and no flush: with the segment exponent E_S >= -102 a
    // subnormal weight rounds to W = 0 as the flushed one does, and with |A| in [1, 2^45) the scaled result
    // is a normal number for E_S in -102 .. 105. The general form runs otherwise.
    // Returns whether every batch was the common case.
    __device__ __forceinline__ bool segment(uint32_t seg, Loads & L, float m, const ExpkNeg & en,
                                            const double * s_td, float * s_c, float * s_l, uint8_t * dg) const {
        bool common = true;
        // ---- phase A: lane = (head row, 4 cells) ----------------------------------------------
        const bool cv = 4u * seg + kk < nu;
        const float ss[4] = { L.sv.x, L.sv.y, L.sv.z, L.sv.w };
        float pz[4];
        uint32_t pm = 0u;                                          // largest p (not negative; NaN above all)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // EXPK results are zero, normal or NaN (never subnormal)
            const float ez = expk_neg_diff(ss[i], m, a.scale, en, s_td);   // straight-line, then the select
            pz[i] = (cv && head_ok) ? ez : 0.0f;
            pm = max(pm, fb(pz[i]));
        }
        const bool pfin = __ballot(pm >= 0x7F800000u) == 0ull;
        // LSUM of the segment (AT 6.5): block float of its p values; NaN when one is (EXPK of a value <= 0 is
        // at most 1, so a p that is not finite is NaN)
        if (vh == 0u) {
            pm = row16_umax(pm);
            const int32_t pe = (int32_t)(pm >> 23);                // the largest exponent field (255: the sum is not used)
            int32_t lsum = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) lsum += bf_int_n(pm >= 0x7F800000u ? 0.0f : pz[i], pe - 127);
            lsum = row16_isum(lsum);
            if ((lane & 15u) == 0u)
                s_l[seg * 4u + hr] = pe == 255 ? bf(kNaN) : (pe == 0 ? 0.0f : bf_scale((float)lsum, pe - 150));
        }

#pragma unroll
        for (uint32_t bt = 0; bt < NBT; ++bt) {                    // BB value blocks (32 BB values) at a time
            const uint32_t vb = vb0 + bt * BB;
            if (bt > 0u) loads(seg, vb, L, false);
            static_assert(BB == 2, "one 64-value slice a batch");
            const uint32_t chk = ((L.mb[0][0] & 0x7C007C00u) + 0x04000400u) | ((L.mb[0][1] & 0x7C007C00u) + 0x04000400u) |
                                 ((L.mb[1][0] & 0x7C007C00u) + 0x04000400u) | ((L.mb[1][1] & 0x7C007C00u) + 0x04000400u);
            float wf[4][BB], mx = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (uint32_t e = 0; e < BB; ++e)
                    wf[i][e] = pz[i] * h2f_fast((L.mb[e][i >> 1] >> (16u * (i & 1u))) & 0xFFFFu);
                mx = __builtin_fmaxf(mx, __builtin_fmaxf(__builtin_fabsf(wf[i][0]), __builtin_fabsf(wf[i][1])));
            }
            const uint32_t mr = row16_umax(fb(mx));                // largest |w| of the head row (not negative)
            const int32_t ef = (int32_t)(mr >> 23) - 127;
            const bool okf = pfin && (chk & 0x80008000u) == 0u && (mr == 0u || (ef >= -102 && ef <= 105));
            if (__builtin_expect(__ballot(!okf) == 0ull, 1)) {
                digits(wf, ef, dg);
#pragma unroll
                for (uint32_t e = 0; e < BB; ++e) {
                    const v4i_fa Aop = *(const v4i_fa *)(dg + ((e * 16u + (lane & 15u)) * 4u + (lane >> 4)) * 16u);
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int4 bq = L.bq[2 * e + half];
                        const v4i_fa Bop = { bq.x, bq.y, bq.z, bq.w };
                        v4i_fa acc = { 0, 0, 0, 0 };
                        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop, Bop, acc, 0, 0, 0);
                        s_c[(seg * 4u + hr) * DV + 32u * (bt * BB + e) + 16u * (uint32_t)half + (lane & 15u)] =
                            __builtin_ldexpf(digits_rne24(acc), ef - 23);
                    }
                }
                continue;
            }
            common = false;
            // weights of the 4 cells for the BB blocks: w = p dV, a subnormal product flushed to zero
            float w[4][BB];
            uint32_t ex[BB / 2], nfm = 0u;
#pragma unroll
            for (uint32_t sa = 0; sa < BB / 2; ++sa) ex[sa] = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool live = (fb(pz[i]) & 0x7FFFFFFFu) != 0u;
#pragma unroll
                for (uint32_t e = 0; e < BB; ++e) {
                    const uint32_t dv = (L.mb[e][i >> 1] >> (16u * (i & 1u))) & 0xFFFFu;
                    const float we = live ? pz[i] * h2f_fast(dv) : 0.0f;
                    const uint32_t f = f_field(we);
                    nfm |= (f == 255u ? 1u : 0u) << e;
                    w[i][e] = f == 0u ? 0.0f : we;
                    ex[e >> 1] = max(ex[e >> 1], f == 255u ? 0u : f);
                }
            }
            int32_t es[BB / 2];
            bool any[BB / 2];
#pragma unroll
            for (uint32_t sa = 0; sa < BB / 2; ++sa) {
                const uint32_t ef = row16_umax(ex[sa]);
                any[sa] = ef != 0u;
                es[sa] = (int32_t)ef - 127;
            }
            const uint32_t badm = row16_or(nfm);
#pragma unroll
            for (uint32_t e = 0; e < BB; ++e)
                if (!any[e >> 1] || ((badm >> e) & 1u) != 0u) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[i][e] = 0.0f;
                }
            digits(w, es[0], dg);
            // ---- phase B: 2 BB tiles of 16 values; lane = (head row l / 16 of the result, value l % 16)
#pragma unroll
            for (uint32_t e = 0; e < BB; ++e) {
                // A operand: row l % 16 = (head, digit), K = the 16 cells of group l / 16
                const v4i_fa Aop = *(const v4i_fa *)(dg + ((e * 16u + (lane & 15u)) * 4u + (lane >> 4)) * 16u);
                const bool bad = ((badm >> e) & 1u) != 0u;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int4 bq = L.bq[2 * e + half];
                    const v4i_fa Bop = { bq.x, bq.y, bq.z, bq.w };
                    v4i_fa acc = { 0, 0, 0, 0 };
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop, Bop, acc, 0, 0, 0);
                    const float cval = bad ? bf(kNaN) : (any[e >> 1] ? bf_scale(digits_rne24(acc), es[e >> 1] - 23) : 0.0f);
                    s_c[(seg * 4u + hr) * DV + 32u * (bt * BB + e) + 16u * (uint32_t)half + (lane & 15u)] = cval;
                }
            }
        }
        return common;
    }

    // After a block barrier: the segment chains in order (AT 6.4 O, 6.5 l) -> the channel partials.
    // Thread = (head row, value of the part). common: every batch of every segment was the common case, so
    // every result is a multiple of 2^(E_S - 23) >= 2^-125, and so is every rounded sum of them: none is
    // subnormal, and the chain needs no FTZ.
    __device__ __forceinline__ void chains(uint32_t item, uint32_t hg, const float * s_c, const float * s_l,
                                           bool common) const {
        const uint32_t G = a.G, nh = a.n_head;
        for (uint32_t idx = threadIdx.x; idx < 4u * DV; idx += blockDim.x) {
            const uint32_t r4 = idx / DV, v = idx % DV, hi2 = 4u * hg + r4;
            if (hi2 >= G) continue;
            const uint32_t h2 = g * G + hi2;
            float O = 0.0f;
            if (__builtin_expect(common, 1)) {
                for (uint32_t seg = 0; seg < nseg; ++seg) O = O + s_c[(seg * 4u + r4) * DV + v];
            } else {
                for (uint32_t seg = 0; seg < nseg; ++seg) O = sadd_z(O, s_c[(seg * 4u + r4) * DV + v]);
            }
            const size_t slot = ((size_t)item * 4u + c) * nh + h2;
            a.OP[slot * D + vh * DV + v] = canon(O);
            if (vh == 0u && v == 0u) {
                float l = 0.0f;
                for (uint32_t seg = 0; seg < nseg; ++seg) l = l + s_l[seg * 4u + r4];   // see ctree4_l
                a.LP[slot] = l;
            }
        }
    }
};

// ---------------------------------------------------------------------------------------------
// scores: block (tile, KV head g), thread = one cell of the tile. The block quantizes the query
// values of the KV head's G heads (QACT A32: its 32-blocks never cross a head, so they are the
// blocks of the whole query row) while the K rows of its cells load.
// ---------------------------------------------------------------------------------------------
// The work list is inline in the kernel arguments (INL, decode) or in device memory: a compile-time
// choice, so that reading an item is never a branch around a load.
template <bool INL>
__device__ __forceinline__ FaItem fa_item(const FaArgs & a, const FaPlan & p, uint32_t i) {
    if constexpr (INL) return p.items[i];
    else return a.items[i];
}

// LDS of the score kernel: the query quants and scales, the per-wave maxima and (ROPE) the new k row.
__host__ __device__ inline uint32_t fa_qk_lds(uint32_t G, uint32_t D, bool rope) {
    const uint32_t b = G * D + 4u * G * (D / 32u) + 16u * G;
    return rope ? ((b + 15u) & ~15u) + D + D / 8u : b;
}
// ROPE (T == 1, D <= 128, (G + 2) D <= 1024): the block also rotates the query heads (rope4, angles
// per lane by rope_cs_lane) before their QACT, rotates and QACTs the token's k row of head g and
// QACTs its v row (threads after the query slots, A32 as SET_ROWS_KV); the thread of the new cell
// scores with that fresh k row, and the first block of each KV head stores the k and v rows in the
// caches -- ROPE, SET_ROWS_KV and the scores in one launch.
template <int D, bool INL, bool ROPE>
__global__ __launch_bounds__(256) void k_fa_qk(FaArgs a, FaPlan p) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr uint32_t NBD = D / 32u;                             // blocks per head
    constexpr bool KREG = D <= 128;                                // K row of the cell kept in registers
    static_assert(!ROPE || KREG, "the fused ROPE keeps the K rows in registers");
    const uint32_t tt = blockIdx.x % p.maxtiles;
    const FaItem it = fa_item<INL>(a, p, blockIdx.x / p.maxtiles);
    if (tt >= it.ntiles) return;                                  // the item has fewer tiles (block-uniform)
    const uint32_t g = blockIdx.y, G = a.G;
    int8_t * s_q = (int8_t *)lds;                                 // G*D quants of the KV head's query heads
    float * s_dx = (float *)(lds + G * D);                        // G*D/32 scales
    uint32_t * s_red = (uint32_t *)(s_dx + G * NBD);              // 4 waves x G maxima (keys)
    int8_t * s_kq = (int8_t *)lds + ((G * D + 4u * G * NBD + 16u * G + 15u) & ~15u);   // ROPE: the new k row of
    float * s_kd = (float *)(s_kq + D);                           //       head g (D quants) and its D/32 scales
    const int lane = (int)__lane_id(), wave = (int)(threadIdx.x >> 6);
    int32_t pos = 0;
    int64_t cell64 = -1;
    if constexpr (ROPE) {                                         // scalar loads: not behind the vector loads
        if (a.rtab == nullptr) pos = *a.pos;
        cell64 = *a.cell;
    }

    const uint32_t n16 = 16u * it.n, j = 256u * tt + threadIdx.x;
    const bool in = j < n16;
    const uint32_t cell = 16u * it.u0 + j;
    const uint32_t ng = (a.kc.kv_size + 15u) / 16u;
    const uint32_t u = min(cell >> 4, ng - 1u), rr = cell & 15u;  // clamped: loads stay inside the plane
    const bool vis = in && (it.general || (j >= it.c_lo && j < it.c_hi));
    const uint32_t E = a.E, nbk = E / 32u;
    const uint16_t * kmeta = (const uint16_t *)a.kc.base + ((size_t)u * nbk + (size_t)g * NBD) * 16u + rr;
    const uint8_t * kq = a.kc.base + a.kc.quant_off + (size_t)u * 16u * E + (size_t)rr * 16u;
    const uint32_t ci0 = g * D / 16u;                             // first 16-byte chunk of the head

    // the query values of round 0 first (vector-memory counters retire in order: the QACT then waits
    // for them only, not for the K rows)
    const float * qrow = a.q + (size_t)it.t * a.q_stride + (size_t)g * G * D;
    const uint32_t nslot = G * D / 4u;                             // 8 lanes per 32-block
    const uint32_t half = a.n_dims / 2u;
    // ROPE: threads nslot .. nslot + D/4 - 1 hold the k row of head g, the next D/4 its v row
    const uint32_t kslot = threadIdx.x - nslot, vslot = kslot - D / 4u;
    const bool is_k = ROPE && threadIdx.x >= nslot && kslot < D / 4u, is_v = ROPE && !is_k && threadIdx.x >= nslot &&
                                                                             vslot < D / 4u;
    const float * src = a.q + (size_t)a.n_head * D + (size_t)g * D + (is_v ? E + 4u * vslot : 4u * (is_k ? kslot : 0u));
    const uint32_t jq = 4u * min(threadIdx.x, nslot - 1u);        // first query value of the thread
    const float4 qv0 = (ROPE && threadIdx.x >= nslot) ? *(const float4 *)src : *(const float4 *)(qrow + jq);
    float4 qpart = qv0;                                           // ROPE NEOX: the values half away
    // value index in the head of a rotated thread (q or k); D for the others (nothing to rotate)
    const uint32_t jh0 = threadIdx.x < nslot ? jq % D : (is_k ? 4u * kslot : D);
    if constexpr (ROPE) {
        if (a.neox && jh0 < a.n_dims) {                           // the partner lies in the same head row
            const int32_t dj = jh0 < half ? (int32_t)half : -(int32_t)half;
            qpart = *(const float4 *)((threadIdx.x < nslot ? qrow + jq : src) + dj);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    int4 kr[KREG ? 2 * NBD : 1];
    uint32_t km[NBD];
#pragma unroll
    for (uint32_t kb = 0; kb < NBD; ++kb) km[kb] = kmeta[(size_t)kb * 16u];
    if constexpr (KREG) {
#pragma unroll
        for (uint32_t c = 0; c < 2 * NBD; ++c) kr[c] = *(const int4 *)(kq + (size_t)(ci0 + c) * 256u);
    }
    __builtin_amdgcn_sched_barrier(0);

    auto qact_slot = [&](uint32_t slot, const float4 v) {
        float Dq;
        const uint32_t qq = qact_a32_lane(v, &Dq);
        if (slot < nslot) {
            *(uint32_t *)(s_q + 4u * slot) = qq;
            if ((lane & 7) == 0) s_dx[slot >> 3] = Dq;
        }
    };
    if constexpr (ROPE) {
        float c_l, s_l;
        if (a.rtab != nullptr) {                                  // the token's table (block-uniform)
            const float2 cs = *(const float2 *)(a.rtab + 2u * min((uint32_t)lane, half - 1u));
            c_l = cs.x;
            s_l = cs.y;
        } else {
            rope_cs_lane(pos, half, a.ts, a.m, (uint32_t)lane, &c_l, &s_l);
        }
        // every lane runs rope4 (its table reads are cross-lane: a lane that skipped it would hide its
        // entries from the others); v lanes then keep their values (jh0 = D leaves them unrotated anyway)
        const float4 rot = rope4(qv0, qpart, jh0, a.n_dims, a.neox != 0u, c_l, s_l);
        const float4 r = is_v ? qv0 : rot;
        float Dq;
        const uint32_t qq = qact_a32_lane(r, &Dq);                // every lane (8-lane groups)
        if (threadIdx.x < nslot) {
            *(uint32_t *)(s_q + 4u * threadIdx.x) = qq;
            if ((lane & 7) == 0) s_dx[threadIdx.x >> 3] = Dq;
        } else if (is_k) {
            *(uint32_t *)(s_kq + 4u * kslot) = qq;
            if ((lane & 7) == 0) s_kd[kslot >> 3] = Dq;
        }
        const bool cell_ok = cell64 >= 0 && cell64 < (int64_t)a.kc.kv_size && cell64 < (int64_t)a.vc.kv_size;
        if (blockIdx.x == 0u) {                                   // the caches' copy of the new rows
            if (cell_ok && (is_k || is_v)) {
                KvArgs kv;                                        // per-lane choice of the plane, field by field
                kv.base = is_k ? a.kc.base : a.vc.base;
                kv.quant_off = is_k ? a.kc.quant_off : a.vc.quant_off;
                kv.E = a.kc.E;
                kv.kv_size = is_k ? a.kc.kv_size : a.vc.kv_size;
                kv_store_unit(kv, is_k ? 0u : 1u, (uint32_t)cell64, g * D + 4u * (is_k ? kslot : vslot), qq, Dq,
                              (lane & 7) == 0);
            }
            if (!cell_ok && threadIdx.x == 0u && g == 0u && a.bad != nullptr) *a.bad = 1;
        }
    } else {
        qact_slot(threadIdx.x, qv0);
        for (uint32_t s0 = blockDim.x; s0 < nslot; s0 += blockDim.x)   // G D > 1024 only
            qact_slot(s0 + threadIdx.x, *(const float4 *)(qrow + 4u * min(s0 + threadIdx.x, nslot - 1u)));
    }
    lds_barrier();                                                // the K rows stay in flight
    if constexpr (ROPE) {                                         // the new cell scores with the fresh k row
        if ((int64_t)cell == cell64 && in) {
#pragma unroll
            for (uint32_t c = 0; c < 2 * NBD; ++c) kr[c] = *(const int4 *)(s_kq + 16u * c);
#pragma unroll
            for (uint32_t kb = 0; kb < NBD; ++kb) km[kb] = f2h_exact(s_kd[kb]);
        }
    }

    float * S = a.S + (size_t)it.s_off * a.n_head;
    for (uint32_t i = 0; i < G; ++i) {
        const uint32_t h = g * G + i;
        float s = bf(kNegInf);
        if (vis) {
            float p[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) p[k] = 0.0f;
#pragma unroll
            for (uint32_t kb = 0; kb < NBD; ++kb) {
                int4 w0, w1;
                if constexpr (KREG) { w0 = kr[2 * kb]; w1 = kr[2 * kb + 1]; }
                else {
                    w0 = *(const int4 *)(kq + (size_t)(ci0 + 2 * kb) * 256u);
                    w1 = *(const int4 *)(kq + (size_t)(ci0 + 2 * kb + 1) * 256u);
                }
                const int4 * xq = (const int4 *)(s_q + (size_t)i * D + 32u * kb);
                const int4 x0 = xq[0], x1 = xq[1];
                int is = dot4(w0.x, x0.x, 0);
                is = dot4(w0.y, x0.y, is);
                is = dot4(w0.z, x0.z, is);
                is = dot4(w0.w, x0.w, is);
                is = dot4(w1.x, x1.x, is);
                is = dot4(w1.y, x1.y, is);
                is = dot4(w1.z, x1.z, is);
                is = dot4(w1.w, x1.w, is);
                // SEG (AT 6.2): p_k = +0 + (dK Dx) f32(isum); |terms| >= 2^-48 or 0 (fp16 scales), so
                // the plain operations never meet a subnormal; NaN is canonicalized below. The +0 is
                // added once to the tree's result instead: a -0 term changes a node only when every
                // term under it is -0, and then the node is -0 where the rule's is +0
                p[kb] = (h2f_fast(km[kb]) * s_dx[i * NBD + kb]) * (float)is;
            }
#pragma unroll
            for (int w = 16; w > 1; w >>= 1)
#pragma unroll
                for (int k = 0; k < w / 2; ++k) p[k] = p[2 * k] + p[2 * k + 1];
            s = canon(p[0] + 0.0f);
            if (it.general) {
                const float m = a.mask[(size_t)it.t * a.mstride + cell];
                s = fb(m) == kNegInf ? bf(kNegInf) : sadd(s, m);
            }
        }
        if (in) S[(size_t)h * n16 + j] = s;
        const uint32_t mk = wave_max_u(in ? maxt_key_f(s) : maxt_key_f(bf(kMFloor)));
        if (lane == 0) s_red[wave * G + i] = mk;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < G; i += blockDim.x) {
        uint32_t m = s_red[i];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = umax_u(m, s_red[w * G + i]);
        a.Mpart[(size_t)(it.tile0 + tt) * a.n_head + g * G + i] = maxt_unkey(m);
    }
}

// ---------------------------------------------------------------------------------------------
// scores of many rows on the matrix cores: block (256-cell tile, 32 rows, query head), 4 waves of two 32-cell
// subtiles. The rows' runs start at one cell and their items on tile boundaries from there (the host's rule,
// fa_score_tiles), so every row's 256-cell tiles are the same cells; the item of each (tile, row) comes from
// the host's map.
//
// Per 32 rows x 32 cells and 32-value block, as in the prefill MUL_MAT: the integer block sums are one
// v_mfma_i32_32x32x32_i8 (rows: queries, columns: cells) and the products dK Dx one
// v_mfma_f32_32x32x2f32 with a zero second column; the score is the block terms' tree. A lane holds one
// cell of 16 rows, so 32 lanes store 32 consecutive scores of a row. While every scale of the wave is finite
// no score is Inf or NaN: the canonicalization and the NaN rule of the maximum are left to waves that met
// one (sticky). The rows' store offsets are read from LDS where they are needed: with them in registers the
// kernel spilled them too, and a reload waits for the stores in front of it (the memory counter retires in order).
// (D 128, at its 168 registers for three waves a SIMD: three of the 16 maxima pass through scratch once.)
//
// The one-row kernel below reads each K row per query row and spends ~130 VALU operations a score; this one
// ~20.
// ---------------------------------------------------------------------------------------------
typedef float v16f_fa __attribute__((ext_vector_type(16)));
typedef int v16i_fa __attribute__((ext_vector_type(16)));

template <int D>
__global__ __launch_bounds__(256, 3) void k_fa_qk_mm(FaArgs a, uint32_t T) {
    constexpr uint32_t NBD = D / 32u;
    __shared__ uint32_t s_hi[32], s_end[32], s_tile[32];           // of the block's rows: run end, item end, Mpart row
    __shared__ __align__(16) uint32_t s_vo[32];                    // byte offset of the row's score of the tile's first cell
    __shared__ __align__(16) float s_mx[4][64][20];                // each wave's maxima of the lane's 16 rows (padded)
    const uint32_t at = blockIdx.x, t0 = 32u * blockIdx.y, h = blockIdx.z, g = h / a.G;
    const uint32_t lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t c = lane & 31u, hh = lane >> 5;
    const uint32_t cell0 = 16u * (a.u_lo + 16u * at);              // first cell of the tile
    const uint32_t ng = (a.kc.kv_size + 15u) / 16u, E = a.E, nbk = E / 32u;
    // this wave's first K operands and its query operands: they depend on no item
    const uint32_t t = min(t0 + c, T - 1u);
    v4i_fa kr[NBD], xv[NBD];
    uint32_t km[NBD];
    float dx[NBD];
    auto load_k = [&](uint32_t sub) {                              // clamped: loads stay inside the plane
        const uint32_t u0 = min((cell0 + 32u * sub) >> 4, ng - 1u), u = min(u0 + (c >> 4), ng - 1u) - u0;
        const uint8_t * kq = a.kc.base + a.kc.quant_off + ((size_t)u0 * E + (size_t)g * D) * 16u;
        const uint8_t * kmeta = a.kc.base + ((size_t)u0 * nbk + (size_t)g * NBD) * 32u;
        const uint32_t oq = u * 16u * E + hh * 256u + (c & 15u) * 16u, om = (u * nbk * 16u + (c & 15u)) * 2u;
#pragma unroll
        for (uint32_t b = 0; b < NBD; ++b) {
            kr[b] = *(const v4i_fa *)(kq + (oq + 512u * b));
            km[b] = *(const uint16_t *)(kmeta + (om + 32u * b));
        }
    };
#pragma unroll
    for (uint32_t b = 0; b < NBD; ++b) {                           // block b at xq + ((h NBD + b) T + t) 32
        const uint32_t o = (h * NBD + b) * T + t;
        xv[b] = *(const v4i_fa *)(a.xq + (size_t)o * 32u + 16u * hh);
        dx[b] = a.xd[o];
    }
    load_k(2u * wave);
    __builtin_amdgcn_sched_barrier(0);
    // the rows' items (every wave reads them; wave 0 publishes)
    const uint32_t idx = t0 + c < T ? a.tmap[(size_t)at * T + t] : 0xFFFFFFFFu;
    uint32_t end = 0u, hi = 0u;
    if (idx != 0xFFFFFFFFu) {
        const FaItem it = a.items[idx];
        const uint32_t c0 = 16u * it.u0, n16 = 16u * it.n;
        end = c0 + n16;
        hi = a.hi[t];                                              // a run ends inside its last item
        if (threadIdx.x < 32u) {
            s_vo[c] = 4u * (it.s_off * a.n_head + h * n16 + (cell0 - c0));
            s_tile[c] = it.tile0 + (cell0 - c0) / 256u;
        }
    }
    if (threadIdx.x < 32u) {
        s_hi[c] = hi;
        s_end[c] = end;
    }
    uint32_t top = end, all = hi;       // the last item end of the rows; the cells below `all` are visible to every row
#pragma unroll
    for (int sh = 16; sh >= 1; sh >>= 1) {
        top = max(top, (uint32_t)shfl_i((int)top, (int)(lane ^ (uint32_t)sh)));
        all = min(all, (uint32_t)shfl_i((int)all, (int)(lane ^ (uint32_t)sh)));
    }
    top = __builtin_amdgcn_readfirstlane(top);
    all = __builtin_amdgcn_readfirstlane(all);
    if (top <= cell0) return;                                      // no row reaches the tile (block-uniform)
    lds_barrier();

    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(a.S, 0, (int)a.s_bytes, 0x00020000);
    const float ninf = bf(kNegInf);
    bool fin = true;
    float mx[16];
#pragma unroll
    for (uint32_t b = 0; b < NBD; ++b) {
        fin = fin && !__builtin_amdgcn_classf(dx[b], 0x207);
        dx[b] = hh ? 0.0f : dx[b];                                 // the k = 1 column of the scale product
    }
#pragma unroll
    for (uint32_t r = 0; r < 16u; ++r) mx[r] = bf(kMFloor);
    bool slow = __ballot(!fin) != 0ull;
#pragma unroll
    for (uint32_t k2 = 0; k2 < 2u; ++k2) {
        const uint32_t sub = 2u * wave + k2, cs = cell0 + 32u * sub;
        bool kfin = true;
        v16f_fa s[NBD / 2u];                                       // the tree's first level
#pragma unroll
        for (uint32_t b = 0; b < NBD; ++b) {
            v16i_fa is = {};
            is = __builtin_amdgcn_mfma_i32_32x32x32_i8(xv[b], kr[b], is, 0, 0, 0);
            kfin = kfin && (km[b] & 0x7C00u) != 0x7C00u;
            v16f_fa P = {};
            P = __builtin_amdgcn_mfma_f32_32x32x2f32(dx[b], hh ? 0.0f : h2f_fast(km[b]), P, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = P[r] * (float)is[r];
                if (b & 1u) s[b >> 1][r] = s[b >> 1][r] + p;
                else s[b >> 1][r] = p;
            }
            __builtin_amdgcn_sched_barrier(0);                     // one block's products in registers at a time
        }
        slow = slow || __ballot(!kfin) != 0ull;
#pragma unroll
        for (uint32_t w = NBD / 4u; w >= 1u; w >>= 1)
#pragma unroll
            for (uint32_t k = 0; k < w; ++k)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[k][r] = s[2u * k][r] + s[2u * k + 1u][r];
        __builtin_amdgcn_sched_barrier(0);
        if (k2 == 0u) load_k(sub + 1u);                            // ahead of the stores (the counter retires in order)
        __builtin_amdgcn_sched_barrier(0);
        // +0 once (see k_fa_qk); cells outside a row's run are -inf, outside its item not stored
        const uint32_t vc = 128u * sub + 4u * c;
        if (!slow && cs >= a.lo && cs + 32u <= all) {              // wave-uniform: every cell visible to every row
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) {
                const uint4 vo = *(const uint4 *)&s_vo[8u * q + 4u * hh];
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) {
                    const float v = s[0][4u * q + e] + 0.0f;
                    const uint32_t o = e == 0u ? vo.x : (e == 1u ? vo.y : (e == 2u ? vo.z : vo.w));
                    __builtin_amdgcn_raw_buffer_store_b32(fb(v), rs, (int)(o + vc), 0, 0);
                    mx[4u * q + e] = __builtin_fmaxf(mx[4u * q + e], v);
                }
            }
        } else {
#pragma unroll
            for (uint32_t r = 0; r < 16u; ++r) {
                const uint32_t row = 8u * (r >> 2) + 4u * hh + (r & 3u), cell = cs + c;
                const float x = canon(s[0][r] + 0.0f);
                const float v = cell >= a.lo && cell < s_hi[row] ? x : ninf;
                const bool in = cell < s_end[row];
                if (in) __builtin_amdgcn_raw_buffer_store_b32(fb(v), rs, (int)(s_vo[row] + vc), 0, 0);
                const float w = in ? v : bf(kMFloor);
                mx[r] = slow ? maxt(mx[r], w) : __builtin_fmaxf(mx[r], w);
            }
        }
    }
    // the rows' maxima over the tile: value r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q)
        *(float4 *)&s_mx[wave][lane][4u * q] = make_float4(mx[4u * q], mx[4u * q + 1u], mx[4u * q + 2u], mx[4u * q + 3u]);
    lds_barrier();
    {
        const uint32_t row = threadIdx.x >> 3, l8 = threadIdx.x & 7u, r = 4u * (row >> 3) + (row & 3u), half = (row >> 2) & 1u;
        uint32_t k = 0u;
#pragma unroll
        for (uint32_t w = 0; w < 4u; ++w)
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) k = umax_u(k, maxt_key_f(s_mx[w][32u * half + 8u * e + l8][r]));
        k = umax_u(k, (uint32_t)dpp_i<kDppXor1>((int)k));
        k = umax_u(k, (uint32_t)dpp_i<kDppXor2>((int)k));
        k = umax_u(k, (uint32_t)dpp_i<kDppRowHalfMirror>((int)k));
        if (l8 == 0u && s_end[row] > cell0) a.Mpart[(size_t)s_tile[row] * a.n_head + h] = maxt_unkey(k);
    }
}

template <int D, bool INL, int VS>
__global__ __launch_bounds__(64 * kPvWaves) void k_fa_pv(FaArgs a, FaPlan p) {
    extern __shared__ __align__(16) uint8_t lds[];
    using PB = PvBlock<D, VS>;
    constexpr uint32_t DV = PB::DV, BB = PB::BB;
    const uint32_t G = a.G, nh = a.n_head;
    // the launch has one wave per segment of its longest channel (fa_segments), so the segment results need nw slots:
    // the LDS is sized by the launch
    const uint32_t nw = blockDim.x >> 6;
    double * s_td = (double *)lds;                                // EXPK table
    float * s_c = (float *)(lds + 512);                           // [seg][4 heads][DV]
    float * s_l = s_c + nw * 4u * DV;                             // [seg][4 heads]
    uint8_t * s_dg = (uint8_t *)(s_l + nw * 4u);                  // per wave: [BB blocks][4 heads][4 digits][4 groups][16]
    const uint32_t t64v = a.ex.t64[threadIdx.x & 63u];            // first: the table write waits for it only
    const uint32_t item = blockIdx.x >> 2, c = blockIdx.x & 3u, g = blockIdx.y;
    const uint32_t hg = blockIdx.z / VS, vh = blockIdx.z % VS;
    const FaItem it = fa_item<INL>(a, p, item);
    const uint32_t lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t h = g * G + min(4u * hg + (lane >> 4), G - 1u);
    const PB pb(a, it, c, g, hg, vh, a.S + (size_t)it.s_off * nh + (size_t)h * (16u * it.n));
    uint8_t * dg = s_dg + (size_t)wave * (BB * 1024u);
    const uint32_t mkey = maxt_key_f(a.Mpart[(size_t)(it.tile0 + min(lane & 15u, it.ntiles - 1u)) * nh + h]);

    typename PB::Loads L;
    if (wave < pb.nseg) pb.loads(wave, pb.vb0, L, true);
    __builtin_amdgcn_sched_barrier(0);
    if (threadIdx.x < 64u) s_td[threadIdx.x] = (double)t64v * 0x1p-32;
    const ExpkNeg & en = a.en;
    lds_barrier();

    // chunk maximum of head h: MAXOUT of the floor and the tile maxima (row lanes < ntiles read one each)
    float m = maxt_unkey(row16_umax(max(mkey, maxt_key_f(bf(kMFloor)))));
    f64_round_to_zero(m);
    bool common = true;
    // No loop (nseg <= nw): the loads of a second segment kept 24 to 36 more registers alive, 84 .. 100 instead of 60 .. 64,
    // which left five waves a SIMD instead of eight. us, with the loop -> without: 512 rows behind 1536 cells, 32 / 8
    // heads of D 128 177 -> 160; 1994 rows behind 130 882 -> 602; 1870 rows behind 246, 24 / 24 heads of D 64 1694 -> 1081.
    if (wave < pb.nseg) common = pb.segment(wave, L, m, en, s_td, s_c, s_l, dg);
    pb.chains(item, hg, s_c, s_l, __syncthreads_and(common) != 0);
}

// ---------------------------------------------------------------------------------------------
// merge: block (token, KV head g x group of 4 heads, slice sl), lane = (head of the group, value).
// Each lane loads the channel partials, row sums and maxima of up to kMergeItems chunks at once (the
// first round's before the EXPK table is published), then runs CTREE over the 4 channels, the online
// merge in chunk order and finally ANORM (AT 5.6, 5.7). The running maxima of a round are
// wave-uniform, so its 2 kMergeItems merge factors are evaluated by as many lanes at once and read
// back with readlane. A row of one chunk has nothing to merge: its lanes load the four channel
// partials and row sums only and go straight to CTREE and ANORM (the general path's bits for cnt 1).
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kMergeItems = 4;                              // chunks loaded per round
constexpr uint32_t kMergeHeads = 4;                              // heads per block

// VW values a lane. A wave's time is its chain of loads (counts -> items -> maxima), so when there are more waves
// than the chip holds, two values a lane halve the rounds (and the factors formed); with fewer waves one value
// keeps more loads in flight. Rows of two chunks load two, not four. 512 rows x 32 heads x 128 values of two
// chunks (67 MB of partials) 26.8 -> 17.7 us, 300 rows 16.8 -> 11.2.
template <bool INL, int VW>
__global__ __launch_bounds__(256) void k_fa_merge(FaArgs a, FaPlan p) {
    typedef float vw_t __attribute__((ext_vector_type(VW)));
    const uint32_t G = a.G, D = a.D, nh = a.n_head;
    const uint32_t ngrp = (G + kMergeHeads - 1u) / kMergeHeads;
    const uint32_t t = blockIdx.x, g = blockIdx.y / ngrp, h0 = g * G + (blockIdx.y % ngrp) * kMergeHeads;
    const uint32_t hn = min(kMergeHeads, g * G + G - h0), sl = blockIdx.z;
    const uint32_t i = threadIdx.x >> 6, L = threadIdx.x & 63u;
    __shared__ uint32_t s_t64[64];
    const uint32_t t64v = a.ex.t64[L];                            // first: the table write waits for it only
    const uint32_t first = INL ? p.tok_first[t] : a.tok_first[t];
    const uint32_t cnt = INL ? p.tok_count[t] : a.tok_count[t];  // >= 1 (a row without cells has one empty chunk)
    const uint32_t h = h0 + min(i, hn - 1u);                      // waves past the group load, then leave
    const uint32_t v0 = VW * (64u * sl + L);                      // the lane's first value of the head
    float * out = a.out + (size_t)t * a.out_stride + (size_t)h * D + v0;

    if (cnt == 1u) {                                              // one chunk (workgroup-uniform): no merge,
        vw_t op[4];                                               // so no maxima, items or factors to load
        float lp[4];
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) {
            const size_t slot = ((size_t)first * 4u + c) * nh + h;
            op[c] = *(const vw_t *)(a.OP + slot * D + v0);
            lp[c] = a.LP[slot];
        }
        if (i >= hn) return;
        const float rl = srcp(maxt(ctree4_l(lp[0], lp[1], lp[2], lp[3]), bf(kLFloor)));
#pragma unroll
        for (int e = 0; e < VW; ++e) out[e] = smul_n(ctree4_o(op[0][e], op[1][e], op[2][e], op[3][e]), rl);
        return;
    }

    struct Round {
        vw_t op[kMergeItems][4];
        float lp[kMergeItems][4];
        uint32_t key;                                             // MAXT key of one tile maximum
    };
    auto load_round = [&](uint32_t k0, Round & R) {
        const uint32_t kn = min(kMergeItems, cnt - k0);
#pragma unroll
        for (uint32_t k = 0; k < kMergeItems; ++k) {                // every load is issued up front
            if (!INL && k >= kn) break;                           // (inline lists: clamped, the latency counts)
            const size_t kk = first + k0 + min(k, kn - 1u);
#pragma unroll
            for (uint32_t c = 0; c < 4u; ++c) {
                const size_t slot = (kk * 4u + c) * nh + h;
                R.op[k][c] = *(const vw_t *)(a.OP + slot * D + v0);
                R.lp[k][c] = a.LP[slot];
            }
        }
        // lane 8 k + j (k < kMergeItems) reads tile j (clamped) of chunk k: an item has at most 8
        // tiles (NCG <= 128 groups of 16 cells)
        uint32_t tile = 0;
#pragma unroll
        for (uint32_t k = 0; k < kMergeItems; ++k) {                // uniform item reads, per-lane select
            const FaItem itk = fa_item<INL>(a, p, first + k0 + min(k, kn - 1u));
            if ((L >> 3) == k) tile = itk.tile0 + min(L & 7u, itk.ntiles - 1u);
        }
        R.key = maxt_key_f(a.Mpart[(size_t)tile * nh + h]);
    };

    Round R;
    load_round(0u, R);
    __builtin_amdgcn_sched_barrier(0);
    if (threadIdx.x < 64u) s_t64[threadIdx.x] = t64v;
    lds_barrier();
    if (i >= hn) return;                                          // whole waves

    vw_t O = {};
    float l = 0.0f, mr = 0.0f;
    for (uint32_t k0 = 0; k0 < cnt; k0 += kMergeItems) {
        if (k0 != 0u) load_round(k0, R);
        const uint32_t kn = min(kMergeItems, cnt - k0);
        // chunk maxima: MAXOUT of the floor and the chunk's tile maxima over each 8-lane group
        uint32_t key = max(R.key, maxt_key_f(bf(kMFloor)));
        key = umax_u(key, (uint32_t)dpp_i<kDppXor1>((int)key));
        key = umax_u(key, (uint32_t)dpp_i<kDppXor2>((int)key));
        key = umax_u(key, (uint32_t)dpp_i<kDppRowHalfMirror>((int)key));
        float mk[kMergeItems], mrun[kMergeItems];
#pragma unroll
        for (uint32_t k = 0; k < kMergeItems; ++k) {
            mk[k] = maxt_unkey((uint32_t)__builtin_amdgcn_readlane((int)key, 8 * (int)k));
            const float prev = k == 0u ? mr : mrun[k - 1u];
            mrun[k] = k0 + k == 0u ? mk[k] : maxt(prev, mk[k]);
        }
        // lane 2 k + b: factor of chunk k, EXP((prev - mrun_k) scale) for b = 0 (the running sums),
        // EXP((m_k - mrun_k) scale) for b = 1 (the chunk's); the first chunk of a row uses none
        const uint32_t jk = (L >> 1) & (kMergeItems - 1u);
        float from = 0.0f, to = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < kMergeItems; ++k)
            if (jk == k) {
                from = (L & 1u) ? mk[k] : (k == 0u ? mr : mrun[k - 1u]);
                to = mrun[k];
            }
        const float fx = expk_diff(from, to, a.scale, a.ex, s_t64);
#pragma unroll
        for (uint32_t k = 0; k < kMergeItems; ++k) {
            if (k >= kn) break;
            vw_t ok;
#pragma unroll
            for (int e = 0; e < VW; ++e) ok[e] = ctree4_o(R.op[k][0][e], R.op[k][1][e], R.op[k][2][e], R.op[k][3][e]);
            const float lk = ctree4_l(R.lp[k][0], R.lp[k][1], R.lp[k][2], R.lp[k][3]);
            if (k0 + k == 0u) { O = ok; l = lk; }
            else {
                const float fa = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fx), 2 * (int)k));
                const float fbv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fx), 2 * (int)k + 1));
                l = sadd_c(smul_c(l, fa), smul_c(lk, fbv));
#pragma unroll
                for (int e = 0; e < VW; ++e) O[e] = sadd_z(smul_z(O[e], fa), smul_z(ok[e], fbv));
            }
            mr = mrun[k];
        }
    }
    const float rl = srcp(maxt(l, bf(kLFloor)));
#pragma unroll
    for (int e = 0; e < VW; ++e) out[e] = smul_n(O[e], rl);
}

}  // namespace tsr

template <bool INL>
static int launch_fa(const tsr::FaArgs & a, const tsr::FaPlan & p, uint32_t T, uint32_t n_cu, hipStream_t s) {
    const bool rope = a.cell != nullptr;                          // ROPE + SET_ROWS_KV fused (host-checked shape)
    const size_t lds_qk = tsr::fa_qk_lds(a.G, a.D, rope);
    const dim3 gqk(p.n_items * p.maxtiles, a.n_head_kv);
    if (a.tmap != nullptr) {                                      // many rows: scores on the matrix cores (host-checked)
        const dim3 gmm(a.n_map, (T + 31u) / 32u, a.n_head), bmm(256);
        switch (a.D) {
            case 64: hipLaunchKernelGGL(tsr::k_fa_qk_mm<64>, gmm, bmm, 0, s, a, T); break;
            case 128: hipLaunchKernelGGL(tsr::k_fa_qk_mm<128>, gmm, bmm, 0, s, a, T); break;
            default: return -2;
        }
    } else if (rope) {
        switch (a.D) {
            case 64: hipLaunchKernelGGL((tsr::k_fa_qk<64, INL, true>), gqk, dim3(256), lds_qk, s, a, p); break;
            case 128: hipLaunchKernelGGL((tsr::k_fa_qk<128, INL, true>), gqk, dim3(256), lds_qk, s, a, p); break;
            default: return -2;
        }
    } else {
        switch (a.D) {
            case 64: hipLaunchKernelGGL((tsr::k_fa_qk<64, INL, false>), gqk, dim3(256), lds_qk, s, a, p); break;
            case 128: hipLaunchKernelGGL((tsr::k_fa_qk<128, INL, false>), gqk, dim3(256), lds_qk, s, a, p); break;
            case 256: hipLaunchKernelGGL((tsr::k_fa_qk<256, INL, false>), gqk, dim3(256), lds_qk, s, a, p); break;
            case 512: hipLaunchKernelGGL((tsr::k_fa_qk<512, INL, false>), gqk, dim3(256), lds_qk, s, a, p); break;
            default: return -2;
        }
    }
    if (hipGetLastError() != hipSuccess) return -4;
    // P.V: waves = the most segments of any item (<= 8), LDS = table, segment results, digits; the
    // values of a head are split over VS blocks while the grid holds fewer than two blocks per CU
    uint32_t maxn = 0;
    if (INL) {
        for (uint32_t i = 0; i < p.n_items; ++i) maxn = std::max(maxn, p.items[i].n);
    } else {
        maxn = a.max_groups;
    }
    const uint32_t nwv = tsr::fa_segments(maxn);
    if (nwv > tsr::kPvWaves) return -2;
    const uint64_t blocks = 4ull * p.n_items * a.n_head_kv * ((a.G + 3u) / 4u);
    uint32_t vs = 1;
    while (vs < 4u && a.D / (2u * vs) >= 64u && blocks * vs < 2ull * n_cu) vs *= 2u;
    const uint32_t dv = a.D / vs, bb = 2u;                        // PvBlock::BB
    const size_t lds_pv = 512u + 4u * (size_t)nwv * 4u * dv + 4u * nwv * 4u + 1024u * bb * nwv;
    const dim3 gpv(4u * p.n_items, a.n_head_kv, (a.G + 3u) / 4u * vs);
    const dim3 bpv(64u * nwv);
#define TSR_PV(DD, VV) hipLaunchKernelGGL((tsr::k_fa_pv<DD, INL, VV>), gpv, bpv, lds_pv, s, a, p)
    switch (a.D * 8u + vs) {
        case 64 * 8 + 1: TSR_PV(64, 1); break;
        case 128 * 8 + 1: TSR_PV(128, 1); break;
        case 128 * 8 + 2: TSR_PV(128, 2); break;
        case 256 * 8 + 1: TSR_PV(256, 1); break;
        case 256 * 8 + 2: TSR_PV(256, 2); break;
        case 256 * 8 + 4: TSR_PV(256, 4); break;
        case 512 * 8 + 1: TSR_PV(512, 1); break;
        case 512 * 8 + 2: TSR_PV(512, 2); break;
        case 512 * 8 + 4: TSR_PV(512, 4); break;
        default: return -2;
    }
#undef TSR_PV
    if (hipGetLastError() != hipSuccess) return -4;
    const uint32_t ngrp = (a.G + tsr::kMergeHeads - 1u) / tsr::kMergeHeads;
    // two values a lane: more waves than run at once (see the kernel)
    const uint64_t waves = 4ull * T * a.n_head_kv * ngrp * (a.D / 64u);
    bool wide = false;
    if constexpr (!INL) {
        wide = a.D >= 128u && waves > 32ull * n_cu;
        if (wide) hipLaunchKernelGGL((tsr::k_fa_merge<INL, 2>), dim3(T, a.n_head_kv * ngrp, a.D / 128u), dim3(256), 0, s, a, p);
    }
    if (!wide) hipLaunchKernelGGL((tsr::k_fa_merge<INL, 1>), dim3(T, a.n_head_kv * ngrp, a.D / 64u), dim3(256), 0, s, a, p);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int tsr_launch_fa(const tsr::FaArgs & a, const tsr::FaPlan & p, uint32_t T, uint32_t n_cu, hipStream_t s) {
    return a.items ? launch_fa<false>(a, p, T, n_cu, s) : launch_fa<true>(a, p, T, n_cu, s);
}
