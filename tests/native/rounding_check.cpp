// The device's forms of three rounding rules against the rules themselves, on the CPU: EXPK of arguments <= 0 in
// truncating f64 (expk.hpp: expk_neg_diff) and the A32 quantizer's rounding (tsr_dev.hpp: round_away, round_away8)
// against the oracle's, the digit sums' rounding (fa_common.hpp: digits_rne24) against an exact integer's. Arguments:
// the step between the tried f32 bit patterns (1: all of them, some minutes) and the number of threads. Exit status 1
// and the first value that differs.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

typedef double f64;
#define double Rz
#define __builtin_fma rz_fma
#include "expk.hpp"
#undef __builtin_fma
#include "fa_common.hpp"
#undef double

extern "C" float oc_expk(float);
extern "C" int32_t oc_round_away8(float);

using tsr::bf;
using tsr::fb;

static tsr::ExpkNeg en;                                           // as the host sets it up (runtime.hpp, tsr_attn.hip)
static Rz td[64];
static void constants() {
    const long double ln2 = M_LN2l;
    const f64 lk = (f64)llroundl(ldexpl(M_LOG2El, 38)), c1 = (f64)llroundl(ldexpl(ln2, 32)),
              c2 = (f64)llroundl(ldexpl(ln2 * ln2 / 2.0L, 32)), c3 = (f64)llroundl(ldexpl(ln2 * ln2 * ln2 / 6.0L, 32));
    en = { lk * 0x1p-6, c3, c2 - 0x1p52, c1 - 0x1p52 };
    for (int j = 0; j < 64; ++j) td[j] = (f64)llroundl(ldexpl(exp2l((long double)j / 64.0L), 30)) * 0x1p-32;
}

static bool one(uint32_t u) {
    const float x = bf(u);
    if ((u >> 31) != 0u || x != x || x == 0.0f) {                 // EXPK of a difference <= 0 or NaN
        const float got = tsr::expk_neg_diff(x, 0.0f, 1.0f, en, td), want = oc_expk(x);
        if (fb(got) != fb(want)) return printf("EXPK of %08x: %08x, not %08x\n", u, fb(got), fb(want)), false;
    }
    const int32_t want = oc_round_away8(x);
    if (tsr::round_away8(x) != want) return printf("round_away8 of %08x: %d, not %d\n", u, tsr::round_away8(x), want), false;
    if (std::fabs(x) < 127.5f && tsr::round_away(x) != want)      // a32_pack: |x id| <= 127 (1 + 2^-22)
        return printf("round_away of %08x: %d, not %d\n", u, tsr::round_away(x), want), false;
    return true;
}

static bool digits(int32_t d0, int32_t d1, int32_t d2, int32_t d3) {
    const tsr::v4i_fa d = { d0, d1, d2, d3 };
    const float got = tsr::digits_rne24(d), want = (float)(d0 + 256ll * d1 + 65536ll * d2 + (1ll << 24) * d3);
    if (fb(got) == fb(want)) return true;
    printf("digits %d %d %d %d: %08x, not %08x\n", d0, d1, d2, d3, fb(got), fb(want));
    return false;
}

int main(int argc, char ** argv) {
    const uint64_t step = argc > 1 ? strtoull(argv[1], nullptr, 0) : 4099u;
    const uint32_t nt = argc > 2 ? (uint32_t)atoi(argv[2]) : 1u;
    constants();
    for (uint32_t u = 0; u < 0x10000u; ++u)                       // every exponent with its first and last significands
        if (!one(u << 16) || !one((u << 16) | 0xFFFFu) || !one((u << 16) | 1u)) return 1;
    for (int n = 0; n <= 1300; ++n)                               // around the quantizer's half steps
        for (int k = -3; k <= 3; ++k)
            for (uint32_t s : { 0u, 0x80000000u })
                if (!one((fb((float)n * 0.5f) + (uint32_t)k) ^ s)) return 1;
    std::vector<char> ok(nt, 1);
    std::vector<std::thread> th;
    for (uint32_t i = 0; i < nt; ++i)
        th.emplace_back([&, i] {
            for (uint64_t u = i * step; u < (1ull << 32) && ok[i]; u += nt * step) ok[i] = one((uint32_t)u);
        });
    for (auto & t : th) t.join();
    for (char o : ok)
        if (!o) return 1;
    std::mt19937_64 rng(1);
    const int32_t top = 1 << 20;
    for (int32_t a : { -top, -1, 0, 1, top })                     // the ends of the digit sums, then any
        for (int32_t b : { -top, -1, 0, 1, top })
            for (int32_t c : { -top, -1, 0, 1, top })
                for (int32_t d : { -top, -1, 0, 1, top })
                    if (!digits(a, b, c, d)) return 1;
    for (int i = 0; i < 4000000; ++i) {
        int32_t d[4];
        for (int32_t & v : d) v = (int32_t)(rng() % (2u * top + 1u)) - top;
        if (i & 1) d[3] = (int32_t)(rng() % 64u) - 32;            // small ones: ties of the 24 bits
        if ((i & 3) == 3) d[3] = 0, d[2] = (int32_t)(rng() % 1024u) - 512;
        if (!digits(d[0], d[1], d[2], d[3])) return 1;
    }
    printf("every value rounds by its rule\n");
    return 0;
}
