// What the headers of csrc/ need to compile for the host. The arithmetic of the device headers runs on the CPU
// (the wave exchanges are declared only); a test that defines `double` as Rz computes f64 rounded toward zero,
// as the wave does behind f64_round_to_zero, while float rounds to nearest even. The runtime's calls are
// declared; a test that needs them defines them.
#pragma once

#include <immintrin.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1 };
typedef struct ihipStream_t * hipStream_t;
typedef struct ihipEvent_t * hipEvent_t;
constexpr unsigned hipEventDisableTiming = 2u, hipHostMallocDefault = 0u, hipHostMallocCoherent = 0x40000000u;
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *);
hipError_t hipStreamSynchronize(hipStream_t);
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned);
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned);
hipError_t hipEventRecord(hipEvent_t, hipStream_t);
hipError_t hipEventSynchronize(hipEvent_t);
hipError_t hipEventDestroy(hipEvent_t);
hipError_t hipDeviceSynchronize();
hipError_t hipMalloc(void **, size_t);
hipError_t hipFree(void *);
hipError_t hipHostMalloc(void **, size_t, unsigned);
hipError_t hipHostFree(void *);
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t);
hipError_t hipGetLastError();

struct float2 { float x, y; };
struct float4 { float x, y, z, w; };
struct int4 { int x, y, z, w; };
struct uint2 { uint32_t x, y; };
struct uint4 { uint32_t x, y, z, w; };
inline float2 make_float2(float x, float y) { return { x, y }; }
inline float4 make_float4(float x, float y, float z, float w) { return { x, y, z, w }; }
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return { x, y, z, w }; }
using std::max;
using std::min;

inline float __uint_as_float(uint32_t u) { return __builtin_bit_cast(float, u); }
inline uint32_t __float_as_uint(float f) { return __builtin_bit_cast(uint32_t, f); }
inline float __int_as_float(int u) { return __builtin_bit_cast(float, u); }
inline int __float_as_int(float f) { return __builtin_bit_cast(int, f); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
uint32_t __lane_id();
#define __HIP_MEMORY_SCOPE_AGENT 4
#define __hip_atomic_load(p, ...) (*(p))
#define __hip_atomic_store(p, v, ...) (void)(*(p) = (v))
#define __hip_atomic_fetch_add(p, v, ...) (*(p) += (v))

extern "C" {
int __builtin_amdgcn_update_dpp(int, int, int, int, int, bool);
int __builtin_amdgcn_ds_swizzle(int, int);
int __builtin_amdgcn_ds_bpermute(int, int);
int __builtin_amdgcn_readlane(int, int);
int __builtin_amdgcn_sdot4(int, int, int, bool);
uint32_t __builtin_amdgcn_perm(uint32_t, uint32_t, uint32_t);
uint32_t __builtin_amdgcn_ubfe(uint32_t, uint32_t, uint32_t);
void __builtin_amdgcn_s_waitcnt(int);
void __builtin_amdgcn_s_barrier();
void __builtin_amdgcn_sched_barrier(int);
uint64_t __ballot(bool);
}
inline bool __builtin_amdgcn_classf(float f, int mask) {          // v_cmp_class_f32
    const uint32_t u = __float_as_uint(f), a = u & 0x7FFFFFFFu, s = u >> 31;
    int c;
    if (a > 0x7F800000u) c = (a & 0x00400000u) ? 1 : 0;
    else if (a == 0x7F800000u) c = s ? 2 : 9;
    else if (a >= 0x00800000u) c = s ? 3 : 8;
    else if (a != 0u) c = s ? 4 : 7;
    else c = s ? 5 : 6;
    return ((mask >> c) & 1) != 0;
}

// v_cvt_i32_f32: toward zero, NaN to 0, saturating (the only asm statement of the headers with that form)
inline int32_t host_cvt_i32(float x) {
    if (x != x) return 0;
    if (x >= 2147483648.0f) return INT32_MAX;
    if (x < -2147483648.0f) return INT32_MIN;
    return (int32_t)x;
}
#define asm(...) r = host_cvt_i32(x)

struct Rz {
    double v;
    Rz() = default;
    template <class T> constexpr Rz(T x) : v(x) {}
    explicit operator float() const { return (float)v; }
    constexpr Rz operator-() const { return Rz(-v); }
};
namespace rz {
// one f64 operation toward zero: MXCSR.RC (bits 14:13) around it, nothing moved across
inline double op(double a, double b, double c, int kind) {
    volatile double x = a, y = b, z = c, r;
    const uint32_t csr = _mm_getcsr();
    _mm_setcsr(csr | 0x6000u);
    switch (kind) {
        case 0: r = x + y; break;
        case 1: r = x - y; break;
        case 2: r = x * y; break;
        default: r = __builtin_fma(x, y, z); break;
    }
    _mm_setcsr(csr & ~0x6000u);
    return r;
}
}
inline Rz operator+(Rz a, Rz b) { return rz::op(a.v, b.v, 0, 0); }
inline Rz operator-(Rz a, Rz b) { return rz::op(a.v, b.v, 0, 1); }
inline Rz operator*(Rz a, Rz b) { return rz::op(a.v, b.v, 0, 2); }
inline Rz rz_fma(Rz a, Rz b, Rz c) { return rz::op(a.v, b.v, c.v, 3); }
