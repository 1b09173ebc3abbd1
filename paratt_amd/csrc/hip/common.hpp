// common.hpp -- shared helpers for the gfx950 kernels of the TT library.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "ptt_hip.h"

namespace ptt {

extern hipStream_t g_stream;
extern hipStream_t g_launch;  // g_stream, or the side stream between side_begin / side_end
[[noreturn]] void fatal_hip(hipError_t e, const char *what, const char *file,
                            int line);

#define HIPCHECK(x)                                              \
    do {                                                         \
        hipError_t e_ = (x);                                     \
        if (e_ != hipSuccess) ptt::fatal_hip(e_, #x, __FILE__, __LINE__); \
    } while (0)

// Records HIP events around the launches issued in its lifetime when
// profiling is on; the elapsed time is attributed to `name`.
struct ProfScope {
    bool active;
    const char *nm;
    double flops, bytes;
    hipEvent_t a;
    explicit ProfScope(const char *name, double flops = 0.0, double bytes = 0.0);
    ~ProfScope();
};

// Launch on the current library stream; with profiling on, HIP events
// bracket the launch and its algorithmic flops / bytes are credited to `name`.
#define PTT_LAUNCH_FB(name, flops, bytes, kern, grid, block, shmem, ...) \
    do {                                                                \
        ptt::ProfScope ps_(name, flops, bytes);                         \
        hipLaunchKernelGGL(kern, grid, block, shmem, ptt::g_launch,     \
                           __VA_ARGS__);                                \
        HIPCHECK(hipGetLastError());                                    \
    } while (0)
#define PTT_LAUNCH(name, kern, grid, block, shmem, ...) \
    PTT_LAUNCH_FB(name, 0.0, 0.0, kern, grid, block, shmem, __VA_ARGS__)

inline unsigned cdiv(long a, long b) { return (unsigned)((a + b - 1) / b); }

// Grid-stride cap for streaming kernels: enough waves to fill 256 CUs.
inline unsigned stream_blocks(long n, int threads) {
    long b = (n + threads - 1) / threads;
    long cap = 256L * 16;
    return (unsigned)(b < 1 ? 1 : (b > cap ? cap : b));
}

// 1/x (x normal) and sqrt(x) (x > 0, normal) from the hardware approximations
// and Newton steps: to about an ulp, in a third of the library calls' latency.
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}
__device__ __forceinline__ double sqrt_nr(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    e = fma(-g, g, x);
    g = fma(e, h, g);
    e = fma(-g, g, x);
    return fma(e, h, g);
}

// ---- sums across the lanes of a wave
// DPP move of a double inside a quad / row (dpp_ctrl CTRL); every source lane
// used below is a valid lane of the same row.
template <int CTRL>
__device__ __forceinline__ double dppd(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, false);
    hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// Sum over each aligned quad of lanes (xor 1, xor 2 quad permutations).
__device__ __forceinline__ double quad_sum(double x) {
    x += dppd<0xB1>(x);
    x += dppd<0x4E>(x);
    return x;
}
// x + (x of lane ^ 16) and x + (x of lane ^ 32): the gfx950 lane-swap
// instructions exchange the 16-lane rows of each half / the two halves.
__device__ __forceinline__ double xor16_sum(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
// x of lane ^ 16
__device__ __forceinline__ double xor16_other(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    // one of the pair is x itself
    const bool odd = (threadIdx.x & 16) != 0;
    return __hiloint2double(odd ? h[0] : h[1], odd ? l[0] : l[1]);
}
__device__ __forceinline__ double xor32_sum(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
// Sum over the 64 lanes of a wave (every lane receives it): quad
// permutations, half-row and row mirrors inside each 16-lane row, then the
// two cross-row swaps.
__device__ __forceinline__ double wave_sum(double x) {
    x = quad_sum(x);
    x += dppd<0x141>(x);
    x += dppd<0x140>(x);
    x = xor16_sum(x);
    return xor32_sum(x);
}
// Value of lane N of each row of 16 lanes, on all of them.
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp(0LL, __double_as_longlong(v), 0x150 + N, 0xF, 0xF, true));
}
__device__ __forceinline__ double row16_sum(double x) {
    x = quad_sum(x);
    x += dppd<0x141>(x);
    return x + dppd<0x140>(x);
}
// Largest over the 64 lanes of a wave, the way of wave_sum.
__device__ __forceinline__ double wave_max(double x) {
    x = fmax(x, dppd<0xB1>(x));
    x = fmax(x, dppd<0x4E>(x));
    x = fmax(x, dppd<0x141>(x));
    x = fmax(x, dppd<0x140>(x));
    {
        const int lo = __double2loint(x), hi = __double2hiint(x);
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        x = fmax(__hiloint2double(h[0], l[0]), __hiloint2double(h[1], l[1]));
    }
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return fmax(__hiloint2double(h[0], l[0]), __hiloint2double(h[1], l[1]));
}

// Workgroup barrier that orders LDS traffic only: outstanding global stores
// do not hold the barrier.
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace ptt
