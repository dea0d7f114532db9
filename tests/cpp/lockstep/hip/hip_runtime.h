// A CPU stand-in for the HIP runtime, under which a test compiles the operators' .hip sources with the
// host compiler and runs their kernels: one workgroup after another, its lanes as fibers, its waves in
// lockstep at every wave-wide operation.  Between two barriers a wave runs as far as it can before the
// next one starts, in ascending or descending order (lockstep_set): the most uneven progress that the
// barriers allow, so that a missing barrier gives wrong results every time.
//
// A wave-wide operation or barrier that not all of a wave's (a workgroup's) running lanes reach ends the
// program with a message.  lockstep_set can also keep kernels from running and only record the launches.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <ucontext.h>

#include <functional>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ thread_local
#define __align__(n) __attribute__((aligned(n)))

struct dim3 {
    uint32_t x, y, z;
    dim3(uint32_t a = 1, uint32_t b = 1, uint32_t c = 1) : x(a), y(b), z(c) {}
};
struct alignas(8) uint2 {
    uint32_t x, y;
};
struct alignas(16) uint4 {
    uint32_t x, y, z, w;
};

// ---- host side --------------------------------------------------------------------------------------------
typedef void *hipStream_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipDeviceAttributeMultiprocessorCount };
enum { hipFuncAttributeMaxDynamicSharedMemorySize };
hipError_t hipMalloc(void **p, size_t bytes);
hipError_t hipFree(void *p);
hipError_t hipMemset(void *p, int v, size_t bytes);
hipError_t hipDeviceGetAttribute(int *v, int what, int dev);
hipError_t hipGetDevice(int *dev);
hipError_t hipSetDevice(int dev);
hipError_t hipFuncSetAttribute(const void *fn, int what, int value);
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return "lockstep"; }
inline hipError_t hipGetDeviceCount(int *n) {
    *n = 2;
    return hipSuccess;
}
inline hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 2;
    return hipSuccess;
}

namespace lockstep {
enum Op : int { kNone, kBarrier, kBallot, kShfl, kFirst, kRead, kDpp, kSync };
void launch(const char *name, dim3 grid, dim3 block, const std::function<void()> &kernel);
uint32_t thread_id();
void count_cas();
uint32_t block_id();
uint32_t block_size();
uint32_t grid_size();
bool barrier(int line, bool any);                            // true: any lane passed true
const uint64_t *wave_op(Op op, uint64_t v, uint64_t *lanes);  // the wave's 64 values; *lanes: who took part

struct Index {
    uint32_t x;
};
template <class T>
inline uint64_t bits(T v) {
    uint64_t b = 0;
    memcpy(&b, &v, sizeof(T));
    return b;
}
template <class T>
inline T value(uint64_t b) {
    T v;
    memcpy(&v, &b, sizeof(T));
    return v;
}
inline uint32_t lane() { return thread_id() & 63u; }
template <class T>
inline T from_lane(Op op, T v, int64_t src) {  // own value where there is no such lane
    uint64_t on = 0;
    const uint64_t *x = wave_op(op, bits(v), &on);
    return src >= 0 && src < 64 && ((on >> src) & 1u) ? value<T>(x[src]) : v;
}
inline uint64_t ballot(bool p) {
    uint64_t on = 0, b = 0;
    const uint64_t *x = wave_op(kBallot, p ? 1 : 0, &on);
    for (int l = 0; l < 64; ++l) b |= (((on >> l) & 1u) & x[l]) << l;
    return b;
}
inline uint32_t first_lane(uint32_t v) {
    uint64_t on = 0;
    const uint64_t *x = wave_op(kFirst, v, &on);
    return static_cast<uint32_t>(x[__builtin_ctzll(on)]);
}
inline void wave_sync() {
    uint64_t on = 0;
    wave_op(kSync, 0, &on);
}
inline uint32_t mbcnt(uint32_t mask, uint32_t base, uint32_t from) {
    const uint32_t l = lane();
    const uint32_t below = l <= from ? 0u : l - from >= 32u ? ~0u : (1u << (l - from)) - 1u;
    return base + static_cast<uint32_t>(__builtin_popcount(mask & below));
}
}  // namespace lockstep

#define hipLaunchKernelGGL(kern, grid, block, lds, stream, ...) \
    lockstep::launch(#kern, grid, block, [=]() mutable { (kern)(__VA_ARGS__); })

// ---- device side ------------------------------------------------------------------------------------------
#define threadIdx (lockstep::Index{lockstep::thread_id()})
#define blockIdx (lockstep::Index{lockstep::block_id()})
#define blockDim (lockstep::Index{lockstep::block_size()})
#define gridDim (lockstep::Index{lockstep::grid_size()})
#define __syncthreads() lockstep::barrier(__LINE__, false)
#define __syncthreads_or(v) lockstep::barrier(__LINE__, (v) != 0)
#define __ballot(p) lockstep::ballot(p)
#define __lane_id() lockstep::lane()
#define __threadfence() ((void)0)
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) __atomic_load_n(p, order)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)
#define __builtin_amdgcn_readfirstlane(x) lockstep::first_lane(x)
#define __builtin_amdgcn_readlane(x, l) lockstep::from_lane(lockstep::kRead, x, l)
// (the one DPP control in use: the value of the lane below, lane 0 keeps `old`)
#define __builtin_amdgcn_update_dpp(old, x, ctrl, rows, banks, bound) \
    (static_assert_dpp<(ctrl) == 0x138>(), lockstep_dpp(old, x))
#define __builtin_amdgcn_mbcnt_lo(m, b) lockstep::mbcnt(m, b, 0)
#define __builtin_amdgcn_mbcnt_hi(m, b) lockstep::mbcnt(m, b, 32)
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_wave_barrier() lockstep::wave_sync()
#define __builtin_amdgcn_s_sleep(n) ((void)0)
template <bool OK>
inline void static_assert_dpp() {
    static_assert(OK, "DPP control not modelled");
}
inline int lockstep_dpp(int old, int x) {
    const int below = lockstep::from_lane(lockstep::kDpp, x, static_cast<int64_t>(lockstep::lane()) - 1);
    return lockstep::lane() == 0 ? old : below;
}

template <class T>
inline T __shfl(T v, int src, int = 64) { return lockstep::from_lane(lockstep::kShfl, v, src & 63); }
template <class T>
inline T __shfl_xor(T v, int d, int = 64) { return lockstep::from_lane(lockstep::kShfl, v, lockstep::lane() ^ static_cast<unsigned>(d)); }
template <class T>
inline T __shfl_up(T v, unsigned d, int = 64) { return lockstep::from_lane(lockstep::kShfl, v, static_cast<int64_t>(lockstep::lane()) - d); }
template <class T>
inline T __shfl_down(T v, unsigned d, int = 64) { return lockstep::from_lane(lockstep::kShfl, v, static_cast<int64_t>(lockstep::lane()) + d); }

template <class T, class U>
inline T atomicAdd(T *p, U v) { return __atomic_fetch_add(p, static_cast<T>(v), __ATOMIC_RELAXED); }
template <class T, class U>
inline T atomicOr(T *p, U v) { return __atomic_fetch_or(p, static_cast<T>(v), __ATOMIC_RELAXED); }
template <class T, class U>
inline T atomicMin(T *p, U v) {
    const T o = *p;
    if (static_cast<T>(v) < o) *p = static_cast<T>(v);
    return o;
}
template <class T, class U>
inline T atomicMax(T *p, U v) {
    const T o = *p;
    if (static_cast<T>(v) > o) *p = static_cast<T>(v);
    return o;
}
template <class T>
inline T atomicCAS(T *p, T c, T v) {
    lockstep::count_cas();
    const T o = *p;
    if (o == c) *p = v;
    return o;
}
inline int __popc(uint32_t x) { return __builtin_popcount(x); }
inline int __popcll(uint64_t x) { return __builtin_popcountll(x); }
inline int __ffs(uint32_t x) { return __builtin_ffs(static_cast<int>(x)); }
inline int __clz(int x) { return x ? __builtin_clz(static_cast<unsigned>(x)) : 32; }
inline int __clzll(long long x) { return x ? __builtin_clzll(static_cast<unsigned long long>(x)) : 64; }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return static_cast<uint32_t>((static_cast<uint64_t>(a) * b) >> 32); }
inline uint32_t __umul24(uint32_t a, uint32_t b) { return (a & 0xFFFFFFu) * (b & 0xFFFFFFu); }
