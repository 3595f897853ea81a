// Device helpers shared by the sync-free sweeps: the "not there yet" sentinel
// of polled vectors, agent-scope loads and stores, and widening of factor
// values.
#pragma once

#include "ssgpu_common.h"
#include "ssgpu_kernels.h"

namespace ssgpu {

constexpr unsigned long long kSentinel = kSweepSentinel;

__device__ inline bool sent(double v) { return (unsigned long long)__double_as_longlong(v) == kSentinel; }
__device__ inline bool sent(zc v) { return sent(v.re) || sent(v.im); }
__device__ inline double sent_val(double*) { return __longlong_as_double((long long)kSentinel); }
__device__ inline zc sent_val(zc*) {
    const double s = __longlong_as_double((long long)kSentinel);
    return zc{s, s};
}

__device__ inline double gload(const double* p) {
    return __longlong_as_double((long long)__hip_atomic_load((unsigned long long*)p, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline zc gload(const zc* p) {
    const double* d = reinterpret_cast<const double*>(p);
    return zc{gload(d), gload(d + 1)};
}
__device__ inline void gstore(double* p, double v) {
    __hip_atomic_store((unsigned long long*)p, (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void gstore(zc* p, zc v) {
    double* d = reinterpret_cast<double*>(p);
    gstore(d, v.re);
    gstore(d + 1, v.im);
}
template <typename T, typename F> __device__ inline T wid(F a);
template <> __device__ inline double wid<double, double>(double a) { return a; }
template <> __device__ inline double wid<double, float>(float a) { return (double)a; }
template <> __device__ inline zc wid<zc, zc>(zc a) { return a; }
template <> __device__ inline zc wid<zc, fc>(fc a) { return zc{(double)a.re, (double)a.im}; }

}  // namespace ssgpu
