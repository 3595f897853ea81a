// Device code shared by the partitioned sweeps (one column: ssgpu_part.hip;
// several columns: ssgpu_part_block.hip).
#pragma once

#include <atomic>

#include "ssgpu_kernels.h"
#include "ssgpu_quot.h"
#include "ssgpu_sweep_dev.h"

namespace ssgpu {

namespace {

constexpr int kAbort = -(1 << 30);   // progress of a part whose workgroup gave up

// keep the compiler from moving LDS accesses across (the hardware keeps their order)
__device__ inline void lds_order() { __asm__ __volatile__("" ::: "memory"); }
// computed here and kept in a register: not sunk to the first use, which is on
// the chain of levels
__device__ inline void settle(unsigned& v) { __asm__ __volatile__("" : "+v"(v)); }
__device__ inline void settle(float& v) { __asm__ __volatile__("" : "+v"(v)); }
__device__ inline void settle(double& v) { __asm__ __volatile__("" : "+v"(v)); }
__device__ inline void settle(zc& v) { __asm__ __volatile__("" : "+v"(v.re), "+v"(v.im)); }
__device__ inline void settle(fc& v) { __asm__ __volatile__("" : "+v"(v.re), "+v"(v.im)); }

__device__ inline double unit(double*) { return 1.0; }
__device__ inline zc unit(zc*) { return zc{1.0, 0.0}; }

// s / d for a divisor known in advance (ssgpu_quot.h); operands outside its
// range take the division itself
struct Recip {
    double d, y;
    bool ok;
    __device__ explicit Recip(double dd) : d(dd), y(1.0 / dd), ok(quot_divisor(dd)) { settle(y); }
    __device__ double quot(double s) const {
        double q = quot_from(s, d, y);
        const bool plain = ok & quot_dividend(s);
        if (__any(!plain)) q = plain ? q : s / d;
        return q;
    }
};
struct RecipC {
    zc d;
    __device__ explicit RecipC(zc dd) : d(dd) {}
    __device__ zc quot(zc s) const { return Num<zc>::div(s, d); }
};
template <typename T> struct RecipOf { using type = Recip; };
template <> struct RecipOf<zc> { using type = RecipC; };

using LdsInt = __attribute__((address_space(3))) int;
using LdsDouble = const __attribute__((address_space(3))) double;
template <typename P> __device__ inline unsigned lds_at(P* p) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) P*)p;
}
__device__ inline void lds_get(unsigned at, double& v) { v = *(LdsDouble*)(uintptr_t)at; }
__device__ inline void lds_get(unsigned at, zc& v) {
    LdsDouble* p = (LdsDouble*)(uintptr_t)at;
    v = zc{p[0], p[1]};
}

// four values of a row
__device__ inline void load4(const double* p, double* v) {
    const double2 a = *reinterpret_cast<const double2*>(p), b = *reinterpret_cast<const double2*>(p + 2);
    v[0] = a.x, v[1] = a.y, v[2] = b.x, v[3] = b.y;
}
__device__ inline void load4(const float* p, float* v) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
}
__device__ inline void load4(const zc* p, zc* v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double2 a = *reinterpret_cast<const double2*>(p + j);
        v[j] = zc{a.x, a.y};
    }
}
__device__ inline void load4(const fc* p, fc* v) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 2);
    v[0] = fc{a.x, a.y}, v[1] = fc{a.z, a.w}, v[2] = fc{b.x, b.y}, v[3] = fc{b.z, b.w};
}

// Whether a sweep of this solve has given up: looked at once in kErrPasses
// polling passes, so that a workgroup that starts after that, or waits, leaves
// soon instead of at its own limit (round after round of the compute units).
// Not with the ticket: there it lengthens the start of every workgroup, 1% of a
// backward sweep at 95^3.
constexpr long kErrPasses = 64;
__device__ inline bool sweep_failed(long spins, const int* err) {
    return spins % kErrPasses == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// what a wave's step holds in registers
template <typename T, typename F, int KMAX> struct PartRow {
    F vals[KMAX];
    unsigned at[KMAX];   // LDS addresses of the inputs
    T r_i, d_i;
};

// Waits until `need` steps of the part are done; false if the workgroup gave
// up, or this wave did (the limit).  The hop from one step to the next is this
// loop's latency: its shortest pass is one LDS read and two branches, the
// bookkeeping done while the read is under way.  Waves whose turn is further
// off sleep between passes and leave the LDS and their SIMD to those before
// them.
__device__ inline bool wait_steps(int need, unsigned done_at, int limit) {
    need = __builtin_amdgcn_readfirstlane(need);
    int tmp, done, off, passes = __builtin_amdgcn_readfirstlane(limit);
    __asm__ __volatile__(
        "1:\n\t"
        "ds_read_b32 %0, %4\n\t"
        "s_sub_i32 %3, %3, 1\n\t"
        "s_cmp_lt_i32 %3, -1\n\t"
        "s_waitcnt lgkmcnt(0)\n\t"
        "s_cbranch_scc1 2f\n\t"
        "v_readfirstlane_b32 %1, %0\n\t"
        "s_sub_i32 %2, %5, %1\n\t"
        "s_cmp_le_i32 %2, 0\n\t"
        "s_cbranch_scc1 2f\n\t"
        "s_cmp_le_i32 %2, 2\n\t"
        "s_cbranch_scc1 1b\n\t"
        "s_cmp_lt_i32 %1, 0\n\t"
        "s_cbranch_scc1 2f\n\t"
        "s_sleep 2\n\t"
        "s_cmp_le_i32 %2, 4\n\t"
        "s_cbranch_scc1 1b\n\t"
        "s_sleep 8\n\t"
        "s_branch 1b\n"
        "2:"
        : "=&v"(tmp), "=&s"(done), "=&s"(off), "+s"(passes)
        : "v"(done_at), "s"(need)
        : "scc", "memory");
    return off <= 0 && passes >= -1;
}

// The rows of one step, the last (forward) or first (backward) LATE entries
// of which wait for the levels just below.
template <typename T, typename F, int MODE, int KMAX, int LATE>
__device__ inline bool part_rows(const PartStep& S, PartRow<T, F, KMAX>& R, const typename RecipOf<T>::type& rc,
                                 unsigned done_at, int limit, T& res) {
    constexpr bool kFwd = MODE == FWD_DIV_LAST;
    constexpr int E0 = kFwd ? 0 : LATE, E1 = kFwd ? KMAX - LATE : KMAX;    // the early entries
    constexpr int L0 = kFwd ? KMAX - LATE : 0, L1 = kFwd ? KMAX : LATE;    // the late ones
    T acc = (MODE == BWD_IC) ? Num<T>::zero() : R.r_i;
    T prod[KMAX];
    bool ok = true;
    if (LATE < KMAX) {
        ok = wait_steps(S.need0, done_at, limit);
        lds_order();
#pragma unroll
        for (int k = E0; k < E1; ++k) lds_get(R.at[k], prod[k]);
#pragma unroll
        for (int k = E0; k < E1; ++k) {
            prod[k] = Num<T>::mul(wid<T, F>(R.vals[k]), prod[k]);
            if (kFwd) acc = Num<T>::sub(acc, prod[k]);
            else settle(prod[k]);
        }
        if (kFwd) settle(acc);
    }
    ok &= wait_steps(S.need, done_at, limit);
    lds_order();
    __builtin_amdgcn_s_setprio(3);
#pragma unroll
    for (int k = L0; k < L1; ++k) lds_get(R.at[k], prod[k]);
#pragma unroll
    for (int k = L0; k < L1; ++k) {
        prod[k] = Num<T>::mul(wid<T, F>(R.vals[k]), prod[k]);
        if (kFwd) acc = Num<T>::sub(acc, prod[k]);
    }
    if (!kFwd) {
#pragma unroll
        for (int k = 0; k < KMAX; ++k) acc = Num<T>::sub(acc, prod[k]);
    }
    res = (MODE == BWD_IC) ? Num<T>::add(Num<T>::mul(acc, R.d_i), R.r_i) : rc.quot(acc);
    return ok;
}


// More shared memory than a launch may take by default: allowed once per
// kernel and device.
constexpr size_t kPartLdsMax = (160 << 10) - 256;
void allow_lds(const void* fn, std::atomic<uint64_t>& allowed) {
    int dev = 0;
    SSGPU_HIP(hipGetDevice(&dev));
    const uint64_t bit = dev < 64 ? uint64_t(1) << dev : 0;
    if (bit != 0 && (allowed.load(std::memory_order_relaxed) & bit)) return;
    SSGPU_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPartLdsMax));
    allowed.fetch_or(bit);
}

}  // namespace

}  // namespace ssgpu
