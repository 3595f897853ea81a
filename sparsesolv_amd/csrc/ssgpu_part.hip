// Partitioned triangular sweeps for gfx950 (layout: ssgpu_parts.h).
//
// A sweep is a chain of dependent levels, and what a level costs is how long
// one result takes to reach the row that waits for it.  Through device memory
// that is about 1.5 us (store, coherence, poll); through LDS it is a few
// hundred clocks.  So each workgroup owns an interval of rows and keeps their
// results in LDS: only the inputs that cross an interval go through device
// memory, and they are polled ahead of the level that needs them.
//
// One workgroup per part, taken by ticket, lowest part first: a part reads
// only parts with smaller numbers, whose workgroups are running or done, so
// the sweep cannot deadlock however workgroups are dispatched and whatever
// else runs on the GPU.  Wave w takes the part's steps w, w + W, ...; it
//   1. loads the step's entries, right-hand side and diagonal into registers,
//   2. polls the step's externals (agent-scope loads, a signalling-NaN
//      sentinel for "not there yet") and stages them in its LDS area,
//   3. waits until the part's steps at lower levels are done (one LDS counter),
//   4. gathers every input from LDS, forms the rows in the reference's
//      sequential order, and publishes: to LDS for its own part, at the level
//      position in device memory for later parts, and by row for the caller.
// 1 and 2 of the next steps run on the other waves while one is in 4, so a
// level costs 3 and 4 alone.
//
// LDS operations of one wave are performed in the order they are issued, so
// the counter's increment after the results needs no wait in between.
//
// Measured (forward / backward sweep, ms; before: one 64-row chunk of the
// level order per wave, all inputs through device memory): 95^3 (N 2,518,260,
// 1588 levels) 0.72 / 0.71, before 2.43 / 2.78; 40^3 0.25 / 0.25, before 0.91
// / 1.08; 10^3 0.047 / 0.046, before 0.185 / 0.190; 64^3 complex 0.73 / 0.79,
// before 2.56 / 2.76.  A level costs about 700 clocks in a part (an LDS hop
// and poll 250, the late inputs' gather and the row's serial sum 250,
// publishing 100), and a step's loads, polls and early sums are hidden as long
// as the W waves together keep ahead of that pace; at 95^3 they are not quite
// (0.45 us a level against 0.30 alone), since polls of device memory take 1.5
// us there.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "ssgpu_kernels.h"
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

// s / d for a divisor known in advance, y = 1 / d rounded to nearest: two
// Newton corrections of s * y, the second of which rounds correctly
// (P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990, theorem 8.3) as long as no intermediate
// leaves the normal range; other operands take the division itself.
struct Recip {
    double d, y;
    bool ok;
    __device__ explicit Recip(double dd) : d(dd), y(1.0 / dd) {
        const double a = __builtin_fabs(dd);
        ok = a >= 0x1p-400 && a <= 0x1p400;
        settle(y);
    }
    __device__ double quot(double s) const {
        const double q0 = s * y;
        const double q1 = __builtin_fma(__builtin_fma(-q0, d, s), y, q0);
        // the corrections of a zero keep its value but not its sign
        double q = __builtin_copysign(__builtin_fma(__builtin_fma(-q1, d, s), y, q1), q0);
        const double a = __builtin_fabs(s);
        const bool plain = ok & ((s == 0.0) | ((a >= 0x1p-400) & (a <= 0x1p400)));
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

// One part, by the whole workgroup; lx: its LDS slots, s_done: its step counter
// (zeroed, with slot 0, before the workgroup's barrier).  ROWS: results are
// polled by row in xo (sentinel-filled) and xp is not used.
template <typename T, typename F, int MODE, int KMAX, int W, bool ROWS>
__device__ inline void part_sweep(const PartArgs& pa, int part, T* lx, int& s_done, int* __restrict__ err,
                                  long spin_limit, const F* __restrict__ eval, const F* __restrict__ dval,
                                  const T* __restrict__ rhs, const T* __restrict__ dd, T* __restrict__ xp,
                                  T* __restrict__ xo) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const T* const polled = ROWS ? xo : xp;
    // a wave that waited past the limit sets the error flag and stops its part
    auto give_up = [&](int* done_p) {
        if ((threadIdx.x & 63) == 0) {
            atomicOr(err, 1);
            __hip_atomic_store(done_p, kAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    const int s0 = pa.part_step[part], s1 = pa.part_step[part + 1];
    T* const stage = lx + 1 + wave * kPartExt;
    T* const mine = lx + 1 + W * kPartExt;
    constexpr int NB = kPartExt / 64;
    constexpr bool kFwd = MODE == FWD_DIV_LAST;
    const unsigned base = lds_at(lx);
    // passes over the LDS counter, far shorter than polling passes of device
    // memory: 64 count as one
    const int wait_limit = (int)(spin_limit < (1L << 24) ? spin_limit * 64 : 1L << 30);
    int st = s0 + wave;
    if (st >= s1) return;
    // a step's header, externals' positions and rows are loaded one step ahead
    PartStep S = pa.steps[st];
    int ep[NB], row;
    auto fetch = [&](const PartStep& Q, int (&e)[NB], int& r) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int j = lane + 64 * b;
            e[b] = j < Q.next ? pa.ext[Q.ext0 + j] : -1;
            if (ROWS && e[b] >= 0) e[b] = pa.srow[e[b]];
        }
        r = lane < Q.cnt ? pa.srow[Q.pos0 + lane] : 0;
    };
    fetch(S, ep, row);
    while (true) {
        const bool active = lane < S.cnt;
        // --- 1: the step's rows and entries ----------------------------------------------
        PartRow<T, F, KMAX> R;
        // Quads the step does not have are read from the padding quads (value
        // 0, LDS slot 0), and idle lanes take the last row's: no condition in
        // the row's sum, one uniform base and one lane offset for every load.
        const int qn = (int)S.quads, qskip = kFwd ? KMAX / 4 - qn : 0;
        const int l4 = 4 * min(lane, (int)S.cnt - 1);
        ushort4 sl[KMAX / 4];
#pragma unroll
        for (int q = 0; q < KMAX / 4; ++q) {
            const int j = q - qskip;
            const int at = j >= 0 && j < qn ? S.ent + 4 * j * (int)S.cnt : 0;
            load4(eval + at + l4, R.vals + 4 * q);
            sl[q] = *reinterpret_cast<const ushort4*>(pa.slot + at + l4);
        }
        R.r_i = Num<T>::zero();
        R.d_i = unit((T*)nullptr);
        if (active) {
            R.r_i = rhs[row];
            if (MODE == BWD_IC) R.d_i = dd[row];
            else R.d_i = wid<T, F>(dval[S.pos0 + lane]);
        }
        const bool more = st + W < s1;
        const PartStep N = pa.steps[more ? st + W : st];
        // --- 2: externals into LDS ------------------------------------------------------
        // Polled once the part is within kPartNear steps of this one: polling
        // earlier only adds traffic, which is what lengthens a poll.
        if (S.next > 0) {
            if (!wait_steps(S.need - (int)S.near, lds_at(&s_done), wait_limit)) {
                give_up(&s_done);
                return;
            }
            long spins = 0;
            unsigned miss = 0;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (ep[b] >= 0) miss |= 1u << b;
            while (true) {
                lds_order();
                const unsigned want = miss;
                T v[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    if ((want >> b) & 1u) v[b] = gload(polled + ep[b]);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    if (((want >> b) & 1u) && !sent(v[b])) {
                        stage[lane + 64 * b] = v[b];
                        miss &= ~(1u << b);
                    }
                if (!__any(miss != 0u)) break;
                if (__any(miss != want) && spin_limit > 0) spins = 0;
                const int done = __builtin_amdgcn_readfirstlane(
                    __hip_atomic_load(&s_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                if (done < 0) return;
                if (++spins > spin_limit) {
                    give_up(&s_done);
                    return;
                }
                if (S.need > done) __builtin_amdgcn_s_sleep(4);
                else __builtin_amdgcn_s_sleep(1);
            }
        }
        const typename RecipOf<T>::type rc(R.d_i);
#pragma unroll
        for (int k = 0; k < KMAX; ++k) {
            const ushort4 v = sl[k / 4];
            const unsigned slot = k % 4 == 0 ? v.x : k % 4 == 1 ? v.y : k % 4 == 2 ? v.z : v.w;
            R.at[k] = slot * (unsigned)sizeof(T) + base;
            settle(R.at[k]);
            settle(R.vals[k]);
        }
        settle(R.r_i);
        settle(R.d_i);
        int epn[NB], rown;
        fetch(N, epn, rown);
        // --- 3, 4: the rows ---------------------------------------------------------------
        T res;
        bool fine;
#define SSGPU_ROWS(K) part_rows<T, F, MODE, KMAX, (K)>(S, R, rc, lds_at(&s_done), wait_limit, res)
        if (S.late <= 3) fine = SSGPU_ROWS(3);
        else if (S.late <= 4) fine = SSGPU_ROWS(4);
        else if (S.late <= 6) fine = SSGPU_ROWS(6);
        else fine = SSGPU_ROWS(KMAX);
#undef SSGPU_ROWS
        if (!fine) {   // nothing is published
            give_up(&s_done);
            return;
        }
        if (active) mine[S.lpos + lane] = res;
        lds_order();
        if (lane == 0)   // no wait on the results before it: a wave's LDS operations are performed in order
            __asm__ __volatile__("ds_add_u32 %0, %1" ::"v"(lds_at(&s_done)), "v"(1) : "memory");
        __builtin_amdgcn_s_setprio(0);
        if (active) {
            if (ROWS) {
                gstore(xo + row, res);
            } else {
                gstore(xp + S.pos0 + lane, res);
                xo[row] = res;
            }
        }
        if (!more) return;
        st += W;
        S = N;
        row = rown;
#pragma unroll
        for (int b = 0; b < NB; ++b) ep[b] = epn[b];
    }
}

template <typename T, typename F, int MODE, int KMAX, int W>
__global__ __launch_bounds__(64 * W) void k_sweep_part(PartArgs pa, int* __restrict__ ticket, int* __restrict__ err,
                                                       long spin_limit, const F* __restrict__ eval,
                                                       const F* __restrict__ dval, const T* __restrict__ rhs,
                                                       const T* __restrict__ dd, T* __restrict__ xp,
                                                       T* __restrict__ xo) {
    extern __shared__ __align__(16) unsigned char part_lds[];
    __shared__ int s_part, s_done;
    T* lx = reinterpret_cast<T*>(part_lds);
    if (threadIdx.x == 0) {
        s_part = atomicAdd(ticket, 1);
        s_done = 0;
        lx[0] = Num<T>::zero();
    }
    __syncthreads();
    const int part = __builtin_amdgcn_readfirstlane(s_part);
    if (part >= pa.nparts) return;
    part_sweep<T, F, MODE, KMAX, W, false>(pa, part, lx, s_done, err, spin_limit, eval, dval, rhs, dd, xp, xo);
}

// The parts of many systems in one launch (batched solves).  order[t] =
// (system, part) in ticket order: a system's parts in their own order, systems
// interleaved by the level a part starts at, so that the workgroups running
// sit at the level fronts of all systems at once; a part's inputs lie at
// smaller tickets.  Parts of systems whose status is not `want` are skipped.
// Bound by the longest system's chain of levels, and by the compute units when
// the parts of all systems are more than they hold.  Outputs are polled by row
// (the update kernels reset them to the sentinel; no second array per system).
// Whole iterations, chunked against in parts: 16 systems of n=8..24 1.13 ->
// 0.43 ms (a sweep 0.22), 64 of n=8..40 3.60 -> 1.88, one of n=60 3.44 -> 1.55,
// 32 of n=60 11.6 -> 7.2, two of n=95 6.87 -> 3.02 ms.
template <typename T, typename F, int MODE, int KMAX, int W>
__global__ __launch_bounds__(64 * W) void k_batch_part(const int2* __restrict__ order, int* __restrict__ ticket,
                                                       int* __restrict__ err, long spin_limit,
                                                       const BatchSys* __restrict__ sys,
                                                       const BatchState* __restrict__ st, int want, int in, int out) {
    extern __shared__ __align__(16) unsigned char part_lds[];
    __shared__ int s_item, s_done;
    T* lx = reinterpret_cast<T*>(part_lds);
    if (threadIdx.x == 0) {
        s_item = atomicAdd(ticket, 1);
        s_done = 0;
        lx[0] = Num<T>::zero();
    }
    __syncthreads();
    const int2 it = order[__builtin_amdgcn_readfirstlane(s_item)];
    const int sy = __builtin_amdgcn_readfirstlane(it.x), part = __builtin_amdgcn_readfirstlane(it.y);
    if (st[sy].status != want) return;
    const BatchSys& S = sys[sy];
    const BatchPart& P = MODE == FWD_DIV_LAST ? S.f_part : S.b_part;
    part_sweep<T, F, MODE, KMAX, W, true>(P.args, part, lx, s_done, err, spin_limit, static_cast<const F*>(P.eval),
                                          static_cast<const F*>(P.dval), static_cast<const T*>(S.vec[in]),
                                          static_cast<const T*>(S.diagD), nullptr, static_cast<T*>(S.vec[out]));
}

// More shared memory than a launch may take by default: allowed once per
// kernel and device.
void allow_lds(const void* fn, std::atomic<uint64_t>& allowed) {
    int dev = 0;
    SSGPU_HIP(hipGetDevice(&dev));
    const uint64_t bit = dev < 64 ? uint64_t(1) << dev : 0;
    if (bit != 0 && (allowed.load(std::memory_order_relaxed) & bit)) return;
    SSGPU_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (160 << 10) - 256));
    allowed.fetch_or(bit);
}

template <typename T, typename F, int MODE, int KMAX, int W>
void launch_one(hipStream_t s, size_t lds, const PartArgs& pa, int* ticket, int* err, long spin_limit, const F* eval,
                const F* dval, const T* rhs, const T* dd, T* xp, T* xo) {
    auto fn = k_sweep_part<T, F, MODE, KMAX, W>;
    static std::atomic<uint64_t> allowed{0};
    if (lds > 65536) allow_lds(reinterpret_cast<const void*>(fn), allowed);
    hipLaunchKernelGGL(fn, dim3(pa.nparts), dim3(64 * W), lds, s, pa, ticket, err, spin_limit, eval, dval, rhs, dd,
                       xp, xo);
}

template <typename T, typename F, int MODE, int KMAX, int W>
void launch_batch_one(hipStream_t s, size_t lds, int nitems, const int2* order, int* ticket, int* err,
                      long spin_limit, const BatchSys* sys, const BatchState* st, int want, int in, int out,
                      GraphRec* rec) {
    auto fn = k_batch_part<T, F, MODE, KMAX, W>;
    static std::atomic<uint64_t> allowed{0};
    if (lds > 65536) allow_lds(reinterpret_cast<const void*>(fn), allowed);
    launch_or_record_lds(rec, fn, dim3(nitems), dim3(64 * W), lds, s, order, ticket, err, spin_limit, sys, st, want, in,
                         out);
}

// the row lengths' register buckets: f(bucket, waves) as integral constants
template <bool CPLX, typename Fn> void part_bucket(int kmax, Fn&& f) {
    constexpr int W1 = part_waves(CPLX, 20), W2 = part_waves(CPLX, 32);
    using std::integral_constant;
    if (kmax <= 8) f(integral_constant<int, 8>{}, integral_constant<int, W1>{});
    else if (kmax <= 12) f(integral_constant<int, 12>{}, integral_constant<int, W1>{});
    else if (kmax <= 16) f(integral_constant<int, 16>{}, integral_constant<int, W1>{});
    else if (kmax <= 20) f(integral_constant<int, 20>{}, integral_constant<int, W1>{});
    else if (kmax <= 24) f(integral_constant<int, 24>{}, integral_constant<int, W2>{});
    else if (kmax <= 28) f(integral_constant<int, 28>{}, integral_constant<int, W2>{});
    else f(integral_constant<int, 32>{}, integral_constant<int, W2>{});
}

}  // namespace

template <typename T, typename F>
void launch_sweep_part(hipStream_t s, int mode, int kmax, size_t lds, const PartArgs& pa, int* ticket, int* err,
                       long spin_limit, const F* eval, const F* dval, const T* rhs, const T* dd, T* xp, T* xo) {
    if (pa.nparts <= 0) return;
    part_bucket<sizeof(T) == 16>(kmax, [&](auto k, auto w) {
        constexpr int K = decltype(k)::value, W = decltype(w)::value;
        if (mode == FWD_DIV_LAST)
            launch_one<T, F, FWD_DIV_LAST, K, W>(s, lds, pa, ticket, err, spin_limit, eval, dval, rhs, dd, xp, xo);
        else if (mode == BWD_IC)
            launch_one<T, F, BWD_IC, K, W>(s, lds, pa, ticket, err, spin_limit, eval, dval, rhs, dd, xp, xo);
        else
            launch_one<T, F, BWD_DIV_FIRST, K, W>(s, lds, pa, ticket, err, spin_limit, eval, dval, rhs, dd, xp, xo);
    });
}

template <typename T, typename F>
void launch_batch_part(hipStream_t s, int mode, int kmax, size_t lds, int nitems, const int2* order, int* ticket,
                       int* err, long spin_limit, const BatchSys* sys, const BatchState* st, int want, int in, int out,
                       GraphRec* rec) {
    if (nitems <= 0) return;
    part_bucket<sizeof(T) == 16>(kmax, [&](auto k, auto w) {
        constexpr int K = decltype(k)::value, W = decltype(w)::value;
        if (mode == FWD_DIV_LAST)
            launch_batch_one<T, F, FWD_DIV_LAST, K, W>(s, lds, nitems, order, ticket, err, spin_limit, sys, st, want, in,
                                                       out, rec);
        else if (mode == BWD_IC)
            launch_batch_one<T, F, BWD_IC, K, W>(s, lds, nitems, order, ticket, err, spin_limit, sys, st, want, in, out,
                                                 rec);
        else
            launch_batch_one<T, F, BWD_DIV_FIRST, K, W>(s, lds, nitems, order, ticket, err, spin_limit, sys, st, want,
                                                        in, out, rec);
    });
}

#define SSGPU_PTI(T, F)                                                                                           \
    template void launch_sweep_part<T, F>(hipStream_t, int, int, size_t, const PartArgs&, int*, int*, long,       \
                                          const F*, const F*, const T*, const T*, T*, T*);                        \
    template void launch_batch_part<T, F>(hipStream_t, int, int, size_t, int, const int2*, int*, int*, long,      \
                                          const BatchSys*, const BatchState*, int, int, int, GraphRec*);
SSGPU_PTI(double, double)
SSGPU_PTI(double, float)
SSGPU_PTI(zc, zc)
SSGPU_PTI(zc, fc)

}  // namespace ssgpu
