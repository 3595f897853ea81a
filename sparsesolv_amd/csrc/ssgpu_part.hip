// Partitioned triangular sweeps for gfx950 (layout: ssgpu_parts.h).
//
// A sweep is a chain of dependent levels, and what a level costs is how long
// one result takes to reach the row that waits for it.  Through device memory
// that is about 1.5 us (store, coherence, poll); through LDS it is a few
// hundred clocks.  So each workgroup owns a part of the rows (an interval of
// the row index, or a cell of a grid) and keeps their results in LDS: only the
// inputs that cross parts go through device memory, and they are polled ahead
// of the level that needs them.
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
// 1588 levels) 0.72 / 0.74, before 2.43 / 2.78; 40^3 0.25 / 0.25, before 0.91
// / 1.08; 10^3 0.050 / 0.049, before 0.185 / 0.190; 64^3 complex 0.73 / 0.78,
// before 2.56 / 2.76.  A level costs about 700 clocks in a part (an LDS hop
// and poll 250, the late inputs' gather and the row's serial sum 250,
// publishing 100), and a step's loads, polls and early sums are hidden as long
// as the W waves together keep ahead of that pace; at 95^3 they are not quite
// (0.45 us a level against 0.35 at 10^3 and 0.39 at 24^3 to 60^3), since polls
// of device memory take 1.5 us there.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "ssgpu_kernels.h"
#include "ssgpu_part_dev.h"

namespace ssgpu {

namespace {

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
    constexpr int kNear = ROWS ? 2 : 1;   // rows lie in more lines than positions do: polled earlier
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
            if (!wait_steps(S.need - kNear * (int)S.near, lds_at(&s_done), wait_limit)) {
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
                if (++spins > spin_limit || sweep_failed(spins, err)) {
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
// Whole iterations, chunked against in parts: 64 systems of n=8..40 3.60 -> 1.66
// ms, one of n=60 3.44 -> 1.35, 8 of n=60 4.99 -> 1.87, 32 of n=60 11.6 -> 6.2,
// two of n=95 6.87 -> 2.71 ms (polled as late as the one-column sweep does:
// 1.88, 1.55, 2.19, 7.2, 3.02).
template <typename T, typename F, int MODE, int KMAX, int W>
__global__ __launch_bounds__(64 * W) void k_batch_part(const int2* __restrict__ order, int nitems,
                                                       int* __restrict__ ticket,
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
    const int item = __builtin_amdgcn_readfirstlane(s_item);
    if (item >= nitems) return;
    const int2 it = order[item];
    const int sy = __builtin_amdgcn_readfirstlane(it.x), part = __builtin_amdgcn_readfirstlane(it.y);
    if (st[sy].status != want) return;
    const BatchSys& S = sys[sy];
    const BatchPart& P = MODE == FWD_DIV_LAST ? S.f_part : S.b_part;
    part_sweep<T, F, MODE, KMAX, W, true>(P.args, part, lx, s_done, err, spin_limit, static_cast<const F*>(P.eval),
                                          static_cast<const F*>(P.dval), static_cast<const T*>(S.vec[in]),
                                          static_cast<const T*>(S.diagD), nullptr, static_cast<T*>(S.vec[out]));
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
    launch_or_record_lds(rec, fn, dim3(nitems), dim3(64 * W), lds, s, order, nitems, ticket, err, spin_limit, sys, st,
                         want, in, out);
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
// of a batch, whose systems share a launch: fewer
template <bool CPLX, typename Fn> void batch_bucket(int kmax, Fn&& f) {
    constexpr int W1 = part_waves(CPLX, 20), W2 = part_waves(CPLX, 32);
    using std::integral_constant;
    if (kmax <= 12) f(integral_constant<int, 12>{}, integral_constant<int, W1>{});
    else if (kmax <= 20) f(integral_constant<int, 20>{}, integral_constant<int, W1>{});
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
    batch_bucket<sizeof(T) == 16>(kmax, [&](auto k, auto w) {
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
