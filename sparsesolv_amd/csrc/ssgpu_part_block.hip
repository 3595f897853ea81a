// Partitioned triangular sweeps of several right-hand sides for gfx950: the
// parts of ssgpu_part.hip, each workgroup with C columns of its part.
#include <type_traits>

#include "ssgpu_part_dev.h"

namespace ssgpu {

namespace {

// The columns of a row lie side by side (entry (i, c) at i * kb + c).  A lane
// holds one row and one column: RL lanes hold a step's rows, and the 64 / RL
// groups of them different columns, so a workgroup solves C = 64 / RL columns
// with one read of the entries.  Ticket t is column group t mod G of part
// t / G: inputs lie at smaller tickets.  Externals are polled by row in x
// (sentinel-filled), the C columns of a row by adjacent lanes, kNear times as
// far ahead as the one-column sweep does: they are more, and lie in more lines.
// LDS holds the one-column layout's slots with C values each.  A column's
// result is formed as the one-column sweep forms it.
//
// Steps of a cell of a grid hold up to 32 rows, so C is 2 there at no cost in
// lanes.  Bound by the chain of levels while the column groups' parts fit the
// compute units, by the units (1 workgroup each) beyond.  An IC-MRTR iteration
// in chunks (k_sweep_il) and in parts, ms: 10^3 x 8 0.53 / 0.21, 24^3 x 8 1.39 /
// 0.58, 40^3 x 2 2.37 / 0.82 (a sweep 0.34), 40^3 x 32 3.05 / 1.60, complex COCG
// 28^3 x 32 2.60 / 1.21.  Two columns in a lane as well (C = 4) need 192
// registers, hence 8 waves instead of 12, and took 0.70 ms a sweep at 40^3 x 32
// against 0.53.  Polled only as far ahead as the one-column sweep does, the
// 40^3 x 2 iteration takes 1.02 ms, 3 times as far the 24^3 x 2 one 5% longer
// than twice.
constexpr int kNear = 2;
template <typename T, typename F, int MODE, int KMAX, int W, int RL>
__global__ __launch_bounds__(64 * W) void k_block_part(PartArgs pa, int kb_log2, int* __restrict__ ticket,
                                                       int* __restrict__ err, long spin_limit,
                                                       const F* __restrict__ eval, const F* __restrict__ dval,
                                                       const T* __restrict__ rhs, const T* __restrict__ dd,
                                                       T* __restrict__ x) {
    constexpr int C = 64 / RL;
    constexpr int EB = 64 / C;   // externals a wave polls per load
    constexpr int NB = 4;        // loads of a polling pass
    constexpr bool kFwd = MODE == FWD_DIV_LAST;
    extern __shared__ __align__(16) unsigned char part_lds[];
    __shared__ int s_item, s_done;
    T* lx = reinterpret_cast<T*>(part_lds);
    if (threadIdx.x == 0) {
        s_item = atomicAdd(ticket, 1);
        s_done = 0;
    }
    if (threadIdx.x < C) lx[threadIdx.x] = Num<T>::zero();
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(s_item);
    const int groups_log2 = kb_log2 - (C - 1);   // C is 1 or 2
    const int part = item >> groups_log2;
    if (part >= pa.nparts) return;
    const int lane = threadIdx.x & 63, lr = lane % RL, lc = lane / RL;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int s0 = pa.part_step[part], s1 = pa.part_step[part + 1];
    T* const stage = lx + (size_t)(1 + wave * kPartExt) * C;
    T* const mine = lx + (size_t)(1 + W * kPartExt) * C;
    const unsigned base = lds_at(lx) + (unsigned)(lc * sizeof(T));
    rhs += (item & ((1 << groups_log2) - 1)) * C;   // the workgroup's columns
    x += (item & ((1 << groups_log2) - 1)) * C;
    const int wait_limit = (int)(spin_limit < (1L << 24) ? spin_limit * 64 : 1L << 30);
    auto give_up = [&](int* done_p) {   // a wave that waited past the limit stops its part
        if ((threadIdx.x & 63) == 0) {
            atomicOr(err, 1);
            __hip_atomic_store(done_p, kAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    int st = s0 + wave;
    if (st >= s1) return;
    PartStep S = pa.steps[st];
    int ep[NB], row;
    auto externals = [&](const PartStep& Q, int from, int (&e)[NB]) {   // their rows, -1 past the last
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int j = from + b * EB + lane / C;
            e[b] = j < Q.next ? pa.ext[Q.ext0 + j] : -1;
            if (e[b] >= 0) e[b] = pa.srow[e[b]];
        }
    };
    externals(S, 0, ep);
    row = lr < S.cnt ? pa.srow[S.pos0 + lr] : 0;
    while (true) {
        const bool active = lr < S.cnt;
        // --- the step's rows and entries (padding as in the one-column sweep) --------
        PartRow<T, F, KMAX> R;
        const int qn = (int)S.quads, qskip = kFwd ? KMAX / 4 - qn : 0;
        const int l4 = 4 * min(lr, (int)S.cnt - 1);
        ushort4 sl[KMAX / 4];
#pragma unroll
        for (int q = 0; q < KMAX / 4; ++q) {
            const int j = q - qskip;
            const int at = j >= 0 && j < qn ? S.ent + 4 * j * (int)S.cnt : 0;
            load4(eval + at + l4, R.vals + 4 * q);
            sl[q] = *reinterpret_cast<const ushort4*>(pa.slot + at + l4);
        }
        const size_t xat = ((size_t)row << kb_log2) + lc;
        R.r_i = Num<T>::zero();
        R.d_i = unit((T*)nullptr);
        if (active) {
            R.r_i = rhs[xat];
            if (MODE == BWD_IC) R.d_i = dd[row];
            else R.d_i = wid<T, F>(dval[S.pos0 + lr]);
        }
        const bool more = st + W < s1;
        const PartStep N = pa.steps[more ? st + W : st];
        // --- externals into LDS -------------------------------------------------------
        if (S.next > 0) {
            if (!wait_steps(S.need - kNear * (int)S.near, lds_at(&s_done), wait_limit)) {
                give_up(&s_done);
                return;
            }
            for (int from = 0; from < S.next; from += NB * EB) {
                if (from > 0) externals(S, from, ep);
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
                        if ((want >> b) & 1u) v[b] = gload(x + ((size_t)ep[b] << kb_log2) + lane % C);
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        if (((want >> b) & 1u) && !sent(v[b])) {
                            stage[(from + b * EB) * C + lane] = v[b];
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
        }
        const typename RecipOf<T>::type rc(R.d_i);
#pragma unroll
        for (int k = 0; k < KMAX; ++k) {
            const ushort4 v = sl[k / 4];
            const unsigned slot = k % 4 == 0 ? v.x : k % 4 == 1 ? v.y : k % 4 == 2 ? v.z : v.w;
            R.at[k] = slot * (unsigned)(C * sizeof(T)) + base;
            settle(R.at[k]);
            settle(R.vals[k]);
        }
        settle(R.r_i);
        settle(R.d_i);
        int epn[NB];
        externals(N, 0, epn);
        const int rown = lr < N.cnt ? pa.srow[N.pos0 + lr] : 0;
        // --- the rows -------------------------------------------------------------------
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
        if (active) mine[(S.lpos + lr) * C + lc] = res;
        lds_order();
        if (lane == 0)   // no wait on the results before it: a wave's LDS operations are performed in order
            __asm__ __volatile__("ds_add_u32 %0, %1" ::"v"(lds_at(&s_done)), "v"(1) : "memory");
        __builtin_amdgcn_s_setprio(0);
        if (active) gstore(x + xat, res);
        if (!more) return;
        st += W;
        S = N;
        row = rown;
#pragma unroll
        for (int b = 0; b < NB; ++b) ep[b] = epn[b];
    }
}

template <typename T, typename F, int MODE, int KMAX, int RL>
bool launch_rows(hipStream_t s, size_t slots, const PartArgs& pa, int kb_log2, int* ticket, int* err, long spin_limit,
                 const F* eval, const F* dval, const T* rhs, const T* dd, T* x) {
    constexpr int C = 64 / RL, W = part_waves(sizeof(T) == 16, KMAX);
    const size_t lds = slots * C * sizeof(T);
    if (C > (1 << kb_log2) || lds > kPartLdsMax) return false;
    auto fn = k_block_part<T, F, MODE, KMAX, W, RL>;
    static std::atomic<uint64_t> allowed{0};
    if (lds > 65536) allow_lds(reinterpret_cast<const void*>(fn), allowed);
    hipLaunchKernelGGL(fn, dim3(pa.nparts << (kb_log2 - (C - 1))), dim3(64 * W), lds, s, pa, kb_log2, ticket, err,
                       spin_limit, eval, dval, rhs, dd, x);
    return true;
}

}  // namespace

template <typename T, typename F>
bool launch_sweep_block_part(hipStream_t s, int mode, int kmax, size_t slots, int step_rows, const PartArgs& pa, int kb,
                             int* ticket, int* err, long spin_limit, const F* eval, const F* dval, const T* rhs,
                             const T* dd, T* x) {
    if (pa.nparts <= 0 || kmax > kPartMaxLen) return false;
    int kb_log2 = 0;
    while ((1 << kb_log2) < kb) ++kb_log2;
    auto rows = [&](auto mode_c, auto kmax_c) {
        constexpr int M = decltype(mode_c)::value, K = decltype(kmax_c)::value;
        return (step_rows <= 32 && launch_rows<T, F, M, K, 32>(s, slots, pa, kb_log2, ticket, err, spin_limit, eval,
                                                               dval, rhs, dd, x)) ||
               launch_rows<T, F, M, K, 64>(s, slots, pa, kb_log2, ticket, err, spin_limit, eval, dval, rhs, dd, x);
    };
    auto bucket = [&](auto mode_c) {
        using std::integral_constant;
        if (kmax <= 12) return rows(mode_c, integral_constant<int, 12>{});
        if (kmax <= 20) return rows(mode_c, integral_constant<int, 20>{});
        return rows(mode_c, integral_constant<int, 32>{});
    };
    if (mode == FWD_DIV_LAST) return bucket(std::integral_constant<int, FWD_DIV_LAST>{});
    if (mode == BWD_IC) return bucket(std::integral_constant<int, BWD_IC>{});
    return bucket(std::integral_constant<int, BWD_DIV_FIRST>{});
}

#define SSGPU_BPI(T, F)                                                                                            \
    template bool launch_sweep_block_part<T, F>(hipStream_t, int, int, size_t, int, const PartArgs&, int, int*, \
                                                int*, long, const F*, const F*, const T*, const T*, T*);
SSGPU_BPI(double, double)
SSGPU_BPI(double, float)
SSGPU_BPI(zc, zc)
SSGPU_BPI(zc, fc)

}  // namespace ssgpu
