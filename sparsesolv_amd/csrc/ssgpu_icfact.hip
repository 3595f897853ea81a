// Shifted IC(0) factorization on gfx950 with a precomputed update list.
//
// The reference computes each entry of row i of lower(A) as
//   L_ij = a_ij - sum_{k<j} L_ik L_jk d_k      (j < i)
//   L_ii = alpha a_ii - sum_{k<i} L_ik^2 d_k,  d_i = 1/L_ii
// by searching row j for every k of row i (SprsPreconditioner.cpp:59-110).
// Which (k) match depends only on the sparsity pattern, so a symbolic pass
// records, for every off-diagonal entry, its list of updates in the
// reference's order: (slot of L_ik within row i, slot of the entry, position
// of L_jk).  The symbolic pass needs no ordering between rows and runs as one
// launch over all rows.
//
// The numeric pass is sync-free: one launch, a wave per row, rows taken by
// ticket in level order.  A row's inputs are the entries L_jk and the pivots
// d_k of rows at lower levels, hence of smaller tickets, so a wave that polls
// for them waits for rows that are running or done.  The factor's and the
// pivots' arrays are pre-filled with the sweeps' sentinel and polled with
// agent-scope loads.  Inside the row the updates run by column: lane m keeps
// entry m's running sum, and once entry k is final it is broadcast and every
// entry with an update by k subtracts (L_ik L_mk) d_k -- for each entry the
// reference's subtractions in the reference's order, so the factor is
// bit-identical to it, but the chain through a row is one broadcast, two
// products and a difference per column.  What bounds it is the chain of levels:
// publish, see, gather, and the chain through the row.  Factor and value
// copies at 95^3 6.8 ms, 40^3 1.6, 64^3 complex 4.6 (a launch per level, entry
// by entry: 24.9, 8.3, 16.9).  Wide levels (a multi-color order) run the same
// rows a launch per level, every row with a wave of its own and nothing polled:
// 60^3 in 12 colors 1.60 ms, 3.92 sync-free.
// Rows over 48 entries take the searching kernel, a launch per level.
#include <cfloat>
#include <type_traits>

#include <hipcub/hipcub.hpp>

#include "ssgpu_kernels.h"
#include "ssgpu_sweep_dev.h"

namespace ssgpu {

namespace {

// count (po == nullptr) or fill the update list of every entry of row p (the
// diagonal's updates are those by every entry of its own row and need no list)
__global__ __launch_bounds__(kBS) void k_ic_symbolic(int n, const int* __restrict__ prp, const int* __restrict__ pci,
                                                     const int* __restrict__ prow, const int* __restrict__ ppos,
                                                     int* __restrict__ cnt, const int* __restrict__ po,
                                                     unsigned char* __restrict__ u_slot,
                                                     unsigned char* __restrict__ u_entry, int* __restrict__ u_pos) {
    const int p = blockIdx.x * kBS + threadIdx.x;
    if (p >= n) return;
    const int i = prow[p];
    const int rs = prp[p], re = prp[p + 1];
    for (int jj = rs; jj < re; ++jj) {
        const int j = pci[jj];
        int c = 0;
        const int base = po ? po[jj] : 0;
        if (j < i) {
            const int q = ppos[j];
            int ll = prp[q];
            const int le = prp[q + 1];
            for (int kk = rs; kk < re; ++kk) {
                const int ck = pci[kk];
                if (!(ck <= j - 1)) break;
                while (ll < le && pci[ll] < ck) ++ll;
                if (ll < le && pci[ll] == ck) {
                    if (po) {
                        u_slot[base + c] = (unsigned char)(kk - rs);
                        u_entry[base + c] = (unsigned char)(jj - rs);
                        u_pos[base + c] = ll;
                    }
                    ++c;
                }
            }
        }
        if (!po) cnt[jj] = c;
    }
}

__device__ inline double absval(double a) { return fabs(a); }
__device__ inline double absval(zc a) { return hypot(a.re, a.im); }
__device__ inline double mulr(double v, double a) { return v * a; }
__device__ inline zc mulr(zc v, double a) { return v * a; }
__device__ inline double recip(double s) { return 1.0 / s; }
__device__ inline zc recip(zc s) { return zdiv(zc{1.0, 0.0}, s); }
// A signalling NaN made quiet, every other value as it is: entries without
// updates go from the matrix to the polled factor, where the sentinel, a
// signalling NaN, would be waited for.
__device__ inline double quiet(double v) { return __builtin_canonicalize(v); }
__device__ inline zc quiet(zc v) { return zc{quiet(v.re), quiet(v.im)}; }
template <typename T> __device__ inline T from_real(double a);
template <> __device__ inline double from_real<double>(double a) { return a; }
template <> __device__ inline zc from_real<zc>(double a) { return zc{a, 0.0}; }

__device__ inline double lane_value(double v, int lane) {
    return __longlong_as_double(((long long)__builtin_amdgcn_readlane(__double2hiint(v), lane) << 32) |
                                (unsigned)__builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ inline zc lane_value(zc v, int lane) { return zc{lane_value(v.re, lane), lane_value(v.im, lane)}; }
__device__ inline double pick(bool c, double a, double b) { return c ? a : b; }
__device__ inline zc pick(bool c, zc a, zc b) { return zc{c ? a.re : b.re, c ? a.im : b.im}; }

template <bool LEVEL, typename T> __device__ inline void put(T* p, T v) {   // LEVEL: no reader before the launch ends
    if (LEVEL) *p = v;
    else gstore(p, v);
}

// One wave per row, a ticket per workgroup.  KROW: most entries of a row, the
// diagonal included.  LEVEL: rows [p0, p1) are one level, whose inputs earlier
// launches have written, so nothing is polled and every row has its own wave.
constexpr int kFactUpd = 4;        // updates per lane in flight
constexpr int kFactWaves = 4096;   // waves in all

template <typename T, int KROW, int WAVES, bool LEVEL>
__global__ __launch_bounds__(64 * WAVES) void k_ic_numeric(int p0, int p1, int nticket, int* __restrict__ ticket,
                                                           int* __restrict__ err, long spin_limit,
                                                           const int* __restrict__ prp, const int* __restrict__ pci,
                                                           const int* __restrict__ prow,
                                                           const int* __restrict__ map, const T* __restrict__ av,
                                                           const int* __restrict__ po,
                                                           const unsigned char* __restrict__ u_slot,
                                                           const unsigned char* __restrict__ u_entry,
                                                           const int* __restrict__ u_pos, T* __restrict__ fv,
                                                           T* __restrict__ diagD, double accel,
                                                           int* __restrict__ nfix) {
    // the row's L_mk by (k, m), and which of them exist
    __shared__ T s_upd[WAVES][KROW * KROW];
    __shared__ unsigned long long s_mask[WAVES][KROW];
    __shared__ int s_ticket, s_stop;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    T* const upd = s_upd[wave];
    unsigned long long* const has = s_mask[wave];
    if (!LEVEL && threadIdx.x == 0) s_stop = 0;
    while (true) {
        int t = blockIdx.x;
        if (!LEVEL) {
            __syncthreads();   // every wave is done with the previous ticket
            if (threadIdx.x == 0) s_ticket = s_stop ? nticket : atomicAdd(ticket, 1);
            __syncthreads();
            t = __builtin_amdgcn_readfirstlane(s_ticket);
            if (t >= nticket) return;
        }
        const int p = p0 + t * WAVES + wave;
        if (p < p1) {
            const int i = prow[p];
            const int rs = prp[p], len = prp[p + 1] - rs;
            const int u0 = po[rs], nu = po[rs + len] - u0;
            const bool mine = lane < len, last = lane == len - 1;
            const int col = mine && !last ? pci[rs + lane] : -1;
            T sum = Num<T>::zero();
            if (mine) sum = quiet(av[map[rs + lane]]);
            if (last) sum = mulr(sum, accel);
            if (lane < KROW) has[lane] = 0;
            // the row's inputs: pivots of its columns, and the entries of its updates
            T d = Num<T>::zero();
            bool wait_d = col >= 0;
            long spins = 0;
            bool ok = true;
            for (int b = 0; (b < nu || b == 0) && ok; b += 64 * kFactUpd) {
                int pos[kFactUpd], at[kFactUpd];
                unsigned miss = 0;
#pragma unroll
                for (int q = 0; q < kFactUpd; ++q) {
                    const int e = b + 64 * q + lane;
                    pos[q] = 0;
                    at[q] = 0;
                    if (e < nu) {
                        const int k = u_slot[u0 + e], m = u_entry[u0 + e];
                        pos[q] = u_pos[u0 + e];
                        at[q] = k * KROW + m;
                        atomicOr(&has[m], 1ull << k);
                        miss |= 1u << q;
                    }
                }
                while (true) {
                    __asm__ __volatile__("" ::: "memory");
                    const unsigned want = miss;
                    const bool want_d = wait_d;
                    T v[kFactUpd];
                    if (want_d) d = LEVEL ? diagD[col] : gload(diagD + col);
#pragma unroll
                    for (int q = 0; q < kFactUpd; ++q)
                        if ((want >> q) & 1u) v[q] = LEVEL ? fv[pos[q]] : gload(fv + pos[q]);
                    if (want_d && (LEVEL || !sent(d))) wait_d = false;
#pragma unroll
                    for (int q = 0; q < kFactUpd; ++q)
                        if (((want >> q) & 1u) && (LEVEL || !sent(v[q]))) {
                            upd[at[q]] = v[q];
                            miss &= ~(1u << q);
                        }
                    if (LEVEL || !__any(miss != 0u || wait_d)) break;
                    if (__any(miss != want || wait_d != want_d) && spin_limit > 0) spins = 0;
                    if (++spins > spin_limit) {
                        ok = false;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                }
            }
            if (!ok) {   // the workgroup leaves at its next ticket, and later rows at their own limits
                if (lane == 0) {
                    atomicOr(err, 1);
                    s_stop = 1;
                }
                continue;
            }
            __asm__ __volatile__("" ::: "memory");
            const unsigned long long mask = lane < KROW ? has[lane] : 0ull;
            T in[KROW];
#pragma unroll
            for (int k = 0; k < KROW; ++k) in[k] = upd[k * KROW + (lane < KROW ? lane : 0)];
#pragma unroll
            for (int k = 0; k < KROW - 1; ++k)
                if (k < len - 1) {
                    const T lik = lane_value(sum, k), dk = lane_value(d, k);
                    // (L_ik * L_mk) * d_k, SprsPreconditioner.cpp:75 / :98
                    const T x = Num<T>::sub(sum, Num<T>::mul(Num<T>::mul(lik, pick(last, lik, in[k])), dk));
                    sum = pick(last || ((mask >> k) & 1ull), x, sum);
                }
            if (mine) put<LEVEL>(fv + rs + lane, sum);
            if (last) {
                T piv;
                if (absval(sum) < 1.0e-12) {
                    piv = from_real<T>(1.0 / DBL_EPSILON);
                    atomicAdd(nfix, 1);
                } else {
                    piv = recip(sum);
                }
                put<LEVEL>(diagD + i, piv);
            }
        }
        if (LEVEL) return;
    }
}

inline int grid_of(int64_t n, int bs) { return (int)std::max<int64_t>(1, (n + bs - 1) / bs); }

}  // namespace

void launch_ic_symbolic_count(hipStream_t s, int n, const int* prp, const int* pci, const int* prow, const int* ppos,
                              int* cnt) {
    hipLaunchKernelGGL(k_ic_symbolic, dim3(grid_of(n, kBS)), dim3(kBS), 0, s, n, prp, pci, prow, ppos, cnt, nullptr,
                       nullptr, nullptr, nullptr);
}

size_t scan_tmp_bytes(int nitems) {
    size_t bytes = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, (const int*)nullptr, (int*)nullptr, nitems);
    return bytes;
}

void launch_exclusive_scan(hipStream_t s, const int* in, int* out, int nitems, void* tmp, size_t tmp_bytes) {
    (void)hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, in, out, nitems, s);
}

void launch_ic_symbolic_fill(hipStream_t s, int n, const int* prp, const int* pci, const int* prow, const int* ppos,
                             const int* po, void* u_slot, void* u_entry, int* u_pos) {
    hipLaunchKernelGGL(k_ic_symbolic, dim3(grid_of(n, kBS)), dim3(kBS), 0, s, n, prp, pci, prow, ppos, nullptr, po,
                       (unsigned char*)u_slot, (unsigned char*)u_entry, u_pos);
}

template <typename T>
void launch_ic_numeric(hipStream_t s, int kmax_row, int p0, int p1, bool level, int* ticket, int* err, long spin_limit,
                       const int* prp, const int* pci, const int* prow, const int* map, const T* av, const int* po,
                       const void* u_slot, const void* u_entry, const int* u_pos, T* fv, T* diagD, double accel,
                       int* nfix) {
    if (p1 <= p0) return;
    const unsigned char *sl = (const unsigned char*)u_slot, *en = (const unsigned char*)u_entry;
    constexpr int C = (int)(sizeof(T) / sizeof(double));
    // a row to each wave of a workgroup per ticket (two rows: 2.4x at 40^3, 1.5x
    // at 95^3: a level then takes two rows' chains), kFactWaves waves in all
    // (95^3: 13.5 ms with 1024, 8.3 with 2048, 6.8 with 4096; 40^3 the same)
    auto go = [&](auto krow, auto w) {
        constexpr int K = decltype(krow)::value, W = decltype(w)::value;
        const int nt = (p1 - p0 + W - 1) / W;
        if (level)
            hipLaunchKernelGGL((k_ic_numeric<T, K, W, true>), dim3(nt), dim3(64 * W), 0, s, p0, p1, nt, ticket, err,
                               spin_limit, prp, pci, prow, map, av, po, sl, en, u_pos, fv, diagD, accel, nfix);
        else
            hipLaunchKernelGGL((k_ic_numeric<T, K, W, false>), dim3(std::min(nt, kFactWaves / W)), dim3(64 * W), 0, s,
                               p0, p1, nt, ticket, err, spin_limit, prp, pci, prow, map, av, po, sl, en, u_pos, fv,
                               diagD, accel, nfix);
    };
    using std::integral_constant;
    if (kmax_row <= 20) go(integral_constant<int, 20>{}, integral_constant<int, 8 / C>{});
    else if (kmax_row <= 32) go(integral_constant<int, 32>{}, integral_constant<int, 4 / C>{});
    else go(integral_constant<int, 48>{}, integral_constant<int, 2 / C>{});
}
template void launch_ic_numeric<double>(hipStream_t, int, int, int, bool, int*, int*, long, const int*, const int*,
                                        const int*, const int*, const double*, const int*, const void*, const void*,
                                        const int*, double*, double*, double, int*);
template void launch_ic_numeric<zc>(hipStream_t, int, int, int, bool, int*, int*, long, const int*, const int*,
                                    const int*, const int*, const zc*, const int*, const void*, const void*,
                                    const int*, zc*, zc*, double, int*);

}  // namespace ssgpu
