// LU with partial pivoting as a pipeline of column groups (LU::new,
// src/linalg/lu.rs:93-122, 337-389).
//
// A workgroup holds W columns of the range in registers (thread t rows t,
// t + CT, ... for CT threads).  It takes the earlier groups in order: their pivots, then their
// L columns, which give it the U rows of its own columns and the update of the
// rest; then it factors its W columns and publishes each L column and pivot as
// it is made.  Every element sees nalgebra's operations in nalgebra's order.
//
// What bounds it is the chain over the columns, a pivot search and an
// elimination each, and the hand-over from group to group:
//   * rows never move: each thread carries the positions of its rows, and a
//     swap is two compares per row, so one barrier per column is left (every
//     wavefront parks its best row before it, and the winner's is used after);
//   * an L column is published under the positions its group started with,
//     which is what the other groups' threads know, so pivots and L columns are
//     fetched together;
//   * a published element is its own flag (the buffer starts as a signalling
//     NaN pattern; a value that is this very pattern is published quieted).
// Group tickets are taken in column order, so the group that is waited for is
// running.  Waits are bounded: a group that gives up takes NaN for what it waited
// for and sets info to -1.
// The range is the whole matrix up to WHOLE_ROWS rows (one launch instead of
// some hundred: 500 x 500 2.45 -> 0.69 ms) and 64 columns above it (the
// trailing matrix then takes rank-64 updates; 4096 x 4096 FAST 25.3 -> 13.3 ms).
#pragma once
#include "lu_kernels.hpp"
#include "solve_sweep.hpp"

namespace nrocm_lu {

// Threads, rows per thread and columns per group by the rows of the range.
// The columns and the L columns being applied to them fill the registers.  Eight
// columns where they fit: 16 make the U rows of a group (one wavefront's
// triangular solve) and the code longer than the hand-overs they save (500 x
// 500: 13.3 us per eight columns against 10.5).
template <int CT_, int RPT_, int W_>
struct Group {
    static constexpr int CT = CT_, RPT = RPT_, W = W_, ROWS = CT * RPT;
};
using Group256 = Group<256, 1, 8>;
using Group512 = Group<512, 1, 8>;
using Group1K = Group<512, 2, 8>;
using Group2K = Group<512, 4, 8>;
using Group4K = Group<512, 8, 4>;
using Group8K = Group<512, 16, 2>;
using Group16K = Group<512, 32, 1>;
constexpr int COLUMNS_ROWS_MAX = Group16K::ROWS;
constexpr long COL_SPIN_LIMIT = 1L << 21;  // some seconds

template <typename T> struct ColWord;
template <> struct ColWord<double> {
    typedef unsigned long long U;
    static constexpr U EMPTY = 0x7ff0000000000001ull, QUIET = 0x0008000000000000ull;
    static __device__ __forceinline__ U bits(double v) { return (U)__double_as_longlong(v); }
    static __device__ __forceinline__ double value(U u) { return __longlong_as_double((long long)u); }
};
template <> struct ColWord<float> {
    typedef unsigned U;
    static constexpr U EMPTY = 0x7f800001u, QUIET = 0x00400000u;
    static __device__ __forceinline__ U bits(float v) { return __float_as_uint(v); }
    static __device__ __forceinline__ float value(U u) { return __uint_as_float(u); }
};

constexpr int PIV_SKIP = 1 << 30;  // the column had no pivot: no swap, no elimination

// acc[q] = fl(fl((-u[q]) * l) + acc[q]) (gauss_step, lu.rs:385-387), operand
// order as in sub_prod; two statements per element, so that the elements of a
// row interleave.
template <int N>
__device__ __forceinline__ void eliminate(double (&acc)[N], const double (&u)[N], double l, int from)
{
    double t[N];
#pragma unroll
    for (int q = 0; q < N; ++q)
        if (q >= from) asm("v_mul_f64 %0, -%1, %2" : "=v"(t[q]) : "v"(u[q]), "v"(l));
#pragma unroll
    for (int q = 0; q < N; ++q)
        if (q >= from) asm("v_add_f64 %0, %1, %0" : "+v"(acc[q]) : "v"(t[q]));
}
template <int N>
__device__ __forceinline__ void eliminate(float (&acc)[N], const float (&u)[N], float l, int from)
{
#pragma unroll
    for (int q = 0; q < N; ++q)
        if (q >= from) {
            const float p = (-u[q]) * l;
            acc[q] = p + acc[q];
        }
}

// A thread's row to LDS, 16 bytes at a time.
template <typename T, int W>
__device__ __forceinline__ void store_row(T *dst, const T (&a)[W])
{
    constexpr int N = W * (int)sizeof(T) < 16 ? W : 16 / (int)sizeof(T);
    typedef T V __attribute__((ext_vector_type(N)));
#pragma unroll
    for (int q = 0; q < W; q += N) {
        V v;
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = a[q + e];
        *(V *)(dst + q) = v;
    }
}

__device__ __forceinline__ double uniform_lane63(double v) { return nrocm_sweep::lane_value(v, 63); }
__device__ __forceinline__ float uniform_lane63(float v)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Columns [c0, c0 + ncols) of the m-row matrix A, diagonal positions c0..;
// columns below kend are factored.  V (ldv rows): published L columns, by
// column - c0 and position; H: pivots.  The rows that a group finishes go to A,
// the L columns below them only if no later group moves rows (last factored
// group); lu_left_kernel stores the others from V.
template <typename T, typename G>
__global__ __launch_bounds__(G::CT) void lu_columns_kernel(T *A, int lda, int m, int c0, int ncols, int kend, int *ipiv,
                                                        int *info, typename ColWord<T>::U *V, int ldv,
                                                        typename ColWord<T>::U *H, int *ticket, long limit)
{
    typedef typename ColWord<T>::U U;
    constexpr U EMPTY = ColWord<T>::EMPTY;
    constexpr int CT = G::CT, RPT = G::RPT, W = G::W, NW = CT / 64;
    __shared__ __align__(16) T cand[2][NW][W];   // every wavefront's best row
    __shared__ int piv_word[W];                  // the group's pivots, as published
    __shared__ T red_v[2][NW];
    __shared__ int red_p[2][NW];
    __shared__ T top[W][W + 1], L11[W][W + 1], Us[W][W];
    __shared__ int my;
    const int t = threadIdx.x, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    if (t == 0) my = atomicAdd(ticket, 1);
    __syncthreads();
    const int g = __builtin_amdgcn_readfirstlane(my);
    const int cg = c0 + g * W;
    const int wc = min(W, c0 + ncols - cg);
    const int nfac = (kend - c0 + W - 1) / W;  // factored groups
    constexpr int NOWHERE = 1 << 29;           // position of a thread's rows past the matrix

    T a[RPT][W];
    int pos[RPT];
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const int r = c0 + t + CT * s;
        pos[s] = r < m ? r : NOWHERE;
        const T *row = A + min(r, m - 1) + (size_t)cg * lda;
#pragma unroll
        for (int q = 0; q < W; ++q) a[s][q] = (r < m && q < wc) ? row[(size_t)q * lda] : T(0);
    }

    // ---- the earlier groups
    const int hend = min(g, nfac);
    for (int h = 0; h < hend; ++h) {
        const int kh = c0 + h * W;
        const int fc = min(W, kend - kh);
        U w[RPT][W], hw[W];
        auto issue = [&]() {
#pragma unroll
            for (int k = 0; k < W; ++k) hw[k] = __hip_atomic_load(H + (kh - c0) + min(k, fc - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int s = 0; s < RPT; ++s) {
                // finished rows and rows past the matrix look at some published row
                const int p = pos[s] < kh ? kh : min(pos[s], m - 1);
                const U *src = V + (size_t)(kh - c0) * ldv + p;
#pragma unroll
                for (int k = 0; k < W; ++k)
                    w[s][k] = __hip_atomic_load(src + (size_t)min(k, fc - 1) * ldv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        long spins = 0;
        bool lost = false;
        for (;;) {
            issue();
            bool ok = true;
#pragma unroll
            for (int k = 0; k < W; ++k) {
                ok = ok && hw[k] != EMPTY;
#pragma unroll
                for (int s = 0; s < RPT; ++s) ok = ok && w[s][k] != EMPTY;
            }
            lost = !ok && ++spins >= limit;
            if (ok || lost) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (__builtin_expect(lost, 0)) {
            __hip_atomic_store(info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int k = 0; k < W; ++k) {
                hw[k] = hw[k] == EMPTY ? (U)(kh + k) : hw[k];  // no swap: positions stay valid
#pragma unroll
                for (int s = 0; s < RPT; ++s) w[s][k] = EMPTY | ColWord<T>::QUIET;
            }
        }
        // the group's swaps
        unsigned skip = 0;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            if (k < fc) {
                const int word = __builtin_amdgcn_readfirstlane((int)hw[k]);
                if (word & PIV_SKIP) skip |= 1u << k;
                const int pk = word & ~PIV_SKIP, at = kh + k;
#pragma unroll
                for (int s = 0; s < RPT; ++s) {
                    const int y = pos[s] == at ? pk : pos[s];
                    pos[s] = pos[s] == pk ? at : y;
                }
            } else {
                skip |= 1u << k;
            }
        }
        // rows that it finished: U12 = L11^{-1} A12 over its W rows
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int i = pos[s] - kh;
            if (i >= 0 && i < fc) {
#pragma unroll
                for (int q = 0; q < W; ++q) {
                    top[i][q] = a[s][q];
                    L11[i][q] = ColWord<T>::value(w[s][q]);
                }
            }
        }
        lds_barrier();
        if (wv == 0) {
            const int q = lane < W ? lane : 0;
            T u[W];
#pragma unroll
            for (int i = 0; i < W; ++i) u[i] = i < fc ? top[i][q] : T(0);
#pragma unroll
            for (int i = 0; i < W; ++i) {
                if (!(skip >> i & 1)) {
#pragma unroll
                    for (int r = i + 1; r < W; ++r) {
                        T x[1] = {u[r]};
                        const T y[1] = {u[i]};
                        eliminate<1>(x, y, L11[r][i], 0);
                        u[r] = x[0];
                    }
                }
            }
            if (lane < W) {
#pragma unroll
                for (int i = 0; i < W; ++i) {
                    Us[i][q] = u[i];
                    if (i < fc && q < wc) A[kh + i + (size_t)(cg + q) * lda] = u[i];
                }
            }
        }
        lds_barrier();
        // the rows below, in increasing k
#pragma unroll
        for (int k = 0; k < W; ++k) {
            if (!(skip >> k & 1)) {
                T u[W];
#pragma unroll
                for (int q = 0; q < W; ++q) u[q] = Us[k][q];
#pragma unroll
                for (int s = 0; s < RPT; ++s) eliminate<W>(a[s], u, ColWord<T>::value(w[s][k]), 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // The columns have arrived on every path: without this the first use of a
    // register that only some path has waited for would wait for every store
    // issued before it, once per column.
#pragma unroll
    for (int s = 0; s < RPT; ++s)
#pragma unroll
        for (int q = 0; q < W; ++q) a[s][q] = pass(a[s][q]);

    // ---- its own columns
    const int fc = g < nfac ? min(W, kend - cg) : 0;
    const bool last = g + 1 >= nfac;
    int first_zero = 0;
    U *Vp[RPT];
    bool live[RPT];
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        live[s] = pos[s] >= cg && pos[s] < m;
        Vp[s] = V + (size_t)(cg - c0) * ldv + (live[s] ? pos[s] : cg);
    }
#pragma unroll
    for (int c = 0; c < W; ++c) {
        if (c < fc) {
            const int k = cg + c, par = c & 1;
            // icamax (src/base/min_max.rs:221-241): the largest |x|, ties to the
            // lowest position, a NaN only where it is at position k.  First the
            // value, then the lowest position that has it: no mask logic on the way
            T v[RPT], bv = T(-1);
#pragma unroll
            for (int s = 0; s < RPT; ++s) {
                T x = fabs(a[s][c]);
                x = (x != x) ? ((pos[s] == k) ? T(__builtin_inf()) : T(-1)) : x;
                v[s] = (pos[s] >= k && pos[s] < m) ? x : T(-1);
                bv = max_dpp(bv, v[s]);
            }
            bv = max_wave<T>(bv);
            const T wmax = uniform_lane63(bv);
            int bp = 0x7fffffff;
#pragma unroll
            for (int s = 0; s < RPT; ++s) bp = min(bp, v[s] == wmax && wmax >= T(0) ? pos[s] : 0x7fffffff);
            bp = min_wave(bp);
            const int best = __builtin_amdgcn_readlane(bp, 63);
#pragma unroll
            for (int s = 0; s < RPT; ++s)
                if (pos[s] == best) {
                    store_row<T, W>(cand[par][wv], a[s]);
                }
            if (lane == 63) {
                red_v[par][wv] = bv;
                red_p[par][wv] = bp;
            }
            lds_barrier();
            // the wavefronts' results, one per lane of each eight, the same way
            static_assert(NW == 8 || NW == 4, "one wavefront per lane of a group");
            const T xv = red_v[par][lane & (NW - 1)];
            const int xp = red_p[par][lane & (NW - 1)];
            T gv = max_dpp(xv, dpp_value<0xb1, 0xf>(xv));       // lane ^ 1
            gv = max_dpp(gv, dpp_value<0x4e, 0xf>(gv));         // lane ^ 2
            if constexpr (NW == 8) gv = max_dpp(gv, dpp_value<0x141, 0xf>(gv));  // the other half of the eight
            int gp = xv == gv ? xp : 0x7fffffff;
            gp = min(gp, dpp32<0xb1, 0xf>(0x7fffffff, gp));
            gp = min(gp, dpp32<0x4e, 0xf>(0x7fffffff, gp));
            if constexpr (NW == 8) gp = min(gp, dpp32<0x141, 0xf>(0x7fffffff, gp));
            const int piv = __builtin_amdgcn_readfirstlane(gp);
            const int from = __builtin_ctzll(__ballot(xp == piv)) & (NW - 1);
            T u[W];
#pragma unroll
            for (int q = 0; q < W; ++q) u[q] = cand[par][from][q];
            const T d = u[c];
            const bool zero = d == T(0);  // lu.rs:107-110: nothing is swapped or eliminated
            if (!zero) {
                const T inv = T(1) / d;
#pragma unroll
                for (int s = 0; s < RPT; ++s) {
                    const int y = pos[s] == k ? piv : pos[s];
                    pos[s] = pos[s] == piv ? k : y;
                    if (pos[s] > k) {  // rows past the matrix too: nothing reads them
                        const T l = a[s][c] * inv;
                        a[s][c] = l;
                        eliminate<W>(a[s], u, l, c + 1);
                    }
                }
            }
            // (after a lost wait a position may be held by no row; what is published stays a row's)
            if (t == 0) piv_word[c] = zero ? (k | PIV_SKIP) : piv < m ? piv : k;
            if (zero && first_zero == 0) first_zero = k + 1;
#pragma unroll
            for (int s = 0; s < RPT; ++s)
                if (live[s]) {
                    U b = ColWord<T>::bits(a[s][c]);
                    b = b == EMPTY ? b | ColWord<T>::QUIET : b;
                    __hip_atomic_store(Vp[s], b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    Vp[s] += ldv;
                }
        }
    }
    if (t < fc) {  // the first wavefront wrote them
        const int word = piv_word[t];
        __hip_atomic_store(H + (cg - c0) + t, (U)word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ipiv[cg + t] = word & ~PIV_SKIP;
    }
    if (first_zero != 0 && t == 0) {  // the first such column of the matrix (after the loop: a load in it would
        // make every column wait for its own stores)
        // a lost wait's -1 stays
        int seen = __hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while ((seen == 0 || seen > first_zero) &&
               !__hip_atomic_compare_exchange_strong(info, &seen, first_zero, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)) {
        }
    }
    // ---- what is final here: the group's rows; everything below them if no
    // later group swaps rows; columns that are not factored, all rows left
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const int p = pos[s];
        if (p >= c0 && p < m) {
#pragma unroll
            for (int q = 0; q < W; ++q) {
                const bool mine = fc > 0 ? p >= cg && (p < cg + fc || last || q >= fc) : p >= kend;
                if (q < wc && mine) A[p + (size_t)(cg + q) * lda] = a[s][q];
            }
        }
    }
}

// Rows below group h = blockIdx.y of a factored range (all groups but the
// last): position x of the final matrix holds what was at `who` when the group
// started, which the range's swaps from there on, followed backwards, give.
// nextV, nextH (or null): what the next panel, columns kend.., publishes into.
template <typename T, int W>
__global__ __launch_bounds__(256) void lu_left_kernel(T *A, int lda, int m, int c0, int kend,
                                                      const int *__restrict__ ipiv,
                                                      const typename ColWord<T>::U *__restrict__ V, int ldv,
                                                      typename ColWord<T>::U *__restrict__ nextV,
                                                      typename ColWord<T>::U *__restrict__ nextH)
{
    if (nextV) {  // 64 columns, rows kend..m
        const int row = kend + blockIdx.x * 256 + threadIdx.x;
        if (row < m)
            for (int c = blockIdx.y; c < 64; c += gridDim.y) nextV[(size_t)c * ldv + row] = ColWord<T>::EMPTY;
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 64) nextH[threadIdx.x] = ColWord<T>::EMPTY;
    }
    const int k0 = c0 + blockIdx.y * W;
    const int x = k0 + W + blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    if (x - lane >= m) return;  // the whole wavefront
    int who = x;
    // 64 pivots per round, one per lane, broadcast by readlane
    for (int b = kend - 1; b >= k0; b -= 64) {
        const int lo = max(k0, b - 63);
        const int pv = ipiv[min(lo + lane, b)];
        for (int i = b; i >= lo; --i) {
            const int p = __builtin_amdgcn_readlane(pv, i - lo);
            const int y = who == i ? p : who;
            who = who == p ? i : y;
        }
    }
    if (x < m) {
#pragma unroll
        for (int q = 0; q < W; ++q)
            A[x + (size_t)(k0 + q) * lda] = ColWord<T>::value(V[(size_t)(k0 - c0 + q) * ldv + who]);
    }
}

// The swaps [k0, k0 + cnt) (cnt <= 64) on the columns [ca0, ca1) and [cb0,
// cb1): a workgroup composes them itself (compose_block) and takes PCOLS
// columns, a quarter of its threads per column at a time; every value of a
// column is read before any is written.
constexpr int PLAN_COLS = 16;

template <typename T>
__global__ __launch_bounds__(512) void swap_rows_kernel(T *A, int lda, int m, const int *__restrict__ ipiv, int k0,
                                                        int cnt, int ca0, int ca1, int cb0, int cb1)
{
    __shared__ int pos[128], who[128];
    const int t = threadIdx.x;
    if (t < 64) {
        const nrocm_sweep::BlockPlan q = nrocm_sweep::compose_block(ipiv, k0, cnt, m, t, nullptr);
        // a position that keeps its content need not be touched
        pos[t] = q.in_who != k0 + t && k0 + t < m ? k0 + t : -1;
        who[t] = q.in_who;
        pos[64 + t] = q.out_pos != q.out_who ? q.out_pos : -1;
        who[64 + t] = q.out_who;
    }
    __syncthreads();
    const int slot = t & 127;
    const int p = pos[slot], from = who[slot];
    const int na = max(ca1 - ca0, 0), nb = max(cb1 - cb0, 0);
    T v[PLAN_COLS / 4];
#pragma unroll
    for (int u = 0; u < PLAN_COLS / 4; ++u) {
        const int ci = blockIdx.x * PLAN_COLS + (t >> 7) + 4 * u;
        const int c = ci < na ? ca0 + ci : cb0 + (ci - na);
        if (p >= 0 && ci < na + nb) v[u] = A[from + (size_t)c * lda];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PLAN_COLS / 4; ++u) {
        const int ci = blockIdx.x * PLAN_COLS + (t >> 7) + 4 * u;
        const int c = ci < na ? ca0 + ci : cb0 + (ci - na);
        if (p >= 0 && ci < na + nb) A[p + (size_t)c * lda] = v[u];
    }
}

template <typename U>
__global__ void fill_words_kernel(U *p, size_t count, U v, int *ints, int nints, int *info)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *info = 0;
    if (i < (size_t)nints) ints[i] = 0;
    for (size_t e = i; e < count; e += (size_t)gridDim.x * blockDim.x) p[e] = v;
}

}  // namespace nrocm_lu
