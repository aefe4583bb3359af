// Device kernels of the blocked LU factorisation and the triangular solves
// shared by LU (double) and the mixed-precision path (float working copy).
//
// Exactness argument (NROCM_EXACT).  nalgebra's LU::new (src/linalg/lu.rs:
// 93-122, 337-389) updates every trailing element (r, c) once per step k as
// A[r,c] = fl(A[r,c] - fl(u_kc * l_rk)), in increasing k, and swaps whole rows.
// A right-looking blocked schedule that (a) factors a panel column by column
// with those same operations, (b) applies the panel's row swaps to the other
// columns, (c) forms U12 by forward substitution in increasing k and (d)
// applies the rank-nb trailing update to each element in increasing k, with
// no fused multiply-add anywhere, performs for every element the identical
// sequence of IEEE operations.  Hence identical values and identical pivots.
#pragma once
#include "nrocm_internal.hpp"

namespace nrocm_lu {

// 32-bit DPP move with `old` kept where the source lane is outside the pattern.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ int dpp32(int old, int v)
{
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWMASK, 0xf, false);
}

template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_f64(double old, double v)
{
    const long long o = __double_as_longlong(old), x = __double_as_longlong(v);
    const int lo = dpp32<CTRL, ROWMASK>((int)o, (int)x);
    const int hi = dpp32<CTRL, ROWMASK>((int)(o >> 32), (int)(x >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int CTRL, int ROWMASK>
__device__ __forceinline__ float dpp_f32(float old, float v)
{
    return __int_as_float(dpp32<CTRL, ROWMASK>(__float_as_int(old), __float_as_int(v)));
}

// one instruction: fmax would first quiet NaNs, of which there are none here
__device__ __forceinline__ double max_dpp(double v, double o)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(v), "v"(o));
    return r;
}
__device__ __forceinline__ float max_dpp(float v, float o)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(v), "v"(o));
    return r;
}
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_value(double v) { return dpp_f64<CTRL, ROWMASK>(-1.0, v); }
template <int CTRL, int ROWMASK>
__device__ __forceinline__ float dpp_value(float v) { return dpp_f32<CTRL, ROWMASK>(-1.0f, v); }

// Wavefront maximum of non-NaN values >= -1; lane 63 ends with it.  Row scans by
// row_shr 1, 2, 4, 8, then row_bcast 15 into rows 1 and 3 and row_bcast 31 into
// rows 2 and 3.
template <typename V>
__device__ __forceinline__ V max_wave(V v)
{
    v = max_dpp(v, dpp_value<0x111, 0xf>(v));
    v = max_dpp(v, dpp_value<0x112, 0xf>(v));
    v = max_dpp(v, dpp_value<0x114, 0xf>(v));
    v = max_dpp(v, dpp_value<0x118, 0xf>(v));
    v = max_dpp(v, dpp_value<0x142, 0xa>(v));
    v = max_dpp(v, dpp_value<0x143, 0xc>(v));
    return v;
}

// Wavefront minimum of int positions; lane 63 ends with it.
__device__ __forceinline__ int min_wave(int p)
{
    constexpr int M = 0x7fffffff;
    p = min(p, dpp32<0x111, 0xf>(M, p));
    p = min(p, dpp32<0x112, 0xf>(M, p));
    p = min(p, dpp32<0x114, 0xf>(M, p));
    p = min(p, dpp32<0x118, 0xf>(M, p));
    p = min(p, dpp32<0x142, 0xa>(M, p));
    p = min(p, dpp32<0x143, 0xc>(M, p));
    return p;
}

// Returns v unchanged.  Copy loops whose values pass through this are not
// turned into memcpy calls, which would keep register arrays in scratch.
template <typename T>
__device__ __forceinline__ T pass(T v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// nalgebra's axpy with factor -x: fl(fl((-x) * y) + acc), the negation on x
// before the product as in gauss_step (lu.rs:353, :386).  In FP64 the operand
// order is pinned (-x first in the product, the product first in the sum), as
// the reference's x86 code has it, so that NaN results carry the same sign
// (with two NaN operands the first one is returned); NROCM_FAST fuses it.
template <typename T>
__device__ __forceinline__ T sub_prod(T acc, T x, T y, bool exact)
{
    if (exact) {
        if constexpr (sizeof(T) == 8) {
            double r;
            asm("v_mul_f64 %0, -%1, %2\n\tv_add_f64 %0, %0, %3" : "=&v"(r) : "v"(x), "v"(y), "v"(acc));
            return r;
        } else {
            const T p = (-x) * y;
            return p + acc;
        }
    }
    return fma(-x, y, acc);
}

// U12 = L11^{-1} A12 for a unit-lower L11 (k x k, k <= 64) at A[r0, r0] and the
// columns [c0, c1): one wavefront per column, lane r holds row r0 + r.
// Per element: A[r,c] = fl(A[r,c] - fl(u_ic * l_ri)) for i = 0..r-1 in order.
template <typename T>
__global__ __launch_bounds__(256) void trsm_unit_lower_kernel(T *A, int lda, int r0, int k, int c0,
                                                              int c1, int exact)
{
    __shared__ T L[64][65];
    {
        // thread t stages row t & 63, columns (t >> 6) + 4 i: 16 loads in
        // flight, clamped in-bounds addresses (entries past k are never read)
        const int rr = threadIdx.x & 63, cq = threadIdx.x >> 6;
        const T *lrow = A + (r0 + (rr < k ? rr : 0));
        T v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = lrow[(size_t)(r0 + (cq + 4 * i < k ? cq + 4 * i : 0)) * lda];
#pragma unroll
        for (int i = 0; i < 16; ++i) L[rr][cq + 4 * i] = v[i];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    for (int c = c0 + blockIdx.x * 4 + wv; c < c1; c += gridDim.x * 4) {
        T *col = A + (size_t)c * lda + r0;
        T v = lane < k ? col[lane] : T(0);
        for (int i = 0; i < k - 1; ++i) {
            const T u = __shfl(v, i);
            if (lane > i && lane < k) v = sub_prod(v, u, L[lane][i], exact != 0);
        }
        if (lane < k) col[lane] = v;
    }
}

// C (m x nc, ldc) -= L (m x K, ldl) * U (K x nc, K <= 64; element (q, c) at
// U[q*rsu + c*csu]).  SIMT register tiles: 256 threads per 64 x 64 tile, 4 x 4
// neighbouring elements per thread, each element's K terms applied in
// increasing k (EXACT: fl(C - fl(u*l)), otherwise fma).  LOWER: only elements
// with r >= c are written (the strict upper triangle stays untouched).
// What bounds it is the FP64 VALU (two instructions per term in EXACT) once the
// operands are there: all of a thread's loads, C among them, are issued
// together, the operands are staged in one pass, and the K steps then run
// without a barrier, a step's operands being four 16-byte LDS reads (before:
// four staged slices of 16 with two barriers each, scalar LDS reads: 1436^2
// lower triangle 23.9 -> 14.1 us).
template <typename T, bool EXACT, bool LOWER>
__global__ __launch_bounds__(256) void update_kernel(T *C, int ldc, int m, int nc, const T *Lp, int ldl,
                                                     const T *Up, long rsu, long csu, int K)
{
    constexpr int TM = 64, KM = 64, PAD = 4;
    typedef T V4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(32) T Ls[KM][TM + PAD];
    __shared__ __align__(32) T Us[KM][TM + PAD];
    const int tr = blockIdx.x * TM;
    const int tc = blockIdx.y * TM;
    if (LOWER && tr + TM - 1 < tc) return;  // tile entirely above the diagonal
    const int t = threadIdx.x;
    const int tx = t % 16, ty = t / 16;
    T acc[4][4];  // [column][row]
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            acc[b][a] = C[min(tr + 4 * tx + a, m - 1) + (size_t)min(tc + 4 * ty + b, nc - 1) * ldc];
    T lv[16], uv[16];
    {
        // clamped addresses; what they bring past the edges is never stored
        const int r = min(tr + (t & 63), m - 1), q0 = t >> 6;
        const int c = rsu == 1 ? t >> 6 : t & 63, k0 = rsu == 1 ? t & 63 : t >> 6;
#pragma unroll
        for (int s = 0; s < 16; ++s) lv[s] = Lp[r + (size_t)min(q0 + 4 * s, K - 1) * ldl];
        if (rsu == 1) {  // columns of U contiguous: threads along k
#pragma unroll
            for (int s = 0; s < 16; ++s) uv[s] = Up[min(k0, K - 1) + (long)min(tc + c + 4 * s, nc - 1) * csu];
        } else {         // rows contiguous: threads along the columns
#pragma unroll
            for (int s = 0; s < 16; ++s) uv[s] = Up[(long)min(k0 + 4 * s, K - 1) * rsu + (long)min(tc + c, nc - 1) * csu];
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) Ls[q0 + 4 * s][t & 63] = lv[s];
        if (rsu == 1) {
#pragma unroll
            for (int s = 0; s < 16; ++s) Us[k0][c + 4 * s] = uv[s];
        } else {
#pragma unroll
            for (int s = 0; s < 16; ++s) Us[k0 + 4 * s][c] = uv[s];
        }
    }
    __syncthreads();
#pragma unroll 2
    for (int q = 0; q < K; ++q) {
        const V4 l = *(const V4 *)&Ls[q][4 * tx];
        const V4 u = *(const V4 *)&Us[q][4 * ty];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if constexpr (EXACT && sizeof(T) == 8) {
                double p[4];
#pragma unroll
                for (int a = 0; a < 4; ++a) asm("v_mul_f64 %0, -%1, %2" : "=v"(p[a]) : "v"(u[b]), "v"(l[a]));
#pragma unroll
                for (int a = 0; a < 4; ++a) asm("v_add_f64 %0, %1, %0" : "+v"(acc[b][a]) : "v"(p[a]));
            } else {
#pragma unroll
                for (int a = 0; a < 4; ++a) acc[b][a] = sub_prod(acc[b][a], u[b], l[a], EXACT);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int r = tr + 4 * tx + a, c = tc + 4 * ty + b;
            if (r < m && c < nc && (!LOWER || r >= c)) C[r + (size_t)c * ldc] = acc[b][a];
        }
}

// Row plan of a window's permutation: plan[0] = number nt of touched
// positions; afterwards position plan[1 + s] holds the value that was at
// position plan[1 + PLAN_MAX + s].
constexpr int PLAN_MAX = 128;

// Applies a row plan to the columns [ca0, ca1) and [cb0, cb1): two columns
// per workgroup, one thread per touched position; every value is read before
// any is written.
template <typename T>
__global__ __launch_bounds__(256) void apply_plan_kernel(T *A, int lda, const int *plan, int ca0, int ca1, int cb0,
                                                         int cb1)
{
    const int t = threadIdx.x;
    const int slot = t & (PLAN_MAX - 1);
    const int na = ca1 > ca0 ? ca1 - ca0 : 0;
    const int nbc = cb1 > cb0 ? cb1 - cb0 : 0;
    const int ci = blockIdx.x * 2 + (t >> 7);
    const bool valid = ci < na + nbc;
    const int c = ci < na ? ca0 + ci : cb0 + (ci - na);
    const int nt = plan[0];
    T v = T(0);
    if (valid && slot < nt) v = A[plan[1 + PLAN_MAX + slot] + (size_t)c * lda];
    __syncthreads();
    if (valid && slot < nt) A[plan[1 + slot] + (size_t)c * lda] = v;
}

// A[r0.., k0..k0+nb) <- A[r0.., k0..k0+nb) U11^{-1} (U11 the upper triangle of
// the factored diagonal block): one thread per row, the row in registers,
// x_q = (a_q - sum_{p<q} x_p U_pq) / U_qq with four partial sums.  U is staged
// transposed in LDS so that a column is contiguous; each column is read in two
// halves of 32 whose reads are all issued before the first use (one LDS round
// trip per half instead of one per pair of values).
constexpr int TRSM_RU_THREADS = 64;

template <typename T>
__global__ __launch_bounds__(TRSM_RU_THREADS) void trsm_right_upper_kernel(T *A, int lda, int k0, int nb, int r0,
                                                                           int m)
{
    __shared__ __align__(16) T Ut[64][64];  // Ut[q][p] = U[p][q]
    __builtin_amdgcn_s_setprio(3);  // on the look-ahead critical path, beside the trailing update
    const int t = threadIdx.x;
    // the row to solve is loaded first, so that its loads overlap the staging
    const int r = r0 + blockIdx.x * TRSM_RU_THREADS + t;
    const bool live = r < m;
    T *row = A + (live ? r : r0);
    T x[64];
#pragma unroll
    for (int q = 0; q < 64; ++q) x[q] = row[(size_t)(k0 + (q < nb ? q : 0)) * lda];
    // thread t stages row t of U; 16 loads in flight (clamped in-bounds
    // addresses, zeros selected afterwards) instead of one load per wait
    const T *urow = A + (k0 + (t < nb ? t : 0));
#pragma unroll
    for (int q0 = 0; q0 < 64; q0 += 16) {
        T v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = urow[(size_t)(k0 + (q0 + j < nb ? q0 + j : 0)) * lda];
#pragma unroll
        for (int j = 0; j < 16; ++j) Ut[q0 + j][t] = (t <= q0 + j && q0 + j < nb) ? v[j] : T(0);
    }
    __syncthreads();
    // x[q] past nb holds column 0 again and is never read: the solve below
    // touches x[p] only for p < q < nb, and rows past m are not stored
#pragma unroll
    for (int q = 0; q < 64; ++q) {
        if (q < nb) {  // uniform
            T s[4] = {x[q], T(0), T(0), T(0)};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (32 * h < q) {
                    T u[32];
#pragma unroll
                    for (int j = 0; j < 32; ++j)
                        if (32 * h + j < q) u[j] = Ut[q][32 * h + j];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < 32; ++j)
                        if (32 * h + j < q) s[j & 3] = fma(-x[32 * h + j], u[j], s[j & 3]);
                }
            }
            x[q] = ((s[0] + s[1]) + (s[2] + s[3])) / Ut[q][q];
        }
    }
    int nbs = nb;
    asm volatile("" : "+s"(nbs));  // recompute the column masks instead of keeping 64 alive
    if (live) {
#pragma unroll
        for (int q = 0; q < 64; ++q)
            if (q < nbs) row[(size_t)(k0 + q) * lda] = x[q];
    }
}

// ---------------------------------------------------------------- LU with windowed pivoting
// (mixed-precision solver only; pivots differ from nalgebra's by design)
//
// Partial pivoting restricted to a window: for the nb (<= 64) columns at k0,
// every pivot is the largest |a| among the rows [k0, kw) not yet chosen,
// kw - k0 <= WINDOW_ROWS.  Rows below the window are eliminated afterwards by
// A21 U11^{-1}.  With a 128-row window at least 65 candidates remain for the
// last column of a block, which keeps |L| and the growth close to full
// partial pivoting on the dense test matrices while the pivot search never
// leaves one workgroup.
constexpr int WINDOW_ROWS = 128;

// Pivot key of window position pos (< 128) for a magnitude av: its top bits
// with the low 7 replaced by 127 - pos.  The unsigned maximum of the keys is
// the largest magnitude to within 2^-16 relative (2^-13 for FP64) and, among
// magnitudes that close, the lowest position: a pivot within that factor of
// the largest is as good for this solver, and the search becomes one integer
// maximum per DPP step.
template <typename T>
__device__ __forceinline__ unsigned pivot_key(T av, int pos)
{
    const unsigned hi =
        sizeof(T) == 8 ? (unsigned)((unsigned long long)__double_as_longlong((double)av) >> 32) : __float_as_uint((float)av);
    return (hi & ~127u) | (unsigned)(127 - pos);
}

// Wavefront maximum of an unsigned value; lane 63 ends with it (same DPP
// pattern as max_wave).
__device__ __forceinline__ unsigned wave_max_u32(unsigned k)
{
    k = max(k, (unsigned)dpp32<0x111, 0xf>(0, (int)k));
    k = max(k, (unsigned)dpp32<0x112, 0xf>(0, (int)k));
    k = max(k, (unsigned)dpp32<0x114, 0xf>(0, (int)k));
    k = max(k, (unsigned)dpp32<0x118, 0xf>(0, (int)k));
    k = max(k, (unsigned)dpp32<0x142, 0xa>(0, (int)k));
    k = max(k, (unsigned)dpp32<0x143, 0xc>(0, (int)k));
    return k;
}

// Each wavefront holds 8 columns of all the window's rows (two rows a lane) and
// the pivot search of a column is a reduction inside the wavefront that owns
// it; the multipliers and the pivot pass to the wavefronts of the columns on its
// right through LDS, each column's word its own flag, so no barrier is met and
// a wavefront's own columns follow one another at the pace of search, division
// and the update of its remaining columns.  Rows are not moved during the
// factorisation: each lane carries the logical positions of its rows, and every
// row is written to its final position at the end.  f32, 64 columns, beside the
// trailing update of an 8192 x 8192 system: 68 -> 43 us (one row a lane, the
// pivot row through LDS and two barriers a column before).
//
// Records ipiv (absolute, LAPACK order: step k0+c exchanged rows k0+c and
// ipiv[k0+c]) and the composed row plan of the window for apply_plan_kernel;
// with perm non-null it also applies the window's permutation to perm[k0, kw)
// (row i of the factors is row perm[i] of the input).  A zero pivot column sets
// info (first one) and is skipped.
constexpr int PANEL_COLS = 8;  // columns of a wavefront

__device__ __forceinline__ double lane_of(double v, int src)
{
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)x, src), hi = __builtin_amdgcn_readlane((int)(x >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ float lane_of(float v, int src)
{
    return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(v), src));
}

template <typename T>
__global__ __launch_bounds__(512) void window_panel_kernel(T *A, int lda, int k0, int nb, int kw, int *ipiv, int *info,
                                                           int *plan, int *perm)
{
    static_assert(WINDOW_ROWS == 128, "two rows a lane");
    constexpr int W = PANEL_COLS;
    constexpr unsigned EMPTY = ~0u, SKIP = 1u << 16;
    __shared__ T mult[64 - W][WINDOW_ROWS];  // the multipliers of a column, by row
    __shared__ unsigned pub[64];             // position and row of its pivot, SKIP
    __shared__ int final_pos[WINDOW_ROWS];
    __shared__ unsigned long long wmask[2];
    __shared__ int bad;  // first column without a pivot
    // this kernel is the critical path of the look-ahead pipeline and shares
    // its CU with trailing-update wavefronts: issue first among them
    __builtin_amdgcn_s_setprio(3);
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wr = kw - k0;
    const int r0 = lane, r1 = lane + 64;
    T a0[W], a1[W];
    {
        const T *p0 = A + (k0 + min(r0, wr - 1)), *p1 = A + (k0 + min(r1, wr - 1));
#pragma unroll
        for (int q = 0; q < W; ++q) {
            const size_t col = (size_t)(k0 + min(W * w + q, nb - 1)) * lda;
            a0[q] = p0[col];
            a1[q] = p1[col];
        }
    }
    if (t < 64) pub[t] = EMPTY;
    if (t == 0) bad = 64;
    __syncthreads();
    int pos0 = r0, pos1 = r1;
    // the pivot of column c moves from position P to c
    auto exchange = [&](int c, int P) {
        pos0 = pos0 == P ? c : pos0 == c ? P : pos0;
        pos1 = pos1 == P ? c : pos1 == c ? P : pos1;
    };
    // the columns on the left, as they come
    const int mine = min(W * w, nb);
    for (int c = 0; c < mine; ++c) {
        unsigned word;
        T l0, l1;
        for (;;) {
            // read in this order: the word is written after the multipliers
            word = __hip_atomic_load(&pub[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            asm volatile("" ::: "memory");
            l0 = mult[c][r0];
            l1 = mult[c][r1];
            asm volatile("" ::: "memory");
            word = (unsigned)__builtin_amdgcn_readfirstlane((int)word);
            if (word != EMPTY) break;
            __builtin_amdgcn_s_sleep(1);
        }
        exchange(c, (int)(word & 127u));
        if (word & SKIP) continue;
        const int src = (int)(word >> 8) & 63;
        const bool upper = (word >> 14) & 1;
        T u[W];
#pragma unroll
        for (int q = 0; q < W; ++q) u[q] = lane_of(upper ? a1[q] : a0[q], src);
        if (pos0 > c) {
#pragma unroll
            for (int q = 0; q < W; ++q) a0[q] = fma(-l0, u[q], a0[q]);
        }
        if (pos1 > c) {
#pragma unroll
            for (int q = 0; q < W; ++q) a1[q] = fma(-l1, u[q], a1[q]);
        }
    }
    // its own
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const int c = W * w + j;
        if (c < nb) {  // uniform
            const unsigned key0 = (r0 < wr && pos0 >= c) ? pivot_key(fabs(a0[j]), pos0) : 0u;
            const unsigned key1 = (r1 < wr && pos1 >= c) ? pivot_key(fabs(a1[j]), pos1) : 0u;
            const unsigned kmax = (unsigned)__builtin_amdgcn_readlane((int)wave_max_u32(max(key0, key1)), 63);
            const unsigned mag = kmax & ~127u;
            // an all-zero (or non-finite) column: nothing to exchange or eliminate
            const bool zero = mag == 0u || mag >= (sizeof(T) == 8 ? 0x7ff00000u : 0x7f800000u);
            const int P = zero ? c : 127 - (int)(kmax & 127u);
            const unsigned long long in0 = __ballot(pos0 == P), in1 = __ballot(pos1 == P);
            const bool upper = in0 == 0ull;
            const int src = __builtin_ctzll(upper ? in1 : in0);
            exchange(c, P);
            if (!zero) {
                const T piv = lane_of(upper ? a1[j] : a0[j], src);
                const T inv = T(1) / piv;
                T u[W];
#pragma unroll
                for (int q = j + 1; q < W; ++q) u[q] = lane_of(upper ? a1[q] : a0[q], src);
                const T l0 = a0[j] * inv, l1 = a1[j] * inv;
                if (w < 64 / W - 1) {
                    mult[c][r0] = l0;
                    mult[c][r1] = l1;
                }
                asm volatile("" ::: "memory");
                if (lane == 0)
                    __hip_atomic_store(&pub[c], (unsigned)P | (unsigned)src << 8 | (upper ? 1u << 14 : 0u),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (pos0 > c) {
                    a0[j] = l0;
#pragma unroll
                    for (int q = j + 1; q < W; ++q) a0[q] = fma(-l0, u[q], a0[q]);
                }
                if (pos1 > c) {
                    a1[j] = l1;
#pragma unroll
                    for (int q = j + 1; q < W; ++q) a1[q] = fma(-l1, u[q], a1[q]);
                }
            } else if (lane == 0) {
                __hip_atomic_store(&pub[c], (unsigned)P | SKIP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                atomicMin(&bad, c);
            }
            if (lane == 0) ipiv[k0 + c] = k0 + P;
        }
    }
    if (w == (nb - 1) / W) {  // the owner of the last column has followed every exchange
        final_pos[r0] = pos0;
        final_pos[r1] = pos1;
    }
    __syncthreads();
    pos0 = final_pos[r0];
    pos1 = final_pos[r1];
    {
        T *d0 = A + (k0 + pos0), *d1 = A + (k0 + pos1);
#pragma unroll
        for (int q = 0; q < W; ++q) {
            const size_t col = (size_t)(k0 + W * w + q) * lda;
            if (W * w + q < nb) {
                if (r0 < wr) d0[col] = a0[q];
                if (r1 < wr) d1[col] = a1[q];
            }
        }
    }
    // row plan: the window row now at position pos came from position t
    const int row = w == 0 ? r0 : r1, pos = w == 0 ? pos0 : pos1;
    const bool moved = w < 2 && row < wr && pos != row;
    const unsigned long long m = __ballot(moved);
    if (w < 2 && lane == 0) wmask[w] = m;
    const int myperm = (perm && w < 2 && row < wr) ? perm[k0 + row] : 0;
    __syncthreads();  // also: perm is read by everyone before it is written
    if (perm && w < 2 && row < wr) perm[k0 + pos] = myperm;
    const int before = __popcll(m & ((1ull << lane) - 1)) + (w ? __popcll(wmask[0]) : 0);
    if (moved) {
        plan[1 + before] = k0 + pos;
        plan[1 + PLAN_MAX + before] = k0 + row;
    }
    if (t == 0) {
        plan[0] = __popcll(wmask[0]) + __popcll(wmask[1]);
        if (bad < 64 && *info == 0) *info = k0 + bad + 1;
    }
}

__global__ void iota_kernel(int *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

__global__ void fill_int_kernel(int *p, int n, int v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace nrocm_lu
