// LU with partial pivoting (nrocm_dgetrf), the windowed variant of the mixed
// solver, and the single-matrix Cholesky entry points (nrocm_dpotrf).
//
// Up to WHOLE_ROWS rows the whole matrix is one pipeline of column groups
// (lu_columns.hpp).  Above:
//   for each 64-wide panel [j0, j0+nb):
//     lu_columns_kernel   the panel, as a pipeline of column groups
//     swap_rows_kernel    its swaps on all other columns
//     trsm                U12 = L11^{-1} A12 for the trailing columns
//     trailing update     A22 -= L21 * U12: EXACT = ordered unfused SIMT,
//                         FAST = FP64 MFMA, float working copies: FP32 or BF16 MFMA
//   where the next panel's 64 columns are updated first and the next panel then
//   runs beside the update of the rest.
#include "gemm_kernels.hpp"
#include "internal_launch.hpp"
#include "lu_columns.hpp"

#include <algorithm>

using namespace nrocm_lu;

namespace {

// Whole matrices of up to this many rows are one pipeline; above it every group
// takes too long to catch up with all the earlier ones (EXACT, one pipeline
// against 64-column panels: n = 700 1.19 and 1.42 ms, 1000 1.94 and 2.15, 1100
// 2.97 and 2.51, 2048 8.2 and 5.3).  FAST and wide matrices take the same rule,
// measured against the panels that came before these pipelines: 1000 x 1000 FAST 1.91
// and 4.45 ms, 1000 x 4096 3.67 and 4.73, 1000 x 16384 5.78 and 5.74.
constexpr int WHOLE_ROWS = 1024;

// The pipeline's buffer, after a header of one ticket per panel: L columns and
// pivots of all columns where the matrix is one range, else of two panels in turn
// (lu_left_kernel, which has read the one, clears the other for the next panel).
constexpr size_t LU_HEADER_BYTES = 2048;
constexpr int LU_NB = 64;  // columns of a panel

bool lu_is_whole(int m, int n) { return m <= WHOLE_ROWS || std::min(m, n) <= LU_NB; }

template <typename T>
struct LuBuffer {
    typedef typename ColWord<T>::U U;
    int *tickets;
    U *words;
    int ldv, cols, parts;

    LuBuffer(void *p, int m, int n)
        : tickets((int *)p), words((U *)((char *)p + LU_HEADER_BYTES)), ldv(m),
          cols(lu_is_whole(m, n) ? std::min(m, n) : LU_NB), parts(lu_is_whole(m, n) ? 1 : 2)
    {
    }
    size_t part_words() const { return (size_t)cols * ldv + cols; }
    size_t bytes() const { return LU_HEADER_BYTES + parts * part_words() * sizeof(U); }
    U *V(int c0) const { return words + (size_t)(c0 / LU_NB % parts) * part_words(); }
    U *H(int c0) const { return V(c0) + (size_t)cols * ldv; }
    hipError_t clear(hipStream_t st, int *info)  // the first part, and info
    {
        const size_t count = part_words();
        hipLaunchKernelGGL((fill_words_kernel<U>), dim3(std::min<size_t>(4096, nrocm_cdiv(count, 1024) + 4)), dim3(256),
                           0, st, words, count, ColWord<T>::EMPTY, tickets, (int)(LU_HEADER_BYTES / sizeof(int)), info);
        return hipGetLastError();
    }
};

template <typename T, typename G>
hipError_t lu_columns_group(hipStream_t st, T *A, int lda, int m, int c0, int ncols, int kend, int *ipiv, int *info,
                            LuBuffer<T> &b, int ticket, long limit)
{
    hipLaunchKernelGGL((lu_columns_kernel<T, G>), dim3(nrocm_cdiv(ncols, G::W)), dim3(G::CT), 0, st, A, lda, m, c0,
                       ncols, kend, ipiv, info, b.V(c0), b.ldv, b.H(c0), b.tickets + ticket, limit);
    return hipGetLastError();
}

template <typename T, typename G>
hipError_t lu_left_group(hipStream_t st, T *A, int lda, int m, int c0, int kend, const int *ipiv, LuBuffer<T> &b,
                         bool next)
{
    const int groups = (int)nrocm_cdiv(kend - c0, G::W);
    if (groups > 1 && m > c0 + G::W)
        hipLaunchKernelGGL((lu_left_kernel<T, G::W>), dim3(nrocm_cdiv(m - c0 - G::W, 256), groups - 1), dim3(256), 0,
                           st, A, lda, m, c0, kend, ipiv, b.V(c0), b.ldv, next ? b.V(kend) : nullptr,
                           next ? b.H(kend) : nullptr);
    return hipGetLastError();
}

#define LU_BY_ROWS(FN, rows, ...)                                                                        \
    ((rows) <= Group256::ROWS   ? FN<T, Group256>(__VA_ARGS__)                                           \
     : (rows) <= Group512::ROWS ? FN<T, Group512>(__VA_ARGS__)                                           \
     : (rows) <= Group1K::ROWS  ? FN<T, Group1K>(__VA_ARGS__)                                            \
     : (rows) <= Group2K::ROWS  ? FN<T, Group2K>(__VA_ARGS__)                                            \
     : (rows) <= Group4K::ROWS  ? FN<T, Group4K>(__VA_ARGS__)                                            \
     : (rows) <= Group8K::ROWS  ? FN<T, Group8K>(__VA_ARGS__) : FN<T, Group16K>(__VA_ARGS__))

// Factors columns [c0, c0 + ncols) (those below kend) and brings them up to date.
template <typename T>
hipError_t lu_columns(hipStream_t st, T *A, int lda, int m, int c0, int ncols, int kend, int *ipiv, int *info,
                      LuBuffer<T> &b, int ticket, long limit)
{
    return LU_BY_ROWS(lu_columns_group, m - c0, st, A, lda, m, c0, ncols, kend, ipiv, info, b, ticket, limit);
}

// The L columns of all but the range's last group, their rows in final order; with
// `next`, a full panel with another one after it, also clears that one's part.
template <typename T>
hipError_t lu_left(hipStream_t st, T *A, int lda, int m, int c0, int kend, const int *ipiv, LuBuffer<T> &b, bool next)
{
    return LU_BY_ROWS(lu_left_group, m - c0, st, A, lda, m, c0, kend, ipiv, b, next);
}

template <typename T>
hipError_t swap_rows(hipStream_t st, T *A, int lda, int m, const int *ipiv, int k0, int cnt, int ca0, int ca1, int cb0,
                     int cb1)
{
    const int cols = std::max(ca1 - ca0, 0) + std::max(cb1 - cb0, 0);
    if (cols > 0)
        hipLaunchKernelGGL((swap_rows_kernel<T>), dim3(nrocm_cdiv(cols, PLAN_COLS)), dim3(512), 0, st, A, lda, m, ipiv,
                           k0, cnt, ca0, ca1, cb0, cb1);
    return hipGetLastError();
}

template <typename T>
hipError_t trsm(hipStream_t st, T *A, int lda, int r0, int k, int c0, int c1, bool exact)
{
    if (c1 <= c0 || k <= 1) return hipSuccess;
    const unsigned grid = std::min<unsigned>(nrocm_cdiv(c1 - c0, 4), 2048);
    hipLaunchKernelGGL((trsm_unit_lower_kernel<T>), dim3(grid), dim3(256), 0, st, A, lda, r0, k, c0, c1,
                       exact ? 1 : 0);
    return hipGetLastError();
}

template <typename T, bool EXACT, bool LOWER>
hipError_t simt_update(hipStream_t st, T *C, int ldc, int m, int nc, const T *Lp, int ldl, const T *Up, long rsu,
                       long csu, int K)
{
    if (m <= 0 || nc <= 0 || K <= 0) return hipSuccess;
    dim3 grid(nrocm_cdiv(m, 64), nrocm_cdiv(nc, 64));
    hipLaunchKernelGGL((update_kernel<T, EXACT, LOWER>), grid, dim3(256), 0, st, C, ldc, m, nc, Lp, ldl, Up, rsu,
                       csu, K);
    return hipGetLastError();
}

// A22 (rows r0.., cols c0..n) -= L21 (rows r0.., cols k0..k0+K) * U12 (rows k0.., cols c0..)
template <typename T>
hipError_t trailing(hipStream_t st, NrocmTrailing trail, T *A, int lda, int r0, int m, int c0, int n, int k0,
                    int K, int max_groups = 0)
{
    const int mm = m - r0, nn = n - c0;
    if (mm <= 0 || nn <= 0 || K <= 0) return hipSuccess;
    T *C = A + r0 + (size_t)c0 * lda;
    const T *Lp = A + r0 + (size_t)k0 * lda;
    const T *Up = A + k0 + (size_t)c0 * lda;
    if (trail == TRAIL_EXACT) return simt_update<T, true, false>(st, C, lda, mm, nn, Lp, lda, Up, 1, lda, K);
    if constexpr (sizeof(T) == 8) {
        return nrocm_rank_update_d(st, mm, nn, K, (const double *)Lp, lda, (const double *)Up, lda, (double *)C, lda,
                                   max_groups);
    } else {
        const int mode = trail == TRAIL_BF16X3 ? 3 : trail == TRAIL_BF16 ? 2 : 1;
        return nrocm_rank_update_s(st, mm, nn, K, (const float *)Lp, lda, (const float *)Up, lda, (float *)C, lda,
                                   mode, max_groups);
    }
}

#define LU_TRY(x)                                      \
    do {                                               \
        hipError_t e__ = (x);                          \
        if (e__ != hipSuccess) return nrocm_fail_hip(h, e__, #x); \
    } while (0)

template <typename T>
int getrf_whole(nrocm_handle h, hipStream_t st, int m, int n, T *A, int lda, int *ipiv, int *info, void *buf)
{
    LuBuffer<T> b(buf, m, n);
    const int mn = std::min(m, n);
    LU_TRY(b.clear(st, info));
    LU_TRY(lu_columns<T>(st, A, lda, m, 0, n, mn, ipiv, info, b, 0, nrocm_wait_limit(h, COL_SPIN_LIMIT)));
    LU_TRY(lu_left<T>(st, A, lda, m, 0, mn, ipiv, b, false));
    return NROCM_OK;
}

template <typename T>
int getrf_panels(nrocm_handle h, hipStream_t st, int m, int n, T *A, int lda, int *ipiv, int *info,
                 NrocmTrailing trail, void *buf)
{
    LuBuffer<T> b(buf, m, n);
    const int mn = std::min(m, n);
    const bool exact = trail == TRAIL_EXACT;
    constexpr int NB = LU_NB;
    const long limit = nrocm_wait_limit(h, COL_SPIN_LIMIT);
    LU_TRY(b.clear(st, info));
    LU_TRY(lu_columns<T>(st, A, lda, m, 0, std::min(NB, mn), std::min(NB, mn), ipiv, info, b, 0, limit));
    for (int j0 = 0; j0 < mn; j0 += NB) {
        const int nb = std::min(NB, mn - j0), j1 = j0 + nb;
        LU_TRY(lu_left<T>(st, A, lda, m, j0, j1, ipiv, b, j1 < mn));
        LU_TRY(swap_rows<T>(st, A, lda, m, ipiv, j0, nb, 0, j0, j1, n));
        if (j1 < n) LU_TRY(trsm<T>(st, A, lda, j0, nb, j1, n, exact));
        const int j2 = j1 < mn ? std::min(mn, j1 + NB) : j1;  // the next panel
        if (j2 > j1) {
            LU_TRY(trailing<T>(st, trail, A, lda, j1, m, j1, j2, j0, nb));
            const int s = nrocm_fork_on(h, st, 1);
            if (s != NROCM_OK) return s;
            LU_TRY(lu_columns<T>(h->aux[0], A, lda, m, j1, j2 - j1, j2, ipiv, info, b, j1 / NB, limit));
        }
        LU_TRY(trailing<T>(st, trail, A, lda, j1, m, j2, n, j0, nb));
        if (j2 > j1) {
            const int s = nrocm_join_on(h, st, 1);
            if (s != NROCM_OK) return s;
        }
    }
    return NROCM_OK;
}

// ---------------------------------------------------------------- blocked Cholesky for n > 64
// One 64-column panel of Cholesky::new (cholesky.rs:226-262) in one launch: the
// diagonal block, then the rows below it, 256 per workgroup.  Every workgroup
// factors the diagonal block for itself (in parallel that costs nothing, and
// saves a launch and a trip through memory between the two), the first one
// keeps it.
//
// Diagonal block: lane = row, wavefront w the columns 4 i + w; step k takes the
// square root and the quotients of column k (three instructions each with the
// root's reciprocal, exact_div.hpp) in the wavefront that holds it, and one
// barrier hands the column to all.  Rows: one per thread, in registers, right-
// looking: element j receives fl(x_j - fl(L_jk * x_k)) in increasing k as soon as
// x_k is known, so the 63 elements of a step interleave (left-looking, each
// element's terms were one dependent chain with an LDS read per term).
// n = 1500: diagonal block and rows together 135 -> 56 us per panel.
constexpr int CP_THREADS = 256;
constexpr int CP_LD = 66;  // column stride of the block in LDS

__device__ __forceinline__ double chol_quotient(double v, double den, double rec, bool dok)
{
    const bool ok = dok && nrocm_div::num_in_range(v);
    double q = nrocm_div::div_with(v, den, rec);
    if (__builtin_expect(__ballot(!ok) != 0, 0)) q = ok ? q : v / den;  // out of the unrolled steps' way
    return q;
}

// acc = fl(fl((-x) * y) + acc) in place, or one fused multiply-add.
template <bool EXACT>
__device__ __forceinline__ void chol_update(double &acc, double x, double y)
{
    if constexpr (EXACT) {
        double p;
        asm("v_mul_f64 %0, -%1, %2" : "=v"(p) : "v"(x), "v"(y));
        asm("v_add_f64 %0, %1, %0" : "+v"(acc) : "v"(p));
    } else {
        asm("v_fma_f64 %0, -%1, %2, %0" : "+v"(acc) : "v"(x), "v"(y));
    }
}

// out11: where the factored block goes (column stride ldo): the matrix itself if
// this is the only workgroup, else a buffer, because workgroups that start
// later still read the block.
template <bool EXACT>
__global__ __launch_bounds__(CP_THREADS) void chol_panel_kernel(double *A, int lda, int n, int j0, int nb,
                                                                double substitute, double *out11, int ldo, int *info)
{
    __shared__ __align__(16) double Ld[64 * CP_LD];  // L_jk at [k * CP_LD + j]
    __shared__ double dg[64], rec[64];
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const double *D = A + j0 + (size_t)j0 * lda;
    double a[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = 4 * i + w;
        const bool in = lane >= c && lane < nb;
        const double v = D[min(lane, nb - 1) + (size_t)min(c, nb - 1) * lda];
        a[i] = in ? v : (lane == c ? 1.0 : 0.0);  // padding holds the identity
    }
    // this thread's row below the block: its loads arrive during the factorisation
    const int r = j0 + nb + blockIdx.x * CP_THREADS + t;
    const bool row = r < n;
    double *xrow = A + (row ? r : n - 1) + (size_t)j0 * lda;
    double x[64];
#pragma unroll
    for (int j = 0; j < 64; ++j) x[j] = xrow[(size_t)min(j, nb - 1) * lda];

    // column k, by the wavefront that holds it
    auto finish = [&](int k, double v) {
        const double d = nrocm_sweep::lane_value(v, k);
        const double den = sqrt((substitute > 0.0 && !(d > 0.0)) ? substitute : d);
        const double y = nrocm_div::recip_refined(den);
        const double l = chol_quotient(lane > k ? v : 1.0, den, y, nrocm_div::div_den_ok(den));
        Ld[k * CP_LD + lane] = lane > k ? l : (lane == k ? den : 0.0);
        if (lane == 0) {
            dg[k] = den;
            rec[k] = y;
        }
    };
    if (w == 0) finish(0, a[0]);
    lds_barrier();
#pragma unroll
    for (int k = 0; k < 63; ++k) {
        // The next column first: its wavefront finishes it while the others
        // update theirs, and makes up for its own updates after the barrier,
        // when another wavefront holds the chain.
        const int next = (k + 1) >> 2;
        const double lr = Ld[k * CP_LD + lane];
        double lj[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (i >= next) lj[i] = Ld[k * CP_LD + 4 * i + w];
        // (columns up to k in the block of four that k is in get values nobody reads)
        chol_update<EXACT>(a[next], lj[next], lr);
        const bool holds = w == ((k + 1) & 3);
        auto rest = [&]() {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (i > next) chol_update<EXACT>(a[i], lj[i], lr);
        };
        if (holds) finish(k + 1, a[next]);
        else rest();
        lds_barrier();
        if (holds) rest();
    }
    if (blockIdx.x == 0) {
        const double dl = lane < nb ? dg[lane] : 1.0;
        const unsigned long long bad = __ballot(!(dl > 0.0));
        if (t == 0 && bad != 0 && *info == 0) *info = j0 + (int)__builtin_ctzll(bad) + 1;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int c = 4 * i + w;
            if (c < nb && lane >= c && lane < nb) out11[lane + (size_t)c * ldo] = Ld[c * CP_LD + lane];
        }
    }
    if (j0 + nb + (int)blockIdx.x * CP_THREADS >= n) return;  // no rows: the whole workgroup
#pragma unroll
    for (int k = 0; k < 64; ++k) {
        if (k < nb) {
            const double den = dg[k];
            const double q = chol_quotient(x[k], den, rec[k], nrocm_div::div_den_ok(den));
            x[k] = q;
            if (row) xrow[(size_t)k * lda] = q;
#pragma unroll
            for (int j = k + 1; j < 64; ++j) chol_update<EXACT>(x[j], Ld[k * CP_LD + j], q);
        }
    }
}

// The block that chol_panel_kernel left in its buffer.
__global__ __launch_bounds__(256) void chol_store_block_kernel(double *D, int lda, const double *__restrict__ L11)
{
    const int lane = threadIdx.x & 63;
    for (int c = threadIdx.x >> 6; c < 64; c += 4)
        if (lane >= c) D[lane + (size_t)c * lda] = L11[lane + c * 64];
}

int potrf_blocked(nrocm_handle h, int n, double *A, int lda, int *info, bool exact, double substitute)
{
    hipStream_t st = h->stream;
    void *ws = nullptr;
    const int s = nrocm_workspace(h, 64 * 64 * sizeof(double), &ws);
    if (s != NROCM_OK) return s;
    double *L11 = (double *)ws;
    hipLaunchKernelGGL(fill_int_kernel, dim3(1), dim3(64), 0, st, info, 1, 0);
    LU_TRY(hipGetLastError());
    for (int j0 = 0; j0 < n; j0 += 64) {
        const int nb = std::min(64, n - j0);
        const int r0 = j0 + nb;
        double *D = A + j0 + (size_t)j0 * lda;
        const unsigned grid = std::max(1u, nrocm_cdiv(n - r0, CP_THREADS));
        double *out11 = grid == 1 ? D : L11;
        const int ldo = grid == 1 ? lda : 64;
        if (exact)
            hipLaunchKernelGGL(chol_panel_kernel<true>, dim3(grid), dim3(CP_THREADS), 0, st, A, lda, n, j0, nb,
                               substitute, out11, ldo, info);
        else
            hipLaunchKernelGGL(chol_panel_kernel<false>, dim3(grid), dim3(CP_THREADS), 0, st, A, lda, n, j0, nb,
                               substitute, out11, ldo, info);
        LU_TRY(hipGetLastError());
        if (r0 < n) {
            if (grid > 1) {
                hipLaunchKernelGGL(chol_store_block_kernel, dim3(1), dim3(256), 0, st, D, lda, L11);
                LU_TRY(hipGetLastError());
            }
            // A22 lower -= L21 * L21^T (U element (k, c) = L21[c, k])
            double *C = A + r0 + (size_t)r0 * lda;
            const double *L21 = A + r0 + (size_t)j0 * lda;
            if (exact)
                LU_TRY((simt_update<double, true, true>(st, C, lda, n - r0, n - r0, L21, lda, L21, lda, 1, nb)));
            else
                LU_TRY((simt_update<double, false, true>(st, C, lda, n - r0, n - r0, L21, lda, L21, lda, 1, nb)));
        }
    }
    return NROCM_OK;
}

// out[0] = the product of the diagonal, 1 * a_00 * a_11 * ... in index order
// (LU::determinant's product, lu.rs:301-314, and Cholesky::determinant's,
// cholesky.rs:155-164), out[1] = out[0] * out[0] (Cholesky::determinant's
// modulus squared), out[2] = 0 + ln(a_00^2) + ln(a_11^2) + ... in index order
// (Cholesky::ln_determinant, cholesky.rs:166-184).  Products and sums are
// one dependent chain: lane 0 walks it while the others prefetch the diagonal.
__global__ __launch_bounds__(64) void diag_det_kernel(const double *A, int lda, int n, double *out)
{
    __shared__ double d[64];
    const int lane = threadIdx.x;
    double prod = 1.0, lnsum = 0.0;
    for (int i0 = 0; i0 < n; i0 += 64) {
        d[lane] = (i0 + lane < n) ? A[(size_t)(i0 + lane) * ((size_t)lda + 1)] : 1.0;
        __syncthreads();
        if (lane == 0) {
            const int cnt = min(64, n - i0);
            for (int q = 0; q < cnt; ++q) {
                prod = prod * d[q];
                lnsum = lnsum + log(d[q] * d[q]);
            }
        }
        __syncthreads();
    }
    if (lane == 0) {
        out[0] = prod;
        out[1] = prod * prod;
        out[2] = lnsum;
    }
}

// The panel step of the windowed LU for the block at k0: the window factor,
// then A21 U11^{-1} for the rows below the window.  Touches only the block's
// own columns, besides ipiv, perm, info and the row plan.
template <typename T>
hipError_t window_panel(hipStream_t st, T *A, int lda, int n, int k0, int *ipiv, int *info, int *plan, int *perm)
{
    const int nb = std::min(64, n - k0);
    const int kw = std::min(n, k0 + WINDOW_ROWS);
    hipLaunchKernelGGL((window_panel_kernel<T>), dim3(1), dim3(512), 0, st, A, lda, k0, nb, kw, ipiv, info,
                       plan, perm);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || kw >= n) return e;
    hipLaunchKernelGGL((trsm_right_upper_kernel<T>), dim3(nrocm_cdiv(n - kw, TRSM_RU_THREADS)),
                       dim3(TRSM_RU_THREADS), 0, st, A, lda, k0, nb, kw, n);
    return hipGetLastError();
}

// Blocked LU with the pivot search of each 64-column block restricted to a
// window of WINDOW_ROWS rows (window_panel_kernel), then the window's row
// plan on the other columns, A21 U11^{-1} for the rows below the window, U12
// and the trailing update.  ipiv has the LAPACK meaning, as for getrf_panels;
// perm (optional) receives the composed row permutation.
//
// Look-ahead of depth one: the panel step of block k+1 needs only the
// trailing update of its own 64 columns, so that part of block k's update
// runs first and the panel step then runs on an auxiliary stream beside the
// update of the remaining columns.  The row plan of block k+1 is applied
// after both have finished (it touches those columns too).
template <typename T>
int getrf_window_impl(nrocm_handle h, hipStream_t st, int n, T *A, int lda, int *ipiv, int *perm, int *info,
                      NrocmTrailing trail)
{
    hipLaunchKernelGGL(fill_int_kernel, dim3(1), dim3(64), 0, st, info, 1, 0);
    LU_TRY(hipGetLastError());
    if (perm) {
        hipLaunchKernelGGL(iota_kernel, dim3(nrocm_cdiv(n, 256)), dim3(256), 0, st, perm, n);
        LU_TRY(hipGetLastError());
    }
    int *plan = (int *)h->small + NROCM_SMALL_PLAN;
    constexpr int NB = 64;
    LU_TRY(window_panel<T>(st, A, lda, n, 0, ipiv, info, plan, perm));
    for (int k0 = 0; k0 < n; k0 += NB) {
        const int nb = std::min(NB, n - k0);
        const int k1 = k0 + nb;
        const int ncol = k0 + (n - k1);
        if (ncol > 0) {
            hipLaunchKernelGGL((apply_plan_kernel<T>), dim3(nrocm_cdiv(ncol, 2)), dim3(256), 0, st, A, lda, plan, 0,
                               k0, k1, n);
            LU_TRY(hipGetLastError());
        }
        if (k1 >= n) break;
        LU_TRY(trsm<T>(st, A, lda, k0, nb, k1, n, false));
        const int k2 = std::min(n, k1 + NB);
        LU_TRY(trailing<T>(st, trail, A, lda, k1, n, k1, k2, k0, nb));
        int s = nrocm_fork_on(h, st, 1);
        if (s != NROCM_OK) return s;
        LU_TRY(window_panel<T>(h->aux[0], A, lda, n, k1, ipiv, info, plan, perm));
        // FP32: two workgroups per CU on all but a few CUs, which stay free for
        // the panel step running beside this update (measured: FP32 gains, the
        // FP64 update with its smaller tiles does not)
        LU_TRY(trailing<T>(st, trail, A, lda, k1, n, k2, n, k0, nb,
                           sizeof(T) == 4 ? 2 * std::max(1, h->num_cus - 8) : 0));
        s = nrocm_join_on(h, st, 1);
        if (s != NROCM_OK) return s;
    }
    return NROCM_OK;
}

}  // namespace

// ---------------------------------------------------------------- internal entry points

// Above WHOLE_ROWS rows the factorisation is some hundred launches on two
// streams, captured once per (shape, buffers, flavour) and replayed.
template <typename T>
int getrf_graph(nrocm_handle h, int m, int n, T *A, int lda, int *ipiv, int *info, NrocmTrailing trail)
{
    if (std::min(m, n) == 0) {
        hipLaunchKernelGGL(fill_int_kernel, dim3(1), dim3(64), 0, h->stream, info, 1, 0);
        NROCM_CHECK_LAUNCH(h);
        return NROCM_OK;
    }
    if (m > COLUMNS_ROWS_MAX) return nrocm_fail(h, NROCM_ERR_UNSUPPORTED, "getrf: more than 16384 rows");
    void *buf = nullptr;
    int s = nrocm_workspace(h, LuBuffer<T>(nullptr, m, n).bytes(), &buf, NROCM_WS_LU);
    if (s != NROCM_OK) return s;
    if (lu_is_whole(m, n)) return getrf_whole<T>(h, h->stream, m, n, A, lda, ipiv, info, buf);
    s = nrocm_aux_init(h);  // streams and events exist before the capture
    if (s != NROCM_OK) return s;
    const long long key[8] = {1000 + (long long)sizeof(T) + 16 * (long long)trail, (long long)m << 32 | n, lda,
                              (long long)A, (long long)ipiv, (long long)info, (long long)buf, h->wait_polls};
    return nrocm_graph_run(h, key, [&](hipStream_t st) {
        return getrf_panels<T>(h, st, m, n, A, lda, ipiv, info, trail, buf);
    });
}

int nrocm_getrf_d(nrocm_handle h, hipStream_t st, int m, int n, double *A, int lda, int *ipiv, int *info,
                  NrocmTrailing trail)
{
    (void)st;
    return getrf_graph<double>(h, m, n, A, lda, ipiv, info, trail);
}

int nrocm_getrf_s(nrocm_handle h, hipStream_t st, int m, int n, float *A, int lda, int *ipiv, int *info,
                  NrocmTrailing trail)
{
    (void)st;
    return getrf_graph<float>(h, m, n, A, lda, ipiv, info, trail);
}

template <typename T>
int getrf_window_graph(nrocm_handle h, int n, T *A, int lda, int *ipiv, int *perm, int *info, NrocmTrailing trail)
{
    if (n <= 64) return getrf_window_impl<T>(h, h->stream, n, A, lda, ipiv, perm, info, trail);
    const int s = nrocm_aux_init(h);  // streams and events exist before the capture
    if (s != NROCM_OK) return s;
    const long long key[8] = {3000 + (long long)sizeof(T) + 16 * (long long)trail, n, lda, (long long)A,
                              (long long)ipiv, (long long)perm, (long long)info, 0};
    return nrocm_graph_run(
        h, key, [&](hipStream_t st) { return getrf_window_impl<T>(h, st, n, A, lda, ipiv, perm, info, trail); });
}

int nrocm_getrf_window_d(nrocm_handle h, int n, double *A, int lda, int *ipiv, int *perm, int *info,
                         NrocmTrailing trail)
{
    return getrf_window_graph<double>(h, n, A, lda, ipiv, perm, info, trail);
}

int nrocm_getrf_window_s(nrocm_handle h, int n, float *A, int lda, int *ipiv, int *perm, int *info,
                         NrocmTrailing trail)
{
    return getrf_window_graph<float>(h, n, A, lda, ipiv, perm, info, trail);
}

// ---------------------------------------------------------------- C ABI

extern "C" {

int nrocm_dgetrf(nrocm_handle h, int m, int n, double *a, int lda, int *ipiv, int *info, int mode)
{
    if (!h) return -1;
    if (m < 0) return -2;
    if (n < 0) return -3;
    if (!a && m > 0 && n > 0) return -4;
    if (lda < std::max(1, m)) return -5;
    if (!ipiv && std::min(m, n) > 0) return -6;
    if (!info) return -7;
    if (mode != NROCM_EXACT && mode != NROCM_FAST) return -8;
    return getrf_graph<double>(h, m, n, a, lda, ipiv, info, mode == NROCM_EXACT ? TRAIL_EXACT : TRAIL_F64);
}

int nrocm_dgetrs(nrocm_handle h, int n, int nrhs, const double *lu, int lda, const int *ipiv, double *b, int ldb,
                 int *info, int mode)
{
    if (!h) return -1;
    if (n < 0) return -2;
    if (nrhs < 0) return -3;
    if (!lu && n > 0) return -4;
    if (lda < std::max(1, n)) return -5;
    if (!ipiv && n > 0) return -6;
    if (!b && n > 0 && nrhs > 0) return -7;
    if (ldb < std::max(1, n)) return -8;
    if (!info) return -9;
    if (mode != NROCM_EXACT && mode != NROCM_FAST) return -10;
    if (n >= NROCM_GETRS_LOOKBACK_MIN)
        return nrocm_getrs_lookback(h, n, nrhs, lu, lda, ipiv, b, ldb, info, mode == NROCM_EXACT);
    return nrocm_getrs_small(h, n, nrhs, lu, lda, ipiv, b, ldb, info, mode == NROCM_EXACT);
}

int nrocm_dpotrf(nrocm_handle h, int n, double *a, int lda, int *info, int mode)
{
    if (!h) return -1;
    if (n < 0) return -2;
    if (!a && n > 0) return -3;
    if (lda < std::max(1, n)) return -4;
    if (!info) return -5;
    if (mode != NROCM_EXACT && mode != NROCM_FAST) return -6;
    if (n <= 64) return nrocm_potrf_small(h, n, a, lda, nullptr, 0, 0, info, mode == NROCM_EXACT);
    return potrf_blocked(h, n, a, lda, info, mode == NROCM_EXACT, 0.0);
}

int nrocm_dpotrf_substitute(nrocm_handle h, int n, double *a, int lda, double substitute, int *info, int mode)
{
    if (!h) return -1;
    if (n < 0) return -2;
    if (!a && n > 0) return -3;
    if (lda < std::max(1, n)) return -4;
    if (!info) return -6;
    if (mode != NROCM_EXACT && mode != NROCM_FAST) return -7;
    if (n <= 64) return nrocm_potrf_small(h, n, a, lda, nullptr, 0, 0, info, mode == NROCM_EXACT, substitute);
    return potrf_blocked(h, n, a, lda, info, mode == NROCM_EXACT, substitute);
}

int nrocm_ddiag_det(nrocm_handle h, int n, const double *a, int lda, double *out)
{
    if (!h) return -1;
    if (n < 0) return -2;
    if (!a && n > 0) return -3;
    if (lda < std::max(1, n)) return -4;
    if (!out) return -5;
    hipLaunchKernelGGL(diag_det_kernel, dim3(1), dim3(64), 0, h->stream, a, lda, n, out);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}

int nrocm_dpotrs(nrocm_handle h, int n, int nrhs, const double *l, int lda, double *b, int ldb, int mode)
{
    if (!h) return -1;
    if (n < 0) return -2;
    if (nrhs < 0) return -3;
    if (!l && n > 0) return -4;
    if (lda < std::max(1, n)) return -5;
    if (!b && n > 0 && nrhs > 0) return -6;
    if (ldb < std::max(1, n)) return -7;
    if (mode != NROCM_EXACT && mode != NROCM_FAST) return -8;
    if (n == 0 || nrhs == 0) return NROCM_OK;
    if (n >= NROCM_GETRS_LOOKBACK_MIN) return nrocm_potrs_lookback(h, n, nrhs, l, lda, b, ldb, mode == NROCM_EXACT);
    return nrocm_potrs_small(h, n, nrhs, l, lda, b, ldb, mode == NROCM_EXACT);
}

}  // extern "C"
