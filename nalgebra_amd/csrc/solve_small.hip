// The single-matrix solves below n = NROCM_GETRS_LOOKBACK_MIN rows: LU::
// solve_mut (src/linalg/lu.rs:242-260), Cholesky::solve_mut (cholesky.rs:
// 122-129) and QR::solve_mut's upper solve (qr.rs:224-256), one launch each.
// A workgroup takes CH right-hand sides through the whole solve, its four
// wavefronts the 64-row blocks in turn (solve_sweep.hpp); everything it
// exchanges is in its own LDS, so calls on several streams share nothing.
// 300 right-hand sides are 150 workgroups of two instead of 300 solves in a row:
// n = 300 with 300 right-hand sides 124.8 ms -> 60 us, n = 500 with one
// 827 -> 72 us (before: one workgroup, a barrier and a load per step).
#include "internal_launch.hpp"
#include "solve_sweep.hpp"

#include <algorithm>

using namespace nrocm_sweep;

namespace {

enum Op { OP_LU, OP_CHOL, OP_QR };

constexpr int THREADS = SWEEP_WAVES * 64;
constexpr int DOT_LOADERS = SWEEP_WAVES - 1;
constexpr int DOT_ROWREGS = dot_lane_elements(NROCM_GETRS_LOOKBACK_MIN - 1, DOT_LOADERS);

// LDS, in doubles: x by sweep position (two sweeps), the staged diagonal
// blocks (or the transposed solve's column slots), then the permutation and
// its plans (ints).
__host__ __device__ constexpr int pad64(int n) { return (n + 63) & ~63; }
__host__ __device__ constexpr int stage_doubles(int n, int ch, int op, bool exact)
{
    const int diag = (n <= LB ? 1 : DSLOTS) * LB * LB;
    const int dot = op == OP_CHOL && exact ? dot_doubles(n, ch) : 0;
    return diag > dot ? diag : dot;
}
constexpr size_t LDS_MOST = NROCM_LDS_BYTES - 64;  // the kernel has a few static words
size_t lds_bytes(int n, int ch, int op, bool exact)
{
    const size_t x = (size_t)pad64(n) * ch * (op == OP_QR || (op == OP_CHOL && exact) ? 1 : 2);
    return (x + stage_doubles(n, ch, op, exact)) * sizeof(double) +
           (op == OP_LU ? (pad64(n) + 192 * SWEEP_WAVES) * sizeof(int) : 0);
}

// All blocks of one sweep; x of sweep position t ends at xs[t * CH + c].
// init(c, r) gives the right-hand sides, out(acc, t, r) takes the results.
template <bool EXACT, int KIND, int CH, typename Init, typename Out>
__device__ __forceinline__ void sweep(const double *__restrict__ M, int lda, int n, const double *__restrict__ dg,
                                      double *xs, double *D, int *done, int base, Init init, Out out)
{
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nblk = (n + LB - 1) / LB;
    for (int k = w; k < nblk; k += SWEEP_WAVES) {
        const int t = k * LB + lane;
        const int tc = min(t, n - 1);
        const int r = from_top(KIND) ? tc : n - 1 - tc;
        const double d = diag_of<KIND>(M, lda, dg, r);
        double acc[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[c] = init(c, r);
        sweep_block<EXACT, KIND, CH>(acc, M, lda, n, k, d, D + (k % DSLOTS) * LB * LB, lane, [&](int J) {
            wait_done(done, base + J + 1);
            return xs + J * LB * CH;
        });
#pragma unroll
        for (int c = 0; c < CH; ++c) xs[t * CH + c] = acc[c];
        signal_done(done, base + k + 1, lane);
        if (t < n) out(acc, r, d);
    }
}

template <bool EXACT, int OP, int CH>
__global__ __launch_bounds__(THREADS) void solve_small_kernel(const double *__restrict__ M, int lda, int n,
                                                              const int *__restrict__ ipiv,
                                                              const double *__restrict__ dg, double *B, int ldb,
                                                              int nrhs, int *info)
{
    extern __shared__ __align__(16) double lds[];
    __shared__ int done, fail;
    const int np = (n + 63) & ~63;
    const int c0 = blockIdx.x * CH;
    constexpr bool ONE_X = OP == OP_QR || (OP == OP_CHOL && EXACT);
    double *x0 = lds, *x1 = ONE_X ? lds : lds + np * CH;
    double *stage = lds + np * CH * (ONE_X ? 1 : 2);
    const int nblk = np / 64;
    if (threadIdx.x == 0) {
        done = 0;
        fail = 0;
    }
    auto b_at = [&](int c, int row) -> double {
        return c0 + c < nrhs ? B[row + (size_t)(c0 + c) * ldb] : 0.0;
    };
    auto store = [&](const double (&acc)[CH], int r) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
            if (c0 + c < nrhs) B[r + (size_t)(c0 + c) * ldb] = acc[c];
    };
    if constexpr (OP == OP_LU) {
        int *perm = (int *)(stage + stage_doubles(n, CH, OP, EXACT));
        compose_perm<SWEEP_WAVES, false>(ipiv, n, perm, perm + np, nullptr);
        sweep<EXACT, LU_FWD, CH>(
            M, lda, n, dg, x0, stage, &done, 0, [&](int c, int r) { return b_at(c, perm[r]); },
            [](const double (&)[CH], int, double) {});
        __syncthreads();
        sweep<EXACT, LU_BWD, CH>(
            M, lda, n, dg, x1, stage, &done, nblk, [&](int c, int r) { return x0[r * CH + c]; },
            [&](const double (&acc)[CH], int r, double d) {
                store(acc, r);
                if (d == 0.0) atomicMax(&fail, r + 1);
            });
    } else if constexpr (OP == OP_QR) {
        __syncthreads();
        sweep<EXACT, QR_BWD, CH>(M, lda, n, dg, x0, stage, &done, 0, b_at,
                                 [&](const double (&acc)[CH], int r, double d) {
                                     store(acc, r);
                                     if (d == 0.0) atomicMax(&fail, r + 1);
                                 });
    } else {
        __syncthreads();
        sweep<EXACT, CHOL_FWD, CH>(M, lda, n, dg, x0, stage, &done, 0, b_at,
                                   [](const double (&)[CH], int, double) {});
        __syncthreads();
        if constexpr (EXACT) {
            chol_dot_backward<DOT_ROWREGS, DOT_LOADERS, CH>(M, lda, n, x0, stage);
            __syncthreads();
            for (int e = threadIdx.x; e < n * CH; e += THREADS) {
                const int c = e / n, r = e % n;
                if (c0 + c < nrhs) B[r + (size_t)(c0 + c) * ldb] = x0[r * CH + c];
            }
        } else {
            sweep<EXACT, CHOL_BWD_FAST, CH>(
                M, lda, n, dg, x1, stage, &done, nblk, [&](int c, int r) { return x0[r * CH + c]; },
                [&](const double (&acc)[CH], int r, double) { store(acc, r); });
        }
    }
    if constexpr (OP != OP_CHOL) {
        // every workgroup finds the same diagonal
        __syncthreads();
        if (threadIdx.x == 0 && info && blockIdx.x == 0) *info = fail;
    }
}

// Up to TINY rows a thread takes a right-hand side through the whole solve, matrix
// and vector in registers: the launch and one trip to memory are all there is.  (LU,
// EXACT, one right-hand side, us, with the kernel above and this one: n = 1 6.2 and 4.1,
// 4 6.4 and 4.3, 8 7.0 and 5.0; Cholesky 4 6.5 and 4.0, 8 8.3 and 4.0.)
constexpr int TINY = 8;

template <bool EXACT, int OP>
__global__ __launch_bounds__(64) void solve_tiny_kernel(const double *__restrict__ M, int lda, int n,
                                                        const int *__restrict__ ipiv, const double *__restrict__ dg,
                                                        double *B, int ldb, int nrhs, int *info)
{
    const int c = blockIdx.x * 64 + threadIdx.x;
    double *const b = B + (size_t)min(c, nrhs - 1) * ldb;
    double m[TINY][TINY], x[TINY], d[TINY];  // m[j][i]: element (i, j)
    int p[TINY];
#pragma unroll
    for (int j = 0; j < TINY; ++j) {
#pragma unroll
        for (int i = 0; i < TINY; ++i) m[j][i] = M[min(i, n - 1) + (size_t)min(j, n - 1) * lda];
        x[j] = b[min(j, n - 1)];
        d[j] = OP == OP_QR ? fabs(dg[min(j, n - 1)]) : m[j][j];
        p[j] = OP == OP_LU ? ipiv[min(j, n - 1)] : j;
    }
    if constexpr (OP == OP_LU) {
#pragma unroll
        for (int i = 0; i < TINY; ++i) {
            if (i >= n) break;
            double t = x[i];
#pragma unroll
            for (int j = 0; j < TINY; ++j) t = j == p[i] && j < n ? x[j] : t;
#pragma unroll
            for (int j = 0; j < TINY; ++j) x[j] = j == p[i] && j < n ? x[i] : x[j];
            x[i] = t;
        }
    }
    auto axpy = [&](int r, int i, double a) {
        double acc[1] = {x[r]};
        const double f[1] = {x[i]};
        step<EXACT, 1>(acc, f, a);
        x[r] = acc[0];
    };
    if constexpr (OP != OP_QR) {
#pragma unroll
        for (int i = 0; i < TINY; ++i) {
            if (i >= n) break;
            if constexpr (OP == OP_CHOL) x[i] = x[i] / d[i];
#pragma unroll
            for (int r = i + 1; r < TINY; ++r) axpy(r, i, m[i][r]);
        }
    }
    int fail = 0;
#pragma unroll
    for (int i = TINY - 1; i >= 0; --i) {
        if (i >= n) continue;
        if constexpr (OP == OP_CHOL && EXACT) {
            double res = 0.0;  // dotx of fewer than eight elements
#pragma unroll
            for (int e = i + 1; e < TINY; ++e)
                if (e < n) res += m[i][e] * x[e];
            x[i] = (x[i] - res) / d[i];
        } else {
            if (d[i] == 0.0 && fail == 0) fail = i + 1;
            x[i] = x[i] / d[i];
#pragma unroll
            for (int r = 0; r < i; ++r) axpy(r, i, OP == OP_CHOL ? m[r][i] : m[i][r]);
        }
    }
#pragma unroll
    for (int i = 0; i < TINY; ++i)
        if (i < n && c < nrhs) b[i] = x[i];
    if (OP != OP_CHOL && info && c == 0) *info = fail;
}

__global__ void zero_info_kernel(int *info) { *info = 0; }

template <bool EXACT, int OP, int CH>
int launch(nrocm_handle h, const double *M, int lda, int n, const int *ipiv, const double *dg, double *B, int ldb,
           int nrhs, int *info)
{
    const size_t lds = lds_bytes(n, CH, OP, EXACT);
    nrocm_allow_lds<solve_small_kernel<EXACT, OP, CH>>(h->device);
    hipLaunchKernelGGL((solve_small_kernel<EXACT, OP, CH>), dim3(nrocm_cdiv(nrhs, CH)), dim3(THREADS), lds, h->stream,
                       M, lda, n, ipiv, dg, B, ldb, nrhs, info);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}

template <int OP>
int solve_small(nrocm_handle h, const double *M, int lda, int n, const int *ipiv, const double *dg, double *B, int ldb,
                int nrhs, int *info, bool exact)
{
    if (n == 0 || nrhs == 0) {
        if (info) {
            hipLaunchKernelGGL(zero_info_kernel, dim3(1), dim3(1), 0, h->stream, info);
            NROCM_CHECK_LAUNCH(h);
        }
        return NROCM_OK;
    }
    if (n <= TINY) {
        const auto kernel = exact ? solve_tiny_kernel<true, OP> : solve_tiny_kernel<OP == OP_QR, OP>;  // QR: always exact
        hipLaunchKernelGGL(kernel, dim3(nrocm_cdiv(nrhs, 64)), dim3(64), 0, h->stream, M, lda, n, ipiv, dg, B, ldb,
                           nrhs, info);
        NROCM_CHECK_LAUNCH(h);
        return NROCM_OK;
    }
    // fewer right-hand sides per workgroup where the LDS does not hold them
    // (QR's solve above n = 2,900)
#define NROCM_SMALL(CH)                                                                       \
    (exact ? launch<true, OP, CH>(h, M, lda, n, ipiv, dg, B, ldb, nrhs, info)                 \
           : launch<OP == OP_QR, OP, CH>(h, M, lda, n, ipiv, dg, B, ldb, nrhs, info))
    const int fit = lds_bytes(n, 4, OP, exact) <= LDS_MOST ? 4 : lds_bytes(n, 2, OP, exact) <= LDS_MOST ? 2 : 1;
    const int ch = std::min(fit, rhs_per_group(h->num_cus, nrhs, 1));
    return ch == 1 ? NROCM_SMALL(1) : ch == 2 ? NROCM_SMALL(2) : NROCM_SMALL(4);
#undef NROCM_SMALL
}

}  // namespace

int nrocm_getrs_small(nrocm_handle h, int n, int nrhs, const double *lu, int lda, const int *ipiv, double *b, int ldb,
                      int *info, bool exact)
{
    return solve_small<OP_LU>(h, lu, lda, n, ipiv, nullptr, b, ldb, nrhs, info, exact);
}

int nrocm_potrs_small(nrocm_handle h, int n, int nrhs, const double *l, int lda, double *b, int ldb, bool exact)
{
    return solve_small<OP_CHOL>(h, l, lda, n, nullptr, nullptr, b, ldb, nrhs, nullptr, exact);
}

int nrocm_qr_rsolve(nrocm_handle h, int n, int nrhs, const double *qr, int lda, const double *diag, double *b, int ldb,
                    int *info)
{
    // one workgroup's LDS holds x up to here; no scratch is shared
    if (lds_bytes(n, 1, OP_QR, true) > LDS_MOST)
        return nrocm_qr_rsolve_lookback(h, n, nrhs, qr, lda, diag, b, ldb, info);
    return solve_small<OP_QR>(h, qr, lda, n, nullptr, diag, b, ldb, nrhs, info, true);
}
