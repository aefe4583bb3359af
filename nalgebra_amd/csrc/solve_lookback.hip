// LU::solve_mut (src/linalg/lu.rs:242-260), Cholesky::solve_mut (cholesky.rs:
// 122-129) and QR::solve_mut's upper solve (qr.rs:224-256) for any n, spread
// over workgroups of four 64-row blocks (solve_sweep.hpp).
//
// Workgroups take tickets in sweep order (all right-hand-side groups of one
// block of 256 rows before the next), so every workgroup that a wait is for is
// already running.  Inside a workgroup finished blocks are handed over in LDS;
// between workgroups a value is published as two 64-bit words, each holding a
// 32-bit half of the double next to the launch's epoch, written as one atomic
// word; a reader polls the words until they carry the epoch, so data and
// readiness arrive together.  Four blocks per workgroup keep three of four
// hand-overs in LDS (about 2 us less each than between XCDs) and still give a
// large solve a workgroup per 256 rows to stream its part of the matrix.
// All right-hand sides go through one launch, CH of them per workgroup.
// n = 4096, 8 right-hand sides: forward 9.5 -> 0.21 ms, backward 18.6 -> 0.25 ms
// (before: one wavefront per 64 rows, one right-hand side at a time, a load and a
// lane mask in every step of the diagonal block).
// The tag array is cleared at the start of every call and every launch of a
// call has its own epoch.  Waits are bounded: a wait that runs out takes NaN for
// the values, sets info to -1 (Cholesky has none) and the kernel still exits.
#include "internal_launch.hpp"
#include "solve_sweep.hpp"

#include <algorithm>
#include <mutex>

using namespace nrocm_sweep;

namespace {

constexpr int THREADS = SWEEP_WAVES * 64;
constexpr int SUPER = SWEEP_WAVES * LB;   // rows per workgroup
constexpr int PERM_LDS_MAX = 16384;       // composed permutation kept in LDS up to this n
constexpr int PREP_WAVES = 16;
constexpr int TICKETS = 60;               // launches per clearing of the header
constexpr size_t HEADER_BYTES = 256;      // tickets

typedef unsigned long long u64;

template <int CH>
__device__ __forceinline__ void publish(u64 *dst, unsigned epoch, const double (&v)[CH])
{
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const u64 bits = (u64)__double_as_longlong(v[c]);
        __hip_atomic_store(dst + 2 * c, ((u64)epoch << 32) | (bits & 0xffffffffull), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(dst + 2 * c + 1, ((u64)epoch << 32) | (bits >> 32), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

__device__ __forceinline__ double untag(u64 lo, u64 hi)
{
    return __longlong_as_double((long long)((hi << 32) | (lo & 0xffffffffull)));
}

template <int CH>
__device__ __forceinline__ void await(const u64 *src, unsigned epoch, double (&v)[CH], int *info, long limit)
{
    u64 w[2 * CH];
    long spins = 0;
    bool lost = false;
    for (;;) {
        bool ok = true;
#pragma unroll
        for (int c = 0; c < 2 * CH; ++c) w[c] = __hip_atomic_load(src + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int c = 0; c < 2 * CH; ++c) ok = ok && (unsigned)(w[c] >> 32) == epoch;
        if (ok) break;
        if (++spins >= limit) {
            lost = true;
            if (info) atomicExch(info, -1);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) v[c] = lost ? __builtin_nan("") : untag(w[2 * c], w[2 * c + 1]);
}

// One sweep of a large solve.  LU_FWD reads b through perm and publishes y;
// LU_BWD takes y from the words LU_FWD left (epoch_in) and writes b, like the
// other kinds, which read b.
template <bool EXACT, int KIND, int CH>
__global__ __launch_bounds__(THREADS) void sweep_lookback_kernel(const double *__restrict__ M, int lda, int n,
                                                                 const double *__restrict__ dg,
                                                                 const int *__restrict__ perm, double *B, int ldb,
                                                                 int nrhs, int ngroups, int *ticket, u64 *tags,
                                                                 unsigned epoch_in, unsigned epoch, int *info, long limit)
{
    __shared__ __align__(16) double D[DSLOTS * LB * LB];
    __shared__ __align__(16) double xs[SUPER * CH];               // this workgroup's blocks
    __shared__ __align__(16) double xw[SWEEP_WAVES][LB * CH];     // a polled block, per wavefront
    __shared__ int my, done;
    if (threadIdx.x == 0) {
        my = atomicAdd(ticket, 1);
        done = 0;
    }
    __syncthreads();
    const int S = my / ngroups, g = my % ngroups;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int k0 = S * SWEEP_WAVES, k = k0 + w;
    const int nblk = (n + LB - 1) / LB;
    if (k >= nblk) return;  // nothing waits for it
    const int c0 = g * CH;
    u64 *const gtags = tags + (size_t)g * n * CH * 2;
    const int t = k * LB + lane;
    const int tc = min(t, n - 1);
    const int r = from_top(KIND) ? tc : n - 1 - tc;
    const double d = diag_of<KIND>(M, lda, dg, r);
    double acc[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        if constexpr (KIND == LU_BWD) {
            const u64 *src = gtags + ((size_t)r * CH + c) * 2;
            acc[c] = untag(src[0], src[1]);
        } else {
            const int row = KIND == LU_FWD ? perm[r] : r;
            acc[c] = c0 + c < nrhs ? B[row + (size_t)(c0 + c) * ldb] : 0.0;
        }
    }
    sweep_block<EXACT, KIND, CH>(acc, M, lda, n, k, d, D + (w % DSLOTS) * LB * LB, lane, [&](int J) -> const double * {
        if (J >= k0) {
            wait_done(&done, J - k0 + 1);
            return xs + (J - k0) * LB * CH;
        }
        // a finished block is never the matrix's last one: it is full
        const int u = J * LB + lane;
        double v[CH];
        await<CH>(gtags + (size_t)(from_top(KIND) ? u : n - 1 - u) * CH * 2, epoch, v, info, limit);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int c = 0; c < CH; ++c) xw[w][lane * CH + c] = v[c];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        return xw[w];
    });
    if (t < n && (KIND == LU_FWD || k0 + SWEEP_WAVES < nblk)) publish<CH>(gtags + (size_t)r * CH * 2, epoch, acc);
#pragma unroll
    for (int c = 0; c < CH; ++c) xs[(w * LB + lane) * CH + c] = acc[c];
    signal_done(&done, w + 1, lane);
    if (t < n) {
        if constexpr (KIND != LU_FWD) {
#pragma unroll
            for (int c = 0; c < CH; ++c)
                if (c0 + c < nrhs) B[r + (size_t)(c0 + c) * ldb] = acc[c];
        }
        if constexpr (KIND == LU_BWD || KIND == QR_BWD) {
            // 1 + the largest i with a zero diagonal; an invalid pivot's -2 stays
            if (d == 0.0 && *info != -2) atomicMax(info, r + 1);
        }
    }
}

// Clears the tags and tickets; the first workgroup also composes the row
// permutation (ipiv non-null) and sets info.
__global__ __launch_bounds__(PREP_WAVES * 64) void prep_kernel(u64 *tags, size_t ntag, int *header, int *info,
                                                               int set_info, const int *__restrict__ ipiv, int n,
                                                               int *perm)
{
    extern __shared__ int sp[];
    __shared__ int plan[PREP_WAVES * 192];
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < ntag; i += (size_t)gridDim.x * blockDim.x)
        tags[i] = 0;
    if (blockIdx.x != 0) return;
    if (threadIdx.x < HEADER_BYTES / sizeof(int)) header[threadIdx.x] = 0;
    if (set_info && threadIdx.x == 0) *info = 0;
    if (!ipiv) return;
    __syncthreads();
    if (n <= PERM_LDS_MAX) {
        compose_perm<PREP_WAVES, false>(ipiv, n, sp, plan, info);
        for (int i = threadIdx.x; i < n; i += blockDim.x) perm[i] = sp[i];
    } else {
        compose_perm<PREP_WAVES, true>(ipiv, n, perm, plan, info);
    }
}

// info = 1 + the largest i with U_ii == 0 (solve_mut returns false), or 0.
__global__ void zero_diag_kernel(const double *__restrict__ LU, int lda, int n, int *info)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && LU[i + (size_t)i * lda] == 0.0 && *info != -2) atomicMax(info, i + 1);
}

// NROCM_EXACT transposed Cholesky solve, CH right-hand sides per workgroup.
template <int NR, int CH>
__global__ __launch_bounds__(512) void chol_dot_kernel(const double *__restrict__ L, int lda, int n, double *B,
                                                       int ldb, int nrhs)
{
    extern __shared__ __align__(16) double lds[];
    double *xs = lds, *slots = lds + (size_t)n * CH;
    const int c0 = blockIdx.x * CH;
    for (int e = threadIdx.x; e < n * CH; e += 512) {
        const int c = e / n, r = e % n;
        xs[r * CH + c] = c0 + c < nrhs ? B[r + (size_t)(c0 + c) * ldb] : 0.0;
    }
    __syncthreads();
    chol_dot_backward<NR, 7, CH>(L, lda, n, xs, slots);
    __syncthreads();
    for (int e = threadIdx.x; e < n * CH; e += 512) {
        const int c = e / n, r = e % n;
        if (c0 + c < nrhs) B[r + (size_t)(c0 + c) * ldb] = xs[r * CH + c];
    }
}

constexpr size_t dot_lds_bytes(int n, int ch)
{
    return ((size_t)n * ch + dot_doubles(n, ch)) * sizeof(double);
}

// Largest n of chol_dot_kernel: three columns of products and x within the LDS.
constexpr int CHOL_DOT_MAX = 4096;
static_assert(dot_lane_elements(2048, 7) <= 5 && dot_lane_elements(CHOL_DOT_MAX, 7) <= 10, "elements per lane");
static_assert(dot_lds_bytes(CHOL_DOT_MAX, 1) <= NROCM_LDS_BYTES, "x and three columns fit the LDS");

// The same for larger n: one wavefront, lanes 0..7 the accumulators, L read
// straight from memory, x kept in LDS (XS_LDS) or, beyond the LDS, in b itself
// (each new x_i is then released to the L2 and the vector L1 dropped before
// the next row reads it: other lanes read values lane 0 wrote in this launch).
template <bool XS_LDS>
__global__ __launch_bounds__(64) void chol_backward_dot_kernel(const double *__restrict__ L, int lda, int n,
                                                               double *b)
{
    extern __shared__ double xs_dyn[];
    const int lane = threadIdx.x;
    double *xb = XS_LDS ? xs_dyn : b;
    if constexpr (XS_LDS) {
        for (int r = lane; r < n; r += 64) xs_dyn[r] = b[r];
        __syncthreads();
    }
    auto xload = [&](int idx) -> double { return xb[idx]; };
    for (int i = n - 1; i >= 0; --i) {
        const int len = n - i - 1;
        const int full = len & ~7;
        const double *li = L + (i + 1) + (size_t)i * lda;
        double a = 0.0;
        if (lane < 8) {
#pragma unroll 4
            for (int e = lane; e < full; e += 8) a += li[e] * xload(i + 1 + e);
        }
        double res = 0.0;
        res += lane_value(a, 0) + lane_value(a, 4);
        res += lane_value(a, 1) + lane_value(a, 5);
        res += lane_value(a, 2) + lane_value(a, 6);
        res += lane_value(a, 3) + lane_value(a, 7);
        for (int e = full; e < len; ++e) res += li[e] * xload(i + 1 + e);
        const double xi = (xload(i) - res) / L[i + (size_t)i * lda];
        __syncthreads();  // every lane has read x_i's old value
        if (lane == 0) xb[i] = xi;
        if constexpr (!XS_LDS) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        if constexpr (!XS_LDS) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    if constexpr (XS_LDS) {
        for (int r = lane; r < n; r += 64) b[r] = xs_dyn[r];
    }
}

// Largest n whose x chol_backward_dot_kernel keeps in LDS.
constexpr int CHOL_XS_LDS_MAX = 19968;

size_t perm_bytes(int n) { return ((size_t)n * sizeof(int) + 255) & ~(size_t)255; }
size_t tag_bytes(int n, int cols) { return (size_t)n * cols * 2 * sizeof(u64); }

// Right-hand sides of one launch: at most 64 MB of tags.
int launch_cols(int n, int nrhs)
{
    const long most = std::max(4L, (64L << 20) / ((long)n * 16) & ~3L);
    return (int)std::min<long>(std::max(nrhs, 1), most);
}

struct Sweeps {
    nrocm_handle h;
    hipStream_t st;
    const double *M;
    int lda, n;
    const double *dg;
    const int *perm;
    int *ticket;
    u64 *tags;
    int *info;
    unsigned epoch = 0;

    template <bool EXACT, int KIND, int CH>
    int launch(double *B, int ldb, int cols)
    {
        const int ngroups = (int)nrocm_cdiv(cols, CH);
        const unsigned in = epoch++;
        hipLaunchKernelGGL((sweep_lookback_kernel<EXACT, KIND, CH>), dim3(nrocm_cdiv(n, SUPER) * ngroups),
                           dim3(THREADS), 0, st, M, lda, n, dg, perm, B, ldb, cols, ngroups, ticket + in % TICKETS,
                           tags, in, epoch, info, nrocm_wait_limit(h, SPIN_LIMIT));
        NROCM_CHECK_LAUNCH(h);
        return NROCM_OK;
    }
    template <bool EXACT, int KIND>
    int run(double *B, int ldb, int cols, int ch)
    {
        return ch == 1 ? launch<EXACT, KIND, 1>(B, ldb, cols)
               : ch == 2 ? launch<EXACT, KIND, 2>(B, ldb, cols)
                         : launch<EXACT, KIND, 4>(B, ldb, cols);
    }
};

enum Op { OP_LU, OP_CHOL, OP_QR };

int chol_dot(nrocm_handle h, hipStream_t st, const double *L, int lda, int n, double *b, int ldb, int nrhs)
{
    if (n <= CHOL_DOT_MAX) {
        const int fit = dot_lds_bytes(n, 4) <= NROCM_LDS_BYTES ? 4 : dot_lds_bytes(n, 2) <= NROCM_LDS_BYTES ? 2 : 1;
        const int ch = std::min(fit, rhs_per_group(h->num_cus, nrhs, 1));
        const size_t lds = dot_lds_bytes(n, ch);
        const dim3 grid(nrocm_cdiv(nrhs, ch));
#define NROCM_DOT(NR, CH)                                                                                 \
    do {                                                                                                  \
        nrocm_allow_lds<chol_dot_kernel<NR, CH>>(h->device);                                                       \
        hipLaunchKernelGGL((chol_dot_kernel<NR, CH>), grid, dim3(512), lds, st, L, lda, n, b, ldb, nrhs);  \
    } while (0)
        if (n <= 2048) {
            if (ch == 4) NROCM_DOT(5, 4);
            else if (ch == 2) NROCM_DOT(5, 2);
            else NROCM_DOT(5, 1);
        } else {
            if (ch == 2) NROCM_DOT(10, 2);
            else NROCM_DOT(10, 1);
        }
#undef NROCM_DOT
        NROCM_CHECK_LAUNCH(h);
        return NROCM_OK;
    }
    const bool lds = n <= CHOL_XS_LDS_MAX;
    if (lds) nrocm_allow_lds<chol_backward_dot_kernel<true>>(h->device);
    for (int c = 0; c < nrhs; ++c) {
        double *bc = b + (size_t)c * ldb;
        if (lds)
            hipLaunchKernelGGL(chol_backward_dot_kernel<true>, dim3(1), dim3(64), (size_t)n * sizeof(double), st, L,
                               lda, n, bc);
        else
            hipLaunchKernelGGL(chol_backward_dot_kernel<false>, dim3(1), dim3(64), 0, st, L, lda, n, bc);
        NROCM_CHECK_LAUNCH(h);
    }
    return NROCM_OK;
}

// Enqueues a solve on st; `scratch` holds the header, the permutation and the
// tags of `cols` right-hand sides at a time.  Allocates nothing.
template <int OP>
int solve(nrocm_handle h, hipStream_t st, int n, int nrhs, const double *M, int lda, const int *ipiv,
          const double *dg, double *b, int ldb, int *info, bool exact, void *scratch, int cols)
{
    char *base = (char *)scratch;
    int *header = (int *)base;
    int *perm = (int *)(base + HEADER_BYTES);
    u64 *tags = (u64 *)(base + HEADER_BYTES + perm_bytes(n));
    Sweeps s{h, st, M, lda, n, dg, perm, header, tags, info};
    const int ch = std::min(cols == 1 ? 1 : cols == 2 ? 2 : 4, rhs_per_group(h->num_cus, std::min(cols, nrhs), nrocm_cdiv(n, SUPER)));
    for (int c0 = 0; c0 == 0 || c0 < nrhs; c0 += cols) {
        const int cc = std::min(cols, nrhs - c0);
        const size_t ntag = cc > 0 ? tag_bytes(n, (int)nrocm_cdiv(cc, ch) * ch) / sizeof(u64) : 0;
        // the tags are cleared before every pair of sweeps, the permutation
        // and info are made once
        const int *piv = c0 == 0 ? ipiv : nullptr;
        const unsigned blocks = std::min<unsigned>(512, std::max(1u, nrocm_cdiv(ntag, PREP_WAVES * 64 * 4)));
        nrocm_allow_lds<prep_kernel>(h->device);
        hipLaunchKernelGGL(prep_kernel, dim3(blocks), dim3(PREP_WAVES * 64),
                           piv && n <= PERM_LDS_MAX ? (size_t)n * sizeof(int) : 0, st, tags, ntag, header, info,
                           c0 == 0 && info, piv, n, perm);
        NROCM_CHECK_LAUNCH(h);
        if (n == 0) return NROCM_OK;
        if (cc <= 0) {  // no right-hand sides: only the diagonal is looked at
            if constexpr (OP == OP_LU) {
                hipLaunchKernelGGL(zero_diag_kernel, dim3(nrocm_cdiv(n, 256)), dim3(256), 0, st, M, lda, n, info);
                NROCM_CHECK_LAUNCH(h);
            }
            return NROCM_OK;
        }
        s.epoch = 0;
        double *bc = b + (size_t)c0 * ldb;
        int e = NROCM_OK;
        if constexpr (OP == OP_LU) {
            e = exact ? s.run<true, LU_FWD>(bc, ldb, cc, ch) : s.run<false, LU_FWD>(bc, ldb, cc, ch);
            if (e == NROCM_OK) e = exact ? s.run<true, LU_BWD>(bc, ldb, cc, ch) : s.run<false, LU_BWD>(bc, ldb, cc, ch);
        } else if constexpr (OP == OP_QR) {
            e = s.run<true, QR_BWD>(bc, ldb, cc, ch);
        } else {
            e = exact ? s.run<true, CHOL_FWD>(bc, ldb, cc, ch) : s.run<false, CHOL_FWD>(bc, ldb, cc, ch);
            if (e == NROCM_OK) e = exact ? chol_dot(h, st, M, lda, n, bc, ldb, cc) : s.run<false, CHOL_BWD_FAST>(bc, ldb, cc, ch);
        }
        if (e != NROCM_OK) return e;
    }
    return NROCM_OK;
}

template <int OP>
int solve_in_workspace(nrocm_handle h, int n, int nrhs, const double *M, int lda, const int *ipiv, const double *dg,
                       double *b, int ldb, int *info, bool exact)
{
    const int cols = launch_cols(n, nrhs);
    void *ws = nullptr;
    const int s = nrocm_workspace(h, HEADER_BYTES + perm_bytes(n) + tag_bytes(n, (cols + 3) & ~3), &ws);
    if (s != NROCM_OK) return s;
    return solve<OP>(h, h->stream, n, nrhs, M, lda, ipiv, dg, b, ldb, info, exact, ws, cols);
}

}  // namespace

int nrocm_getrs_lookback(nrocm_handle h, int n, int nrhs, const double *lu, int lda, const int *ipiv, double *b,
                         int ldb, int *info, bool exact)
{
    return solve_in_workspace<OP_LU>(h, n, nrhs, lu, lda, ipiv, nullptr, b, ldb, info, exact);
}

int nrocm_potrs_lookback(nrocm_handle h, int n, int nrhs, const double *L, int lda, double *b, int ldb, bool exact)
{
    return solve_in_workspace<OP_CHOL>(h, n, nrhs, L, lda, nullptr, nullptr, b, ldb, nullptr, exact);
}

int nrocm_qr_rsolve_lookback(nrocm_handle h, int n, int nrhs, const double *qr, int lda, const double *diag, double *b,
                             int ldb, int *info)
{
    return solve_in_workspace<OP_QR>(h, n, nrhs, qr, lda, nullptr, diag, b, ldb, info, true);
}

// ---------------------------------------------------------------- the allocation-free solve
// nrocm_dgetrs_noalloc keeps the solve's scratch (ticket, permutation, tags)
// in this file-scope device array instead of the handle's workspace: each GPU
// the library runs on holds one copy, NROCM_NOALLOC_SCRATCH_BYTES bytes, until
// the process ends.  Host code never passes the array's name to a kernel (on
// the host it is a stand-in, not a device address): the device address is
// looked up once per device and kept in scratch_dev.
namespace {

constexpr size_t NROCM_NOALLOC_SCRATCH_BYTES =
    256 + (((size_t)NROCM_NOALLOC_MAX_N * sizeof(int) + 255) & ~(size_t)255) +
    2 * (size_t)NROCM_NOALLOC_MAX_N * sizeof(unsigned long long);

}  // namespace

static __device__ __align__(256) unsigned char scratch[NROCM_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
void *scratch_dev[kMaxDevices] = {};

// Device address of `scratch` on the handle's device (looked up on the first
// call for that device, with the device current).
int scratch_ptr(nrocm_handle h, void **out)
{
    if (h->device < 0 || h->device >= kMaxDevices) return nrocm_fail(h, NROCM_ERR_UNSUPPORTED, "device index >= 64");
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_dev[h->device]) {
        int cur = 0;
        NROCM_CHECK_HIP(h, hipGetDevice(&cur));
        if (cur != h->device) NROCM_CHECK_HIP(h, hipSetDevice(h->device));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != h->device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return nrocm_fail_hip(h, e, "hipGetSymbolAddress(scratch)");
        scratch_dev[h->device] = p;
    }
    *out = scratch_dev[h->device];
    return NROCM_OK;
}

}  // namespace

extern "C" int nrocm_dgetrs_noalloc(nrocm_handle h, int n, int nrhs, const double *lu, int lda, const int *ipiv,
                                    double *b, int ldb, int *info, int mode)
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
    if (n > NROCM_NOALLOC_MAX_N)
        return nrocm_fail(h, NROCM_ERR_UNSUPPORTED,
                          "getrs_noalloc: n exceeds NROCM_NOALLOC_MAX_N (16384), the rows its static scratch holds");
    void *ptr = nullptr;
    const int s = scratch_ptr(h, &ptr);
    if (s != NROCM_OK) return s;
    // as many right-hand sides at a time as the static tags hold (one, two or
    // a multiple of four)
    int cols = std::max(1, std::min(nrhs, NROCM_NOALLOC_MAX_N / std::max(n, 1)));
    cols = cols >= 4 ? cols & ~3 : cols == 3 ? 2 : cols;
    return solve<OP_LU>(h, h->stream, n, nrhs, lu, lda, ipiv, nullptr, b, ldb, info, mode == NROCM_EXACT, ptr, cols);
}
