// Adjoint of the batched Cholesky solve X = A^{-1} B (nrocm_dpotrs_backward_batched):
//   Lambda = (L L^T)^{-1} dX in the arithmetic of Cholesky::solve_mut
//   (src/linalg/cholesky.rs:122-129, solve.rs:500-519,697-755: L y = dX by
//   columns, L^T z = y by dots in dotx's order),
//   dB = Lambda, dA = -1/2 (Lambda X^T + X Lambda^T) summed over right-hand sides
//   in order.
//
// Bound by the chains of the two substitutions, a division and a broadcast or a
// dot per row: up to eight members share a wavefront, eight lanes each, no step needs
// a barrier, and members of all sizes run in one launch, the largest first.  Before,
// a member had 16 to 64 lanes, a step one to three barriers and each range of
// sizes its own launch: 4096 members of n = 32, one right-hand side, 90 -> 31 us,
// where reading L and X and writing dA take 10.
#include "adjoint_steps.hpp"
#include "internal_launch.hpp"

namespace {

using namespace nrocm_adjoint;

__device__ const double kZeroCell[1] = {0.0};

// KM: blocks of 8 rows that a lane can hold; CH: right-hand sides at a time.
template <int KM, int CH>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void potrs_backward_kernel(
    const int *__restrict__ order, int count, int per, const int *__restrict__ nsz,
    const double *const *__restrict__ Lptr,
    const double *const *__restrict__ Xptr, const double *const *__restrict__ dXptr,
    double *const *__restrict__ dAptr, double *const *__restrict__ dBptr, int nrhs)
{
    constexpr int NB = 8 * KM, LD = NB + 1;
    __shared__ double v[8][CH][LD];   // a chunk's values by row: dX, y, Lambda
    __shared__ double xs[8][CH][LD];  // the chunk of X
    const int lane = threadIdx.x;
    const int g = lane >> 3, c = lane & 7;
    const int item = (int)blockIdx.x * per + g;
    const bool valid = g < per && item < count;
    const int jm = valid ? order[item] : 0;
    const int n = valid ? nsz[jm] : 0;
    int most = n;
#pragma unroll
    for (int off = 8; off < 64; off *= 2) most = max(most, __shfl_xor(most, off));
    const int blocks = __builtin_amdgcn_readfirstlane((most + 7) >> 3);
    if (blocks == 0) return;
    // a group without a member, or with an empty one, walks a 1 x 1 zero
    Matrix L = (Matrix)(n > 0 ? Lptr[jm] : kZeroCell);
    const int nm = max(n, 1);
    const unsigned long long dA = n > 0 ? (unsigned long long)dAptr[jm] : 0;
    // a chunk reads its dX and X before it writes dB, and L before dA, so that
    // outputs may take the place of inputs
    for (int c0 = 0; c0 == 0 || c0 < nrhs; c0 += CH) {
        const int qn = min(nrhs - c0, CH);
        asm volatile("" : "+v"(L));  // no addresses kept from chunk to chunk
        const double *const dX = n > 0 && qn > 0 ? dXptr[jm] : nullptr;
        const double *const X = n > 0 && qn > 0 ? Xptr[jm] : nullptr;
#pragma unroll
        for (int k = 0; k < KM; ++k) {
            const int i = 8 * k + c;
#pragma unroll
            for (int q = 0; q < CH; ++q) {
                const bool in = i < n && q < qn;
                v[g][q][i] = in ? dX[i + (size_t)(c0 + q) * n] : 0.0;
                xs[g][q][i] = in ? X[i + (size_t)(c0 + q) * n] : 0.0;
            }
        }
        __syncthreads();
        substitute<FORWARD, KM, CH, LD>(L, nm, blocks, c, v[g]);
        __syncthreads();
        substitute<LOWER, KM, CH, LD>(L, nm, blocks, c, v[g]);
        __syncthreads();
        double *const dB = n > 0 && qn > 0 ? dBptr[jm] : nullptr;
        for (int i = c; i < n; i += 8)
#pragma unroll
            for (int q = 0; q < CH; ++q)
                if (q < qn) dB[i + (size_t)(c0 + q) * n] = v[g][q][i];
        // dA[r, k] = -1/2 (Lambda_r X_k + X_r Lambda_k), the whole wavefront on one
        // member at a time, along its columns
#pragma unroll 1
        for (int m = 0; m < per; ++m) {
            const int mn = __builtin_amdgcn_readlane(n, 8 * m);
            if (mn == 0) continue;
            double *const D = (double *)((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)dA, 8 * m) |
                                         (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(dA >> 32), 8 * m) << 32);
            const int dk = 64 / mn, dr = 64 - dk * mn;
            int k = lane / mn, r = lane - k * mn;
#pragma unroll 2
            for (int e = lane; e < mn * mn; e += 64) {
                double s = c0 > 0 ? D[e] : 0.0;
#pragma unroll
                for (int q = 0; q < CH; ++q) {
                    if (q < qn) {
                        const double p = v[m][q][r] * xs[m][q][k];
                        const double t = xs[m][q][r] * v[m][q][k];
                        const double d = -0.5 * (p + t);
                        s = (c0 == 0 && q == 0) ? d : s + d;
                    }
                }
                D[e] = s;  // no right-hand sides: zero
                r += dr;
                k += dk;
                if (r >= mn) {
                    r -= mn;
                    ++k;
                }
            }
        }
        __syncthreads();
    }
}

template <int KM>
void launch(hipStream_t st, int num_cus, const int *order, int count, const int *nsz, const double *const *L,
            const double *const *X, const double *const *dX, double *const *dA, double *const *dB, int nrhs)
{
    const auto kernel = nrhs > 2 ? potrs_backward_kernel<KM, 4>
                      : nrhs > 1 ? potrs_backward_kernel<KM, 2> : potrs_backward_kernel<KM, 1>;
    const int per = members_per_wave(num_cus, count);
    hipLaunchKernelGGL(kernel, dim3((unsigned)nrocm_cdiv(count, per)), dim3(64), 0, st, order, count, per, nsz, L, X, dX,
                       dA, dB, nrhs);
}

}  // namespace

extern "C" int nrocm_dpotrs_backward_batched(nrocm_handle h, nrocm_batch bt, const double *const *L,
                                             const double *const *X, const double *const *dX, double *const *dA,
                                             double *const *dB)
{
    if (!h) return -1;
    if (!bt || bt->handle != h) return -2;
    if (bt->count > 0 && (!L)) return -3;
    if (bt->count > 0 && (!X)) return -4;
    if (bt->count > 0 && (!dX)) return -5;
    if (bt->count > 0 && (!dA)) return -6;
    if (bt->count > 0 && (!dB)) return -7;
    if (bt->count == 0) return NROCM_OK;
    if (bt->max_n > 64)
        return nrocm_fail(h, NROCM_ERR_UNSUPPORTED, "batched Cholesky adjoint supports n <= 64");
    // `order` holds the members by decreasing size
    if (bt->max_n <= 32)
        launch<4>(h->stream, h->num_cus, bt->order_dev, bt->count, bt->n_dev, L, X, dX, dA, dB, bt->nrhs);
    else
        launch<8>(h->stream, h->num_cus, bt->order_dev, bt->count, bt->n_dev, L, X, dX, dA, dB, bt->nrhs);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}
