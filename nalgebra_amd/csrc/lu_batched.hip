// Batched (uneven sizes, n <= 64) LU with partial pivoting and solve:
// LU::new (src/linalg/lu.rs:93-122) then LU::solve_mut (lu.rs:242-260) per
// member, one launch per size class of the batch (padded sizes 8, 16, ..., 64).
//
// Layout: a group of G lanes serves one matrix (64 / G matrices per
// wavefront); lane r holds row r of its matrix in registers for the whole
// kernel.  Rows never move: each lane carries the current position of its
// row, and a swap of positions i and piv exchanges the two lanes' positions,
// which is nalgebra's full-row swap (lu.rs:114 swaps the left part too,
// gauss_step_swap :362-389 the rest).  Step i:
//   1. pivot: the first position >= i holding the strictly largest |a_i|
//      (icamax, src/base/min_max.rs:221-241; a NaN at position i wins, other
//      NaNs never do), reduced over the group;
//   2. a zero pivot skips the step (lu.rs:107-110);
//   3. the pivot row is broadcast through LDS; rows below take
//      l = fl(a_i * fl(1 / d)) and a_k = fl(a_k - fl(u_k * l)) for k > i, the
//      same unfused per-element sequence as gauss_step (NROCM_EXACT), or one
//      fused multiply-add (NROCM_FAST).
// The solve keeps the rows where they are: the right-hand side value of the
// row at position p is b_r of its original row r (PermutationSequence::
// permute_rows applies the same swaps), forward substitution with the unit
// lower factor (solve.rs:106-133) and backward substitution with U
// (solve.rs:137-182) broadcast the solved value of position i from the lane
// holding that position, and x is stored at the row's final position.
#include "adjoint_steps.hpp"
#include "internal_launch.hpp"

#include <algorithm>

using namespace nrocm_adjoint;

namespace {

constexpr int CH = 4;  // right-hand sides held in registers at a time

template <int NB>
constexpr int group_for() { return NB <= 8 ? 8 : NB <= 16 ? 16 : NB <= 32 ? 32 : 64; }

template <bool EXACT>
__device__ __forceinline__ double sub_prod(double acc, double x, double y)
{
    // nalgebra's axpy with factor -x: fl(fl((-x) * y) + acc).  The negation
    // is applied to x before the product, as there, so that a NaN coming from
    // y keeps its sign.  One asm block keeps the product next to its addition
    // (as two IR operations the scheduler hoists every product of a step and
    // spills the row array), and it updates acc in place: with a separate
    // output the elimination of a step writes a second copy of the row and
    // moves it back at the end of the divergent region.
    if constexpr (EXACT) {
        double t;
        asm("v_mul_f64 %1, -%2, %3\n\tv_add_f64 %0, %1, %0" : "+v"(acc), "=&v"(t) : "v"(x), "v"(y));
    } else {
        asm("v_fma_f64 %0, -%1, %2, %0" : "+v"(acc) : "v"(x), "v"(y));
    }
    return acc;
}

// (value, position) under icamax's rule: larger value, then lower position.
__device__ __forceinline__ bool beats(double av, int ap, double bv, int bp)
{
    return av > bv || (av == bv && ap < bp);
}

// One DPP step of the pivot scan: (v, pos) against the pair the pattern CTRL
// brings in (rows outside ROWMASK, and lanes without a source, see the
// non-candidate pair (-1, INT_MAX), which never wins).
template <int CTRL, int ROWMASK>
__device__ __forceinline__ void pivot_dpp_step(double &v, int &pos)
{
    const long long x = __double_as_longlong(v);
    const long long o = __double_as_longlong(-1.0);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)x, CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(x >> 32), CTRL, ROWMASK, 0xf, false);
    const double ov = __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
    const int op = __builtin_amdgcn_update_dpp(0x7fffffff, pos, CTRL, ROWMASK, 0xf, false);
    if (beats(ov, op, v, pos)) {
        v = ov;
        pos = op;
    }
}

// Group-wide pivot: every lane of the group ends with the winner's position.
// Groups of 16 or more lanes reduce by DPP scans (the rule is a total order,
// so the winner does not depend on the combination order): row_shr 1, 2, 4, 8
// leave each 16-lane row's winner in its lane 15; row_bcast 15 into rows 1
// and 3 only joins the rows of each 32-lane half, and row_bcast 31 the two
// halves.  Groups of 8 use a butterfly of lane shuffles (row_shr 4 would
// cross their boundary).
template <int G>
__device__ __forceinline__ void group_argmax(double &v, int &pos)
{
    if constexpr (G >= 16) {
        pivot_dpp_step<0x111, 0xf>(v, pos);
        pivot_dpp_step<0x112, 0xf>(v, pos);
        pivot_dpp_step<0x114, 0xf>(v, pos);
        pivot_dpp_step<0x118, 0xf>(v, pos);
        if constexpr (G >= 32) pivot_dpp_step<0x142, 0xa>(v, pos);
        if constexpr (G == 64) pivot_dpp_step<0x143, 0xc>(v, pos);
        const int lane = threadIdx.x & 63;
        if constexpr (G == 64) {
            pos = __builtin_amdgcn_readlane(pos, 63);
        } else if constexpr (G == 32) {
            const int p0 = __builtin_amdgcn_readlane(pos, 31), p1 = __builtin_amdgcn_readlane(pos, 63);
            pos = lane < 32 ? p0 : p1;
        } else {
            pos = __shfl(pos, lane | 15);
        }
    } else {
#pragma unroll
        for (int off = G / 2; off >= 1; off >>= 1) {
            const double ov = __shfl_xor(v, off, G);
            const int op = __shfl_xor(pos, off, G);
            if (beats(ov, op, v, pos)) {
                v = ov;
                pos = op;
            }
        }
    }
}

__device__ const double kZeroCellLU[1] = {0.0};

// v of lane src (wavefront-uniform) in every lane.
__device__ __forceinline__ double lane_value(double v, int src)
{
    const long long bits = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)bits, src);
    const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int NB, int G, bool EXACT>
__global__ __launch_bounds__(64) void getrf_getrs_batched_kernel(
    const int *__restrict__ order, int begin, int end, const int *__restrict__ nsz, double *const *__restrict__ Aptr,
    int *const *__restrict__ Pptr, double *const *__restrict__ Bptr, int nrhs, int *__restrict__ info)
{
    constexpr int MPW = 64 / G;
    __shared__ __align__(16) double rowbuf[MPW][NB];
    __shared__ double bbuf[MPW][CH];
    __shared__ int where[MPW][NB];  // final position -> lane within the group
    const int lane = threadIdx.x;
    const int g = lane / G, r = lane % G;
    const int item = begin + (int)blockIdx.x * MPW + g;
    const bool valid = item < end;
    const int jm = valid ? order[item] : 0;
    const int n = valid ? nsz[jm] : 0;
    double *const A = valid ? Aptr[jm] : nullptr;
    int *const P = (valid && Pptr) ? Pptr[jm] : nullptr;
    const bool row_ok = r < n;

    double a[NB];
    {
        const double *row = row_ok ? A + r : kZeroCellLU;
        const size_t step = row_ok ? (size_t)n : 0;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const double *src = (c < n) ? row + (size_t)c * step : kZeroCellLU;
            a[c] = *src;
        }
    }
    int pos = r;
    int zmax = 0;  // 1 + the largest step with a zero pivot (U_ii == 0)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const bool live = i < n;  // this group still has step i
        // 1. pivot search over the positions >= i
        double v = __builtin_fabs(a[i]);
        v = (v != v) ? ((pos == i) ? __builtin_inf() : -1.0) : v;
        const bool cand = live && row_ok && pos >= i;
        v = cand ? v : -1.0;
        int bp = cand ? pos : 0x7fffffff;
        group_argmax<G>(v, bp);
        const bool is_piv = cand && pos == bp;
        // 3. the pivot row (its entries from column i on) through LDS
        if (is_piv) {
#pragma unroll
            for (int k = i; k < NB; ++k) rowbuf[g][k] = a[k];
        }
        lds_barrier();
        const double d = live ? rowbuf[g][i] : 1.0;
        if (live && r == 0 && P) P[i] = (d == 0.0) ? i : bp;
        if (live && d == 0.0) zmax = i + 1;  // 2. zero pivot: nothing moves
        // zmax settled now: left to the compiler, its update sinks below the
        // loop and keeps every step's pivot value live to the end
        asm volatile("" : "+v"(zmax));
        if (live && d != 0.0) {
            if (pos == i) pos = bp;
            else if (is_piv) pos = i;
            if (pos > i && row_ok) {
                const double inv = 1.0 / d;
                const double l = a[i] * inv;
                a[i] = l;
#pragma unroll
                for (int k = i + 1; k < NB; ++k) a[k] = sub_prod<EXACT>(a[k], rowbuf[g][k], l);
            }
        }
        lds_barrier();
    }
    // the factors, each row at its final position
    if (row_ok) {
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (c < n) A[pos + (size_t)c * n] = a[c];
    }
    if (valid && r == 0) info[jm] = zmax;
    if (nrhs <= 0 || Bptr == nullptr) return;

    // ---- solve: skipped for a singular U (solve_mut returns false), whose
    // right-hand sides are left unchanged
    double *const B = valid ? Bptr[jm] : nullptr;
    const bool solve = valid && zmax == 0;
    if (row_ok) where[g][pos] = r;
    __syncthreads();
    for (int c0 = 0; c0 < nrhs; c0 += CH) {
        double b[CH];
#pragma unroll
        for (int q = 0; q < CH; ++q) b[q] = (solve && row_ok && c0 + q < nrhs) ? B[r + (size_t)(c0 + q) * n] : 0.0;
        // forward: unit lower, per element the steps i = 0, 1, ... in order.
        // A whole-wavefront group reads position i's values straight from the
        // lane holding it (a wavefront-uniform lane); smaller groups pass them
        // through LDS.
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const bool live = i + 1 < n;
            double bv[CH];
            if constexpr (G == 64) {
                const int src = __builtin_amdgcn_readfirstlane(live ? where[0][i] : 0);
#pragma unroll
                for (int q = 0; q < CH; ++q) bv[q] = lane_value(b[q], src);
            } else {
                if (live && where[g][i] == r) {
#pragma unroll
                    for (int q = 0; q < CH; ++q) bbuf[g][q] = b[q];
                }
                lds_barrier();
#pragma unroll
                for (int q = 0; q < CH; ++q) bv[q] = bbuf[g][q];
            }
            if (live && pos > i && row_ok) {
#pragma unroll
                for (int q = 0; q < CH; ++q) b[q] = sub_prod<EXACT>(b[q], bv[q], a[i]);
            }
            if constexpr (G != 64) lds_barrier();
            // one step at a time: interleaved across the unrolled steps, the
            // broadcasts and index reads run out of registers
            if constexpr (G == 64) __builtin_amdgcn_sched_barrier(0);
        }
        // backward: x_i = b_i / U_ii, then the positions above it
#pragma unroll
        for (int i = NB - 1; i >= 0; --i) {
            const bool live = i < n;
            double bv[CH];
            if constexpr (G == 64) {
                const int src = __builtin_amdgcn_readfirstlane(live ? where[0][i] : 0);
                if (live && src == r) {
#pragma unroll
                    for (int q = 0; q < CH; ++q) b[q] = b[q] / a[i];
                }
#pragma unroll
                for (int q = 0; q < CH; ++q) bv[q] = lane_value(b[q], src);
            } else {
                if (live && where[g][i] == r) {
#pragma unroll
                    for (int q = 0; q < CH; ++q) {
                        b[q] = b[q] / a[i];
                        bbuf[g][q] = b[q];
                    }
                }
                lds_barrier();
#pragma unroll
                for (int q = 0; q < CH; ++q) bv[q] = bbuf[g][q];
            }
            if (live && pos < i && row_ok) {
#pragma unroll
                for (int q = 0; q < CH; ++q) b[q] = sub_prod<EXACT>(b[q], bv[q], a[i]);
            }
            if constexpr (G != 64) lds_barrier();
            // one step at a time: interleaved across the unrolled steps, the
            // broadcasts and index reads run out of registers
            if constexpr (G == 64) __builtin_amdgcn_sched_barrier(0);
        }
        if (solve && row_ok) {
#pragma unroll
            for (int q = 0; q < CH; ++q)
                if (c0 + q < nrhs) B[pos + (size_t)(c0 + q) * n] = b[q];
        }
    }
}

// Adjoint of X = A^{-1} B from LU::new's packed factors and pivots:
//   U^T y = g  (tr_solve_upper_triangular, solve.rs:255-276,411-440),
//   L^T z = y  (tr_solve_lower_triangular on the unit L, solve.rs:232-253,379-409),
//   Lambda = P^T z (inv_permute_rows, permutation_sequence.rs:108-116),
//   dB = Lambda, dA = -Lambda X^T (products summed over right-hand sides in
//   order), each dot in dotx's order.
//
// Bound by the chain of dots, one per row: products, up to 8 additions, the
// joining of the accumulators and the tail, about 300 cycles a step.  One
// member's chain uses few lanes, so up to eight members share a wavefront (eight lanes
// each, the accumulators of a dot side by side), nothing of a step crosses a
// group, and no step needs a barrier; members of the whole range of sizes run in
// one launch, the largest first.  Before, a member had 16 to 64 lanes, a dot
// three barriers and each range of sizes its own launch: 16384 members of
// n = 4..64, 2 right-hand sides, 2250 -> 177 us, where reading the factors and
// writing dA take 85.
// KM: blocks of 8 rows that a lane can hold; CH: right-hand sides at a time.
template <int KM, int CH>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void getrs_backward_batched_kernel(
    const int *__restrict__ order, int count, int per, const int *__restrict__ nsz,
    const double *const *__restrict__ LUptr, const int *const *__restrict__ Pptr, const double *const *__restrict__ Xptr,
    const double *const *__restrict__ dXptr, double *const *__restrict__ dAptr, double *const *__restrict__ dBptr,
    int nrhs)
{
    constexpr int NB = 8 * KM, LD = NB + 1;
    __shared__ double v[8][CH][LD];   // a chunk's values by row: g, y, z, Lambda
    __shared__ double xs[8][CH][LD];  // the chunk of X
    __shared__ int swap[8][NB];
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
    const Matrix LU = (Matrix)(n > 0 ? LUptr[jm] : kZeroCellLU);
    const int nm = max(n, 1);
    if (n > 0) {
        const int *const P = Pptr[jm];
        for (int i = c; i < n; i += 8) swap[g][i] = P[i];
    }
    for (int c0 = 0; c0 < nrhs; c0 += CH) {
        const double *const dX = n > 0 ? dXptr[jm] : nullptr;
        for (int i = c; i < n; i += 8)
#pragma unroll
            for (int q = 0; q < CH; ++q) v[g][q][i] = c0 + q < nrhs ? dX[i + (size_t)(c0 + q) * n] : 0.0;
        __syncthreads();
        substitute<UPPER, KM, CH, LD>(LU, nm, blocks, c, v[g]);
        __syncthreads();
        substitute<UNIT_LOWER, KM, CH, LD>(LU, nm, blocks, c, v[g]);
        __syncthreads();
        // the swaps (i, ipiv[i]) in reverse order, a lane per right-hand side
        if (c < CH) {
            double *const col = v[g][c];
            for (int i = n - 1; i >= 0; --i) {
                const int pv = swap[g][i];
                const double t = col[i], o = col[pv];
                col[i] = o;
                col[pv] = t;
            }
        }
        __syncthreads();
        double *const dB = n > 0 ? dBptr[jm] : nullptr;
        for (int i = c; i < n; i += 8)
#pragma unroll
            for (int q = 0; q < CH; ++q)
                if (c0 + q < nrhs) dB[i + (size_t)(c0 + q) * n] = v[g][q][i];
        __syncthreads();
    }
    // dA[r, k] = -(sum over right-hand sides of fl(Lambda_r * X_k)), the whole
    // wavefront on one member at a time, along its columns
    for (int c0 = 0; c0 == 0 || c0 < nrhs; c0 += CH) {
        const int qn = min(nrhs - c0, CH);
        const double *const X = n > 0 && qn > 0 ? Xptr[jm] : nullptr;
        const double *const dB = n > 0 && qn > 0 ? dBptr[jm] : nullptr;
        for (int i = c; i < n; i += 8)
#pragma unroll
            for (int q = 0; q < CH; ++q) {
                if (q >= qn) break;
                xs[g][q][i] = X[i + (size_t)(c0 + q) * n];
                if (nrhs > CH) v[g][q][i] = dB[i + (size_t)(c0 + q) * n];
            }
        __syncthreads();
        const unsigned long long dA = n > 0 ? (unsigned long long)dAptr[jm] : 0;
        for (int m = 0; m < per; ++m) {
            const int mn = __builtin_amdgcn_readlane(n, 8 * m);
            if (mn == 0) continue;
            double *const D = (double *)((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)dA, 8 * m) |
                                         (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(dA >> 32), 8 * m) << 32);
            const int dk = 64 / mn, dr = 64 - dk * mn;
            int k = lane / mn, r = lane - k * mn;
            for (int e = lane; e < mn * mn; e += 64) {
                double s = c0 > 0 ? -D[e] : 0.0;
#pragma unroll
                for (int q = 0; q < CH; ++q) {
                    if (q < qn) {
                        const double pr = v[m][q][r] * xs[m][q][k];
                        s = (c0 == 0 && q == 0) ? pr : s + pr;
                    }
                }
                D[e] = qn > 0 ? -s : 0.0;  // no right-hand sides: zero
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

// One launch for the whole batch: `order` holds the members by decreasing size.
template <int KM>
void launch_bwd(hipStream_t st, int num_cus, const int *order, int count, const int *nsz, const double *const *LU,
                const int *const *P, const double *const *X, const double *const *dX, double *const *dA,
                double *const *dB, int nrhs)
{
    const int per = members_per_wave(num_cus, count);
    const dim3 grid(nrocm_cdiv(count, per));
    if (nrhs > 1)
        hipLaunchKernelGGL((getrs_backward_batched_kernel<KM, 2>), grid, dim3(64), 0, st, order, count, per, nsz, LU, P,
                           X, dX, dA, dB, nrhs);
    else
        hipLaunchKernelGGL((getrs_backward_batched_kernel<KM, 1>), grid, dim3(64), 0, st, order, count, per, nsz, LU, P,
                           X, dX, dA, dB, nrhs);
}

template <int NB>
int launch_nb(bool exact, hipStream_t st, const int *order, int begin, int end, const int *nsz, double *const *A,
              int *const *P, double *const *B, int nrhs, int *info)
{
    constexpr int G = group_for<NB>();
    constexpr int MPW = 64 / G;
    const unsigned grid = (unsigned)((end - begin + MPW - 1) / MPW);
    if (grid == 0) return 0;
    if (exact)
        hipLaunchKernelGGL((getrf_getrs_batched_kernel<NB, G, true>), dim3(grid), dim3(64), 0, st, order, begin, end,
                           nsz, A, P, B, nrhs, info);
    else
        hipLaunchKernelGGL((getrf_getrs_batched_kernel<NB, G, false>), dim3(grid), dim3(64), 0, st, order, begin,
                           end, nsz, A, P, B, nrhs, info);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

using Launch = int (*)(bool, hipStream_t, const int *, int, int, const int *, double *const *, int *const *,
                       double *const *, int, int *);
const Launch kLaunch[8] = {launch_nb<8>, launch_nb<16>, launch_nb<24>, launch_nb<32>,
                           launch_nb<40>, launch_nb<48>, launch_nb<56>, launch_nb<64>};

}  // namespace

extern "C" int nrocm_dgetrf_getrs_batched(nrocm_handle h, nrocm_batch bt, double *const *a, int *const *ipiv,
                                          double *const *b, int *info, int mode)
{
    if (!h) return -1;
    if (!bt || bt->handle != h) return -2;
    if (bt->count > 0 && !a) return -3;
    if (bt->count > 0 && bt->nrhs > 0 && !b) return -5;
    if (bt->count > 0 && !info) return -6;
    if (mode != NROCM_EXACT && mode != NROCM_FAST) return -7;
    if (bt->count == 0) return NROCM_OK;
    if (bt->max_n > 64) return nrocm_fail(h, NROCM_ERR_UNSUPPORTED, "batched LU supports n <= 64");
    // the bins are independent: dealt round-robin (sizes in decreasing order)
    // to the stream and one auxiliary stream, whose kernels then run side by side
    int s = nrocm_aux_init(h);
    if (s == NROCM_OK) s = nrocm_fork_on(h, h->stream, 1);
    if (s != NROCM_OK) return s;
    int k = 0;
    for (const auto &bin : bt->bins) {
        if (bin.end <= bin.begin) continue;
        hipStream_t bs = (k++ & 1) ? h->aux[0] : h->stream;
        if (kLaunch[bin.kernel](mode == NROCM_EXACT, bs, bt->order_dev, bin.begin, bin.end, bt->n_dev, a, ipiv,
                                bt->nrhs > 0 ? b : nullptr, bt->nrhs, info))
            NROCM_CHECK_LAUNCH(h);
    }
    return nrocm_join_on(h, h->stream, 1);
}

extern "C" int nrocm_dgetrs_backward_batched(nrocm_handle h, nrocm_batch bt, const double *const *lu,
                                             const int *const *ipiv, const double *const *x,
                                             const double *const *dx, double *const *da, double *const *db)
{
    if (!h) return -1;
    if (!bt || bt->handle != h) return -2;
    if (bt->count > 0 && !lu) return -3;
    if (bt->count > 0 && !ipiv) return -4;
    if (bt->count > 0 && bt->nrhs > 0 && !x) return -5;
    if (bt->count > 0 && bt->nrhs > 0 && !dx) return -6;
    if (bt->count > 0 && !da) return -7;
    if (bt->count > 0 && bt->nrhs > 0 && !db) return -8;
    if (bt->count == 0) return NROCM_OK;
    if (bt->max_n > 64) return nrocm_fail(h, NROCM_ERR_UNSUPPORTED, "batched LU adjoint supports n <= 64");
    // up to 32 rows a lane holds half as many values, and the dots have half the terms
    if (bt->max_n <= 32)
        launch_bwd<4>(h->stream, h->num_cus, bt->order_dev, bt->count, bt->n_dev, lu, ipiv, x, dx, da, db, bt->nrhs);
    else
        launch_bwd<8>(h->stream, h->num_cus, bt->order_dev, bt->count, bt->n_dev, lu, ipiv, x, dx, da, db, bt->nrhs);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}
