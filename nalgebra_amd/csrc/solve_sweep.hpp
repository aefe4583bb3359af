// Triangular sweeps of the single-matrix solves (LU::solve_mut, Cholesky::
// solve_mut, QR::solve_mut) in nalgebra's per-element operation order, for one
// or several right-hand sides at a time.
//
// A sweep is a column sweep: with t = 0, 1, ... the sweep order (rows from the
// top, or from the bottom), element t receives fl(b_t - fl(x_u * M_tu)) for
// u = 0, 1, ..., t-1 in that order (solve.rs:106-182, 488-519), then x_t is its
// quotient by the diagonal.  Rows are taken in blocks of 64 in sweep order,
// one wavefront per block, lane = row: the wavefront applies the finished
// blocks one after the other, then solves its own 64 x 64 diagonal block.
//
// What bounds a sweep is the chain of blocks: hand-over of x, 64 dependent
// multiply-subtract steps of the next block, 64 steps of its diagonal block.
// So everything else is kept off it:
//   * the next block of M is in registers (two halves of 32 columns) before
//     x of that block is waited for;
//   * the diagonal block is loaded when the wavefront starts and moved to LDS
//     while the block before is being solved; its steps are a rolled loop
//     (unrolled, 64 steps are fetched from the L2 instruction by instruction
//     in a code path that runs once);
//   * a division by the diagonal is three instructions with the reciprocal
//     refined beforehand (exact_div.hpp); operands outside its range redo the
//     block with the compiler's division.
// CH right-hand sides share every load of M and interleave in the chain.
#pragma once
#include "access_rules.hpp"
#include "exact_div.hpp"

namespace nrocm_sweep {

constexpr int LB = 64;       // rows per block (one wavefront)
constexpr int HALF = LB / 2; // columns per register half of a block
constexpr int DSLOTS = 2;    // diagonal blocks staged in LDS at a time
// Right-hand sides per workgroup (1, 2 or 4) when every group of them takes
// `per_group` workgroups: as few as still leave each workgroup a CU of its own.
// One chain alone is the shortest (a step of the diagonal block is issue-bound
// from two on); sharing M only pays once the chip is full.
inline int rhs_per_group(int num_cus, int nrhs, long per_group)
{
    for (int ch = 1; ch < 4; ch *= 2)
        if ((long)nrocm_cdiv(nrhs, ch) * per_group <= num_cus) return ch;
    return 4;
}

constexpr int SWEEP_WAVES = 4;  // wavefronts per workgroup: one per SIMD, which leaves each 512 registers
constexpr long SPIN_LIMIT = 1L << 26;

// LU_FWD: unit lower, from the top.  CHOL_FWD: lower, from the top.  LU_BWD:
// upper, from the bottom.  QR_BWD: the same with |dg| as the diagonal.
// CHOL_BWD_FAST: U = L^T read from L's columns, from the bottom.
enum Kind { LU_FWD, CHOL_FWD, LU_BWD, QR_BWD, CHOL_BWD_FAST };

__host__ __device__ constexpr bool from_top(int kind) { return kind == LU_FWD || kind == CHOL_FWD; }

__device__ __forceinline__ double lane_value(double v, int src)
{
    const long long bits = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)bits, src);
    const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// acc[c] = fl(fl((-x[c]) * m) + acc[c]) (nalgebra's axpy with factor -x: the
// negation before the product and the product first in the sum, so that NaN
// results carry the reference's sign), or one fused multiply-add.  Two asm
// statements per element: the CH chains interleave.
template <bool EXACT, int CH>
__device__ __forceinline__ void step(double (&acc)[CH], const double (&x)[CH], double m)
{
    if constexpr (EXACT) {
        double t[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) asm("v_mul_f64 %0, -%1, %2" : "=v"(t[c]) : "v"(x[c]), "v"(m));
#pragma unroll
        for (int c = 0; c < CH; ++c) asm("v_add_f64 %0, %1, %0" : "+v"(acc[c]) : "v"(t[c]));
    } else {
#pragma unroll
        for (int c = 0; c < CH; ++c) asm("v_fma_f64 %0, -%1, %2, %0" : "+v"(acc[c]) : "v"(x[c]), "v"(m));
    }
}

// The same with x in scalar registers (a value broadcast by readlane).
template <bool EXACT, int CH>
__device__ __forceinline__ void step_uniform(double (&acc)[CH], const double (&x)[CH], double m)
{
    if constexpr (EXACT) {
        double t[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) asm("v_mul_f64 %0, -%1, %2" : "=v"(t[c]) : "s"(x[c]), "v"(m));
#pragma unroll
        for (int c = 0; c < CH; ++c) asm("v_add_f64 %0, %1, %0" : "+v"(acc[c]) : "v"(t[c]));
    } else {
#pragma unroll
        for (int c = 0; c < CH; ++c) asm("v_fma_f64 %0, -%1, %2, %0" : "+v"(acc[c]) : "s"(x[c]), "v"(m));
    }
}

// Columns u0 .. u0+HALF (sweep order) of matrix row r (the lane's row).  Steps
// past the matrix read its last column again; they are never used.
template <int KIND>
__device__ __forceinline__ void load_half(double (&h)[HALF], const double *__restrict__ M, int lda, int n, int r,
                                          int u0)
{
#pragma unroll
    for (int s = 0; s < HALF; ++s) {
        const int u = min(u0 + s, n - 1);
        if constexpr (KIND == CHOL_BWD_FAST) {
            h[s] = M[(size_t)r * lda + (n - 1 - u)];
        } else {
            const double *col = M + (size_t)(from_top(KIND) ? u : n - 1 - u) * lda;
            h[s] = col[r];
        }
    }
}

// HALF steps of a finished block, x at xs[s * CH + c] in LDS, read four steps
// ahead.
template <bool EXACT, int CH>
__device__ __forceinline__ void apply_half(double (&acc)[CH], const double (&h)[HALF], const double *xs)
{
    constexpr int G = 4;
    double xa[G][CH], xn[G][CH];
#pragma unroll
    for (int s = 0; s < G; ++s)
#pragma unroll
        for (int c = 0; c < CH; ++c) xa[s][c] = xs[s * CH + c];
#pragma unroll
    for (int g = 0; g < HALF; g += G) {
        if (g + G < HALF) {
#pragma unroll
            for (int s = 0; s < G; ++s)
#pragma unroll
                for (int c = 0; c < CH; ++c) xn[s][c] = xs[(g + G + s) * CH + c];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < G; ++s) step<EXACT, CH>(acc, xa[s], h[g + s]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < G; ++s)
#pragma unroll
            for (int c = 0; c < CH; ++c) xa[s][c] = xn[s][c];
    }
}

// The steps of a block's own diagonal block: D[i * LB + lane] = M_(lane, i).
// Every lane takes every step: lane i's value is captured at step i, and what
// it computes afterwards (like the rows past `rows`) is never read.  Masking
// those lanes off costs more than the step's arithmetic (a step took 65 clocks
// with an exec mask, 26 without; 8 clocks are one dependent FP64 addition).
template <bool EXACT, bool DIV, int CH>
__device__ __forceinline__ void diag_solve(double (&acc)[CH], const double *D, int rows, int lane, double d)
{
    constexpr int G = 4;
    double save[CH], res[CH], num[CH];
    double y = 0.0;
    if constexpr (DIV) y = nrocm_div::recip_refined(d);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        save[c] = acc[c];
        res[c] = 0.0;
        num[c] = 1.0;
    }
    double l[G], ln[G];
#pragma unroll
    for (int s = 0; s < G; ++s) l[s] = D[s * LB + lane];
#pragma unroll 1
    for (int i0 = 0; i0 < rows; i0 += G) {
#pragma unroll
        for (int s = 0; s < G; ++s) ln[s] = D[min(i0 + G + s, LB - 1) * LB + lane];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < G; ++s) {
            const int i = i0 + s;
            double q[CH], x[CH];
#pragma unroll
            for (int c = 0; c < CH; ++c) q[c] = DIV ? nrocm_div::div_with(acc[c], d, y) : acc[c];
#pragma unroll
            for (int c = 0; c < CH; ++c) x[c] = lane_value(q[c], i);
            if constexpr (DIV) {
#pragma unroll
                for (int c = 0; c < CH; ++c) num[c] = lane == i ? acc[c] : num[c];
            }
#pragma unroll
            for (int c = 0; c < CH; ++c) res[c] = lane == i ? q[c] : res[c];
            step_uniform<EXACT, CH>(acc, x, l[s]);
        }
#pragma unroll
        for (int s = 0; s < G; ++s) l[s] = ln[s];
    }
    if constexpr (DIV) {
        const bool dok = nrocm_div::div_den_ok(d);
        bool bad = false;
#pragma unroll
        for (int c = 0; c < CH; ++c) bad = bad || !(dok && nrocm_div::num_in_range(num[c]));
        if (__ballot(bad && lane < rows) != 0) {
            // some quotient's operands are outside the short division's range
#pragma unroll 1
            for (int i = 0; i < rows; ++i) {
                const double li = D[i * LB + lane];
                double x[CH];
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    const double q = save[c] / d;
                    x[c] = lane_value(q, i);
                    res[c] = lane == i ? q : res[c];
                }
                step_uniform<EXACT, CH>(save, x, li);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[c] = res[c];
}

// Progress of a workgroup's blocks: *done = blocks finished so far.  Every
// wavefront of a workgroup is resident, so the block waited for is in
// progress on another wavefront of it.
__device__ __forceinline__ void wait_done(const int *done, int need)
{
    while (__hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < need) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ void signal_done(int *done, int value, int lane)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    if (lane == 0) __hip_atomic_store(done, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// One row block k of a sweep by one wavefront: acc holds the right-hand sides
// of the lane's row and ends as its solved values; get(J) waits for finished
// block J and gives its x in LDS; D is LDS slot k % DSLOTS, whose last user,
// block k - DSLOTS, has finished once block k - 2 has been applied.
template <bool EXACT, int KIND, int CH, typename Get>
__device__ __forceinline__ void sweep_block(double (&acc)[CH], const double *__restrict__ M, int lda, int n, int k,
                                            double d, double *D, int lane, Get get)
{
    constexpr bool DIV = KIND != LU_FWD;
    const int tc = min(k * LB + lane, n - 1);
    const int r = from_top(KIND) ? tc : n - 1 - tc;
    double h0[HALF], h1[HALF], d0[HALF], d1[HALF];
    load_half<KIND>(d0, M, lda, n, r, k * LB);
    load_half<KIND>(d1, M, lda, n, r, k * LB + HALF);
    if (k > 0) {
        load_half<KIND>(h0, M, lda, n, r, 0);
        load_half<KIND>(h1, M, lda, n, r, HALF);
    }
    auto stash = [&]() {
#pragma unroll
        for (int s = 0; s < HALF; ++s) {
            D[s * LB + lane] = d0[s];
            D[(s + HALF) * LB + lane] = d1[s];
        }
    };
    if (k == 0) stash();
    for (int J = 0; J < k; ++J) {
        if (J == k - 1) stash();
        const double *xs = get(J);
        apply_half<EXACT, CH>(acc, h0, xs);
        if (J + 1 < k) load_half<KIND>(h0, M, lda, n, r, (J + 1) * LB);
        apply_half<EXACT, CH>(acc, h1, xs + HALF * CH);
        if (J + 1 < k) load_half<KIND>(h1, M, lda, n, r, (J + 1) * LB + HALF);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    diag_solve<EXACT, DIV, CH>(acc, D, min(LB, n - k * LB), lane, d);
}

// The diagonal element of row r.
template <int KIND>
__device__ __forceinline__ double diag_of(const double *__restrict__ M, int lda, const double *__restrict__ dg, int r)
{
    if constexpr (KIND == LU_FWD) return 1.0;
    else if constexpr (KIND == QR_BWD) return __builtin_fabs(dg[r]);
    else return M[(size_t)r * lda + r];
}

// ---------------------------------------------------------------- composed row permutation
// The swaps (k0 + i, ipiv[k0 + i]), i < cnt <= 64, applied in order, composed
// by one wavefront: afterwards position k0 + l holds what was at `in_who` of
// lane l, and position `out_pos` (lane l's pivot; -1 if it is one of k0..k0+63)
// what was at `out_who`.  Each lane follows its two positions back through the
// swaps, two compares and two selects per swap with no exchange between lanes
// (moving the contents by readlane instead took 230 clocks a swap, this 45).
// Several lanes may name the same outside position, with the same content.
// A pivot outside [0, n) is not applied and sets *bad.
struct BlockPlan {
    int in_who, out_pos, out_who;
};

__device__ __forceinline__ BlockPlan compose_block(const int *ipiv, int k0_, int cnt_, int n, int lane, bool *bad)
{
    const int k0 = __builtin_amdgcn_readfirstlane(k0_), cnt = __builtin_amdgcn_readfirstlane(cnt_);
    int p = lane < cnt ? ipiv[k0 + lane] : k0 + lane;
    const bool wrong = lane < cnt && (p < 0 || p >= n);
    if (wrong) p = k0 + lane;
    if (bad) *bad = __ballot(wrong) != 0;
    int x0 = k0 + lane, x1 = p;
    for (int i = cnt - 1; i >= 0; --i) {
        const int pi = __builtin_amdgcn_readlane(p, i), a = k0 + i;
        const int y0 = x0 == a ? pi : x0, y1 = x1 == a ? pi : x1;
        x0 = x0 == pi ? a : y0;
        x1 = x1 == pi ? a : y1;
    }
    return {x0, (unsigned)(p - k0) >= 64u ? p : -1, x1};
}

// perm[i] = the row that the swaps (i, ipiv[i]), i < n, applied in order bring
// to position i (PermutationSequence::permute_rows, permutation_sequence.rs:
// 97-104).  The wavefronts of a workgroup compose 64 swaps each, and the first
// one then applies those compositions one after the other to `perm` (LDS, or
// global memory with GLOBAL).  plan: NW * 192 ints of LDS.  Ends with a barrier.
template <int NW, bool GLOBAL>
__device__ __forceinline__ void compose_perm(const int *ipiv, int n, int *perm, int *plan, int *info)
{
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    for (int i = threadIdx.x; i < n; i += NW * 64) perm[i] = i;
    const int nblk = (n + 63) / 64;
    for (int b0 = 0; b0 < nblk; b0 += NW) {
        if (b0 + w < nblk) {
            const int k0 = (b0 + w) * 64;
            bool bad;
            const BlockPlan q = compose_block(ipiv, k0, min(64, n - k0), n, lane, &bad);
            int *dst = plan + w * 192;
            dst[lane] = q.in_who;
            dst[64 + lane] = q.out_pos;
            dst[128 + lane] = q.out_who;
            if (bad && info && lane == 0) *info = -2;
        }
        __syncthreads();
        if (w == 0) {
            int from = plan[lane], opos = plan[64 + lane], ofrom = plan[128 + lane];
            for (int q = 0; q < NW && b0 + q < nblk; ++q) {
                const int pos = (b0 + q) * 64 + lane;
                int a = 0, b = 0;
                if (pos < n) a = perm[from];
                if (opos >= 0) b = perm[ofrom];
                const int *nx = plan + min(q + 1, NW - 1) * 192;
                const int from1 = nx[lane], opos1 = nx[64 + lane], ofrom1 = nx[128 + lane];
                // every value is read before any is written, and the next
                // composition reads what this one wrote (LDS accesses of one
                // wavefront take effect in order)
                if constexpr (GLOBAL) __threadfence_block();
                else asm volatile("" ::: "memory");
                if (pos < n) perm[pos] = a;
                if (opos >= 0) perm[opos] = b;
                from = from1;
                opos = opos1;
                ofrom = ofrom1;
                if constexpr (GLOBAL) __threadfence_block();
                else asm volatile("" ::: "memory");
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- Cholesky's transposed solve
// L^T x = y in nalgebra's dot order (solve.rs:697-755 with the 8-accumulator
// dot of src/base/blas.rs:93-167): accumulator q of row i sums the products of
// elements q, q + 8, ... of L[i+1.., i] with x[i+1..] over the full chunks of
// eight in order, the sum is ((((0 + (a0 + a4)) + (a1 + a5)) + (a2 + a6)) +
// (a3 + a7)), the remaining elements are added one by one, and
// x_i = (y_i - sum) / L_ii.  Accumulator 0's first product needs x_{i+1}, so
// the rows are one dependent chain of about n^2 / 16 additions; that chain is
// what bounds this solve, and the order allows no shorter one.
//
// Wavefront 0 walks the chain for CH right-hand sides at once (lane q + 8c =
// accumulator q of right-hand side c).  The other NL wavefronts keep everything
// but the additions off it: they bring the columns of L in, each its part of
// every column DOT_AHEAD rows ahead, and leave the products in LDS.  Phase p is
// row i = n-1-p (a dot of p elements) and reads slot p % 3; the slot of phase
// p + 2 is written meanwhile, when x[i+1..] is known, so of that row only the
// elements of its two newest x stay unmultiplied: the chain wavefront holds
// those two in registers.  A step of the chain is then one LDS read and one
// addition instead of two reads, a product and an addition.  n = 1500: 9.6 ms
// per right-hand side (one wavefront reading L from memory) -> 1.3 ms for all
// of them.
// x (and y before it) is in LDS at xs[row * CH + c].  Every wavefront of the
// workgroup calls this.
template <int N>
__device__ __forceinline__ double row_shl(double v)
{
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)x, 0x100 + N, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), 0x100 + N, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// lane l takes lane l - 1's value (within rows of 16 lanes)
__device__ __forceinline__ double row_shr1(double v)
{
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)x, 0x111, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), 0x111, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

constexpr int DOT_SLOTS = 3;
constexpr int DOT_AHEAD = nrocm_rules::DOT_AHEAD;  // columns in flight per loading wavefront
constexpr int DOT_U = 16;     // chain steps per group, read one group ahead
constexpr int DOT_HEAD = 10;  // slot head: L_ii, its reciprocal, the eight tail products

// A slot, per right-hand side: the head, then the products in element order,
// whole groups of the chain (eight accumulators, DOT_U elements each),
// zero-padded.  The padding's zeros are exact: a sum that starts at +0 never
// becomes -0.  The chain reads up to two groups past the last one.
__host__ __device__ constexpr int dot_groups(int p) { return (p / 8 + DOT_U - 1) / DOT_U; }
__host__ __device__ constexpr int dot_stride(int n) { return DOT_HEAD + dot_groups(n) * 8 * DOT_U; }
__host__ __device__ constexpr int dot_doubles(int n, int ch) { return (DOT_SLOTS * dot_stride(n) + 3 * 8 * DOT_U) * ch; }
// Elements per lane of NL loading wavefronts.
__host__ __device__ constexpr int dot_lane_elements(int n, int nl) { return (dot_groups(n) * 8 * DOT_U + 64 * nl - 1) / (64 * nl); }

// NR >= dot_lane_elements(n, NL); slots: dot_doubles(n, CH) doubles.
template <int NR, int NL, int CH>
__device__ __forceinline__ void chol_dot_backward(const double *__restrict__ L, int lda, int n, double *xs,
                                                  double *slots)
{
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cstride = dot_stride(n), sstride = cstride * CH;
    constexpr int U = DOT_U;
    if (w > 0) {
        const int e0 = (w - 1) * 64 + lane;  // element e of row i: L[i+1+e, i] with x[i+1+e]
        struct Col {
            double v[NR], extra;  // extra: the tail element (wavefront 1) or L_ii (wavefront 2)
        };
        // no load is under a condition: with the same loads in every phase the
        // wait for the oldest column leaves the newer ones in flight
        auto fetch = [&](Col &r, int p) {
            const int i = n - 1 - min(p, n - 1);
            const double *col = L + (size_t)i * lda + i;
            const int last = n - 1 - i;
#pragma unroll
            for (int k = 0; k < NR; ++k) r.v[k] = col[min(1 + e0 + 64 * NL * k, last)];
            r.extra = col[w == 1 ? min(1 + (p & ~7) + (lane & 7), last) : 0];
        };
        auto put = [&](const Col &r, int p) {
            const int full = p & ~7, lim = p < n ? dot_groups(p) * 8 * U : 0;
            double *s = slots + (p % DOT_SLOTS) * sstride;
            const double *x = xs + nrocm_rules::dot_first_row(n, p) * CH;
            const int emax = nrocm_rules::dot_last_element(n, p);
            double f[NR][CH], ft[CH];
#pragma unroll
            for (int k = 0; k < NR; ++k)
#pragma unroll
                for (int c = 0; c < CH; ++c) f[k][c] = x[min(e0 + 64 * NL * k, emax) * CH + c];
            const int et = full + (lane & 7);
#pragma unroll
            for (int c = 0; c < CH; ++c) ft[c] = x[min(et, emax) * CH + c];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                const int e = e0 + 64 * NL * k;
                if ((w - 1) * 64 + 64 * NL * k < lim) {
#pragma unroll
                    for (int c = 0; c < CH; ++c) {
                        if (k == 0) f[k][c] = e < 2 ? 1.0 : f[k][c];
                        const double prod = r.v[k] * f[k][c];
                        s[c * cstride + DOT_HEAD + e] = e < full ? prod : 0.0;
                    }
                }
            }
            if (w == 1 && lane < 8 && p < n) {
#pragma unroll
                for (int c = 0; c < CH; ++c) s[c * cstride + 2 + lane] = et < p ? r.extra * (et < 2 ? 1.0 : ft[c]) : 0.0;
            }
            if (w == 2 && lane < CH && p < n) {
                s[lane * cstride] = r.extra;
                s[lane * cstride + 1] = nrocm_div::recip_refined(r.extra);
            }
        };
        Col reg[DOT_AHEAD];
        fetch(reg[0], 0);
        fetch(reg[1], 1);
        put(reg[0], 0);
        put(reg[1], 1);
#pragma unroll
        for (int j = 0; j < DOT_AHEAD; ++j) fetch(reg[j], j + 2);
        lds_barrier();
#pragma unroll 1
        for (int p = 0; p < n; p += DOT_AHEAD) {  // put() up to nrocm_rules::dot_last_phase
#pragma unroll
            for (int j = 0; j < DOT_AHEAD; ++j) {
                put(reg[j], p + j + 2);
                fetch(reg[j], p + j + 2 + DOT_AHEAD);
                lds_barrier();
            }
        }
        return;
    }
    const int q = lane & 7, c = min(lane >> 3, CH - 1);
    const bool owner = q == 0 && (lane >> 3) < CH;
    double va[U], vb[U];
    auto read = [&](double (&v)[U], const double *sp, int g) {
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = sp[8 * (g * U + u)];
        __builtin_amdgcn_sched_barrier(0);
    };
    double acc = 0.0;
    auto sum = [&](const double (&v)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) acc += v[u];
        __builtin_amdgcn_sched_barrier(0);
    };
    lds_barrier();
    double x1 = 0.0, x2 = 0.0;  // x_{i+1} (lane q = 0), x_{i+2} (lane q = 1)
    // what a row needs first is read while the row before ends
    double dii, rec, yi, tp;
    auto head = [&](int p) {
        const double *s = slots + (p % DOT_SLOTS) * sstride + c * cstride;
        dii = s[0];
        rec = s[1];
        tp = s[2 + q];
        yi = xs[(n - 1 - p) * CH + c];
        read(va, s + DOT_HEAD + q, 0);
    };
    head(0);
#pragma unroll 1
    for (int p = 0; p < n; ++p) {
        const int i = n - 1 - p;
        const double *sp = slots + (p % DOT_SLOTS) * sstride + c * cstride + DOT_HEAD + q;
        const int groups = dot_groups(p);
        const double xq = q == 0 ? x1 : q == 1 ? x2 : 1.0;
        va[0] = va[0] * xq;
        tp = p < 8 ? (q < p ? tp * xq : 0.0) : tp;  // p < 8: elements 0 and 1 are in the tail
        acc = 0.0;
        // groups past the last one are read, never added: conditional reads
        // would cost register copies
        read(vb, sp, 1);
        int g = 0;
#pragma unroll 1
        for (; g + 2 <= groups; g += 2) {
            sum(va);
            read(va, sp, g + 2);
            sum(vb);
            read(vb, sp, g + 3);
        }
        if (g < groups) sum(va);
        const double ydn = yi, den = dii, dre = rec, t0 = tp;
        if (p + 1 < n) head(p + 1);
        const double t1 = row_shl<1>(t0), t2 = row_shl<2>(t0), t3 = row_shl<3>(t0), t4 = row_shl<4>(t0),
                     t5 = row_shl<5>(t0), t6 = row_shl<6>(t0);
        const double pair = acc + row_shl<4>(acc);
        const double p1 = row_shl<1>(pair), p2 = row_shl<2>(pair), p3 = row_shl<3>(pair);
        double res = 0.0;
        res += pair;
        res += p1;
        res += p2;
        res += p3;
        res += t0;  // the tail, zero-padded
        res += t1;
        res += t2;
        res += t3;
        res += t4;
        res += t5;
        res += t6;
        const double num = ydn - res;
        const bool ok = nrocm_div::div_den_ok(den) && nrocm_div::num_in_range(num);
        double xnew = nrocm_div::div_with(num, den, dre);
        if (__ballot(owner && !ok) != 0) xnew = ok ? xnew : num / den;
        if (owner) xs[i * CH + c] = xnew;
        x2 = row_shr1(x1);
        x1 = xnew;
        lds_barrier();
    }
    for (int p = n; p % DOT_AHEAD != 0; ++p) lds_barrier();  // the loaders' last round
}

}  // namespace nrocm_sweep
