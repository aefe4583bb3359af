// Householder QR.
//
// 1. nalgebra's representation, exact arithmetic (nrocm_dgeqrf / sgeqrf,
//    nrocm_dqr_qtmul, nrocm_dqr_qmul): every column takes the reflectors in
//    order exactly as QR::new (src/linalg/qr.rs:55-76) ->
//    householder::clear_column_unchecked (householder.rs:61-85) ->
//    reflection_axis_mut (householder.rs:19-53) -> reflect_with_sign
//    (src/geometry/reflection.rs:70-83).  Every dot product uses dotx's eight
//    accumulators (src/base/blas.rs:93-167): independent chains, one lane each.
// 2. Batched tall least squares (nrocm_sgels_batched): qr_batched.inc.
#include "gemm_kernels.hpp"
#include "internal_launch.hpp"
#include "solve_sweep.hpp"

#include <algorithm>
#include <utility>
#include <cmath>

namespace {

// Unfused y = fl(fl(fl(a*x)*c) + fl(b*y)) (blas_uninit.rs:46-52).
template <typename T>
__device__ __forceinline__ T axcpy1(T a, T x, T c, T b, T y)
{
    T p = a * x;
    p = p * c;
    T q = b * y;
    return p + q;
}

// dotx over len elements of x (stride 1) and y (stride 1) using the 8 threads
// t0..t0+7 of the calling group; the result is returned to thread t0 only.
// `part` is 8 slots of shared scratch owned by the group.
template <typename T>
__device__ __forceinline__ T group_dot8(const T *x, const T *y, int len, int sub, T *part)
{
    const int full = len & ~7;
    T acc = 0;
    for (int e = sub; e < full; e += 8) acc += x[e] * y[e];
    part[sub] = acc;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    T res = 0;
    if (sub == 0) {
        res += part[0] + part[4];
        res += part[1] + part[5];
        res += part[2] + part[6];
        res += part[3] + part[7];
        for (int e = full; e < len; ++e) res += x[e] * y[e];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return res;
}

template <typename T>
__device__ __forceinline__ T signum_rs(T x)
{
    // Rust f64::signum: NaN -> NaN, +-0 -> +-1
    if (x != x) return x;
    return signbit(x) ? T(-1) : T(1);
}

// Reflects columns [c0, c1) of C (rows i.., ldc) through axis x (len rows)
// with the given sign; one 8-thread group per column.
template <typename T>
__device__ void reflect_cols(const T *x, int len, T *C, int ldc, int c0, int c1, T sign, T *scratch)
{
    const int grp = threadIdx.x >> 3, sub = threadIdx.x & 7, ngrp = blockDim.x >> 3;
    T *part = scratch + grp * 8;
    const T m_two = sign * T(-2);
    // uniform trip count so every group reaches the wave barriers together
    for (int cb = c0; cb < c1; cb += ngrp) {
        const int c = cb + grp;
        T *col = C + (size_t)(c < c1 ? c : c0) * ldc;
        T d = group_dot8<T>(x, col, len, sub, part);
        if (sub == 0) part[0] = d;  // broadcast within the group
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const T factor = (part[0] - T(0)) * m_two;
        __builtin_amdgcn_wave_barrier();
        if (c < c1)
            for (int r = sub; r < len; r += 8) col[r] = axcpy1<T>(factor, x[r], T(1), sign, col[r]);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void geqrf_exact_kernel(T *A, int m, int n, int lda, T *diag)
{
    __shared__ T scratch[256];
    __shared__ T sh[4];
    const int mn = m < n ? m : n;
    for (int i = 0; i < mn; ++i) {
        T *x = A + i + (size_t)i * lda;
        const int len = m - i;
        // reflection_axis_mut: sq = 0 + dotc(x, x)
        if (threadIdx.x < 8) {
            T d = group_dot8<T>(x, x, len, threadIdx.x, scratch);
            if (threadIdx.x == 0) {
                const T sq = T(0) + d;
                const T nrm = sqrt(sq);
                const T x0 = x[0];
                const T mod = x0 >= T(0) ? x0 : -x0;
                const T sgn = x0 >= T(0) ? T(1) : T(-1);
                const T signed_norm = sgn * nrm;
                const T factor = (sq + mod * nrm) * T(2);
                x[0] = x0 + signed_norm;
                sh[0] = factor;
                sh[1] = signed_norm;
            }
        }
        __syncthreads();
        const T factor = sh[0], signed_norm = sh[1];
        const bool not_zero = factor != T(0);
        if (not_zero) {
            const T s = sqrt(factor);
            for (int r = threadIdx.x; r < len; r += blockDim.x) x[r] = x[r] / s;
            __syncthreads();
            if (threadIdx.x < 8) {
                T d = group_dot8<T>(x, x, len, threadIdx.x, scratch);
                if (threadIdx.x == 0) sh[2] = sqrt(T(0) + d);
            }
            __syncthreads();
            const T nn = sh[2];
            for (int r = threadIdx.x; r < len; r += blockDim.x) x[r] = x[r] / nn;
            __syncthreads();
            const T ret = -signed_norm;
            reflect_cols<T>(x, len, A + i, lda, i + 1, n, signum_rs(ret), scratch);
            if (threadIdx.x == 0) diag[i] = ret;
        } else if (threadIdx.x == 0) {
            diag[i] = signed_norm;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- columns in parallel
//
// A column only ever needs the reflectors before it, in order, so the columns
// are a pipeline: a workgroup holds PC columns in registers (thread t rows t,
// t + PT, ...), applies the reflectors of earlier columns as they are published,
// makes its own PC reflectors one after the other (applying each to its later
// columns straight from registers) and publishes them.  Workgroups take tickets
// in column order, so the one that is waited for is already running.
//
// What bounds the pipeline is the chain through the columns: per column one dot
// product with the previous axis and two with itself (the norm, then the norm
// of the scaled axis), each eight chains of len / 8 dependent additions
// (dotx's accumulators, blas.rs:93-167).  So all wavefronts make the products
// and leave them in LDS, and one wavefront runs the chains of all PC columns
// side by side (lane q + 8c); divisions by the common norm take three
// instructions (exact_div.hpp).  Four columns per workgroup: the hand-over
// between workgroups (about 2 us) then falls on every fourth column, and four
// chains take one chain's time.
// 1500 x 200 f64: 42.1 -> 1.13 ms; Q^T b of one column 8.1 -> 0.35 ms (before:
// one workgroup, a column after the other, columns re-read from memory).
//
// A published element is its own flag: the buffer starts as a signalling NaN
// pattern, which no arithmetic result has (results are quieted), and a reader
// polls until another value is there.  Waits are bounded: a reader that gives up
// goes on with that NaN, which reaches every later column and its diagonal entry.
constexpr int PT = 512;               // threads per workgroup
constexpr long QR_SPIN_LIMIT = 1L << 21;  // some seconds

template <typename T> struct Word;
template <> struct Word<double> {
    typedef unsigned long long U;
    static constexpr U EMPTY = 0x7ff0000000000001ull;
    static __device__ __forceinline__ U bits(double v) { return (U)__double_as_longlong(v); }
    static __device__ __forceinline__ double value(U u) { return __longlong_as_double((long long)u); }
};
template <> struct Word<float> {
    typedef unsigned U;
    static constexpr U EMPTY = 0x7f800001u;
    static __device__ __forceinline__ U bits(float v) { return __float_as_uint(v); }
    static __device__ __forceinline__ float value(U u) { return __uint_as_float(u); }
};

template <int N>
__device__ __forceinline__ double row_shl(double v) { return nrocm_sweep::row_shl<N>(v); }
template <int N>
__device__ __forceinline__ float row_shl(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x100 + N, 0xf, 0xf, true));
}

constexpr int DU = 16;                       // chain steps read ahead
constexpr int DOT_SLACK = 3 * 8 * DU;        // elements read (not used) past the last product

// dotx over the len products p[0], p[1], ... in LDS by one wavefront: lane q of
// each group of eight lanes runs accumulator q; its lane 0 ends with the sum.
// Zeros in place of missing elements are exact: a sum that starts at +0 never
// becomes -0.
template <typename T>
__device__ __forceinline__ T wave_dot(const T *p, int len, int q)
{
    const int M = len >> 3, tail = len & 7;
    const int groups = M / DU, rest = M % DU;
    T tp = p[8 * M + q];
    tp = q < tail ? tp : T(0);
    T va[DU], vb[DU];
    auto read = [&](T (&v)[DU], int g) {
#pragma unroll
        for (int u = 0; u < DU; ++u) v[u] = p[q + 8 * (g * DU + u)];
        __builtin_amdgcn_sched_barrier(0);
    };
    T acc = 0;
    auto sum = [&](const T (&v)[DU]) {
#pragma unroll
        for (int u = 0; u < DU; ++u) acc += v[u];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto last = [&](const T (&v)[DU]) {
#pragma unroll
        for (int u = 0; u < DU - 1; ++u) acc += u < rest ? v[u] : T(0);
    };
    read(va, 0);
    read(vb, 1);
    int g = 0;
#pragma unroll 1
    for (; g + 2 <= groups; g += 2) {
        sum(va);
        read(va, g + 2);
        sum(vb);
        read(vb, g + 3);
    }
    if (g < groups) {
        sum(va);
        last(vb);
    } else {
        last(va);
    }
    const T t1 = row_shl<1>(tp), t2 = row_shl<2>(tp), t3 = row_shl<3>(tp), t4 = row_shl<4>(tp), t5 = row_shl<5>(tp),
            t6 = row_shl<6>(tp);
    const T pair = acc + row_shl<4>(acc);
    const T p1 = row_shl<1>(pair), p2 = row_shl<2>(pair), p3 = row_shl<3>(pair);
    T res = 0;
    res += pair;
    res += p1;
    res += p2;
    res += p3;
    res += tp;
    res += t1;
    res += t2;
    res += t3;
    res += t4;
    res += t5;
    res += t6;
    return res;
}

// x / d for a workgroup-uniform d with its refined reciprocal.
__device__ __forceinline__ double quotient(double x, double d, double rec, bool dok)
{
    const bool ok = dok && nrocm_div::num_in_range(x);
    double r = nrocm_div::div_with(x, d, rec);
    if (__ballot(!ok) != 0) r = ok ? r : x / d;
    return r;
}
__device__ __forceinline__ float quotient(float x, float d, float, bool) { return x / d; }
__device__ __forceinline__ double recip(double d) { return nrocm_div::recip_refined(d); }
__device__ __forceinline__ float recip(float) { return 0.f; }
__device__ __forceinline__ bool den_ok(double d) { return nrocm_div::div_den_ok(d); }
__device__ __forceinline__ bool den_ok(float) { return true; }

// Doubles (or floats) between the columns' products: rows of different columns
// eight elements apart in the banks.
__host__ __device__ constexpr int prod_stride(int m) { return (m + 31) / 32 * 32 + 8; }
__host__ __device__ constexpr size_t qr_lds_elements(int m, int pc) { return (size_t)pc * prod_stride(m) + DOT_SLACK; }

// Reflects columns KB..nc of x through axis v (rows j.., the thread's own)
// with the given sign (reflect_with_sign, reflection.rs:70-83), or, with a sign
// of 0, leaves them.  Every thread of the workgroup calls it: whether there is an
// axis is no reason to skip its barriers, because after a wait that ran out the
// wavefronts may differ about it.
template <typename T, int RPT, int PC, int KB>
__device__ __forceinline__ void reflect(T (&x)[PC][RPT], const T (&v)[RPT], T sign, int j, int m, int nc, T *prod,
                                        T *fac)
{
    const int t = threadIdx.x, lane = t & 63;
    const int ps = prod_stride(m);
#pragma unroll
    for (int c = KB; c < PC; ++c)
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            if (r < m) prod[c * ps + r] = v[s] * x[c][s];
        }
    lds_barrier();
    if (t < 64) {
        const int q = lane & 7, c = min(max(lane >> 3, KB), PC - 1);
        const T d = wave_dot<T>(prod + c * ps + j, m - j, q);
        const T m_two = sign * T(-2);
        if (q == 0 && (lane >> 3) >= KB && (lane >> 3) < PC) fac[c] = (d - T(0)) * m_two;
    }
    lds_barrier();
#pragma unroll
    for (int c = KB; c < PC; ++c) {
        const T f = fac[c];
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            const T y = axcpy1<T>(f, v[s], T(1), sign, x[c][s]);
            x[c][s] = r >= j && sign != T(0) ? y : x[c][s];  // NaN reflects too
        }
    }
}

// Makes reflector i from column K of x (reflection_axis_mut, householder.rs:
// 19-53): the unit axis replaces rows i.. of the column; returns its sign (0:
// no reflection) and stores the diagonal entry.
template <typename T, int RPT, int PC, int K>
__device__ __forceinline__ T make_axis(T (&x)[PC][RPT], int i, int m, T *prod, T *sc, T *diag)
{
    const int t = threadIdx.x;
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const int r = t + PT * s;
        if (r < m) prod[r] = x[K][s] * x[K][s];
        if (r == i) sc[0] = x[K][s];
    }
    lds_barrier();
    if (t < 64) {
        const T d = wave_dot<T>(prod + i, m - i, t & 7);
        if (t == 0) {
            const T sq = T(0) + d;
            const T nrm = sqrt(sq);
            const T x0 = sc[0];
            const T mod = x0 >= T(0) ? x0 : -x0;
            const T sgn = x0 >= T(0) ? T(1) : T(-1);
            const T signed_norm = sgn * nrm;
            const T factor = (sq + mod * nrm) * T(2);
            const T s = sqrt(factor);
            sc[1] = factor;
            sc[2] = signed_norm;
            sc[3] = s;
            sc[4] = x0 + signed_norm;
            sc[5] = recip(s);
        }
    }
    lds_barrier();
    const T factor = sc[1], signed_norm = sc[2];
    const T s = sc[3], x0n = sc[4], srec = sc[5];
#pragma unroll
    for (int k = 0; k < RPT; ++k)
        if (t + PT * k == i) x[K][k] = x0n;
    if (!(factor != T(0))) {
        if (t == 0) diag[i] = signed_norm;
        return T(0);
    }
    const bool sok = den_ok(s);
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int r = t + PT * k;
        const T y = quotient(r >= i ? x[K][k] : T(1), s, srec, sok);
        x[K][k] = r >= i ? y : x[K][k];
        if (r < m) prod[r] = x[K][k] * x[K][k];
    }
    lds_barrier();
    if (t < 64) {
        const T d = wave_dot<T>(prod + i, m - i, t & 7);
        if (t == 0) {
            const T nn = sqrt(T(0) + d);
            sc[6] = nn;
            sc[7] = recip(nn);
        }
    }
    lds_barrier();
    const T nn = sc[6], nrec = sc[7];
    const bool nok = den_ok(nn);
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int r = t + PT * k;
        const T y = quotient(r >= i ? x[K][k] : T(1), nn, nrec, nok);
        x[K][k] = r >= i ? y : x[K][k];
    }
    const T ret = -signed_norm;
    if (t == 0) diag[i] = ret;
    return signum_rs(ret);
}

// Own columns K, K+1, ... of a workgroup in turn.
template <typename T, int RPT, int PC, int K>
__device__ __forceinline__ void own_columns(T (&x)[PC][RPT], int c0, int nc, int m, int mn, T *prod, T *sc, T *fac,
                                            T *diag, typename Word<T>::U *V, typename Word<T>::U *H)
{
    if constexpr (K < PC) {
        const int i = c0 + K;
        if (K >= nc || i >= mn) return;
        const T sign = make_axis<T, RPT, PC, K>(x, i, m, prod, sc, diag);
        if (V) {
            typename Word<T>::U *dst = V + (size_t)i * m;
            if (sign != T(0)) {
#pragma unroll
                for (int s = 0; s < RPT; ++s) {
                    const int r = (int)threadIdx.x + PT * s;
                    if (r >= i && r < m)
                        __hip_atomic_store(dst + r, Word<T>::bits(x[K][s]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (threadIdx.x == 0)
                __hip_atomic_store(H + i, Word<T>::bits(sign), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if constexpr (K + 1 < PC) {
            if (sign != T(0)) {  // NaN reflects too
                T v[RPT];
#pragma unroll
                for (int s = 0; s < RPT; ++s) v[s] = x[K][s];
                reflect<T, RPT, PC, K + 1>(x, v, sign, i, m, nc, prod, fac);
            }
        }
        own_columns<T, RPT, PC, K + 1>(x, c0, nc, m, mn, prod, sc, fac, diag, V, H);
    }
}

template <typename T, int RPT, int PC>
__global__ __launch_bounds__(PT) void geqrf_columns_kernel(T *A, int m, int n, int lda, T *diag,
                                                           typename Word<T>::U *V, typename Word<T>::U *H, int *ticket,
                                                           long limit)
{
    typedef typename Word<T>::U U;
    extern __shared__ __align__(16) unsigned char qr_lds[];
    T *prod = reinterpret_cast<T *>(qr_lds);
    __shared__ T sc[8], fac[PC];
    __shared__ int my;
    const int t = threadIdx.x;
    if (ticket) {
        if (t == 0) my = atomicAdd(ticket, 1);
        __syncthreads();
    }
    const int c0 = (ticket ? my : 0) * PC;
    const int nc = min(PC, n - c0), mn = min(m, n);
    T x[PC][RPT];
#pragma unroll
    for (int c = 0; c < PC; ++c)
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            x[c][s] = (c < nc && r < m) ? A[r + (size_t)(c0 + c) * lda] : T(0);
        }
    const int jend = min(c0, mn);
    U w[RPT], nw[RPT], hw = 0, nh = 0;
    auto issue = [&](U (&d)[RPT], U &h, int j) {
        const U *src = V + (size_t)j * m;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            d[s] = __hip_atomic_load(src + min(max(r, j), m - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        h = __hip_atomic_load(H + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (jend > 0) issue(w, hw, 0);
    for (int j = 0; j < jend; ++j) {
        long spins = 0;
        for (;;) {
            bool ok = hw != Word<T>::EMPTY;
            if (Word<T>::value(hw) != T(0)) {  // else nothing to wait for
#pragma unroll
                for (int s = 0; s < RPT; ++s) ok = ok && w[s] != Word<T>::EMPTY;
            }
            if (ok || ++spins >= limit) break;
            __builtin_amdgcn_s_sleep(1);
            issue(w, hw, j);
        }
        const T sign = Word<T>::value(hw);
        T v[RPT];
#pragma unroll
        for (int s = 0; s < RPT; ++s) v[s] = Word<T>::value(w[s]);
        if (j + 1 < jend) issue(nw, nh, j + 1);
        reflect<T, RPT, PC, 0>(x, v, sign, j, m, nc, prod, fac);
#pragma unroll
        for (int s = 0; s < RPT; ++s) w[s] = nw[s];
        hw = nh;
    }
    // every column has arrived on every path: else its first use after the first
    // published axis would wait for those stores
#pragma unroll
    for (int c = 0; c < PC; ++c)
#pragma unroll
        for (int s = 0; s < RPT; ++s) asm volatile("" : "+v"(x[c][s]));
    own_columns<T, RPT, PC, 0>(x, c0, nc, m, mn, prod, sc, fac, diag, V, H);
#pragma unroll
    for (int c = 0; c < PC; ++c)
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            if (c < nc && r < m) A[r + (size_t)(c0 + c) * lda] = x[c][s];
        }
}

template <typename U>
__global__ void qr_prep_kernel(U *p, size_t count, U empty, int *ticket)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *ticket = 0;
    for (size_t e = i; e < count; e += (size_t)gridDim.x * blockDim.x) p[e] = empty;
}

// QR::q_tr_mul (qr.rs:157-171), or with REVERSE Q B with Q as QR::q builds it
// (qr.rs:108-129: the reflectors in reverse order, each with the sign of its
// diagonal entry; the product with the identity reproduces QR::q up to the sign
// of zero entries left of the diagonal, which q() never touches): PC columns of
// B per workgroup, in registers for all reflectors, the next axis being loaded
// during the current one's dot products.
template <int RPT, int PC, bool REVERSE>
__global__ __launch_bounds__(PT) void qr_apply_kernel(const double *__restrict__ QR, int m, int n, int lda,
                                                      const double *__restrict__ diag, double *B, int ldb, int nrhs)
{
    extern __shared__ __align__(16) unsigned char qr_lds[];
    double *prod = reinterpret_cast<double *>(qr_lds);
    __shared__ double fac[PC];
    const int t = threadIdx.x;
    const int c0 = blockIdx.x * PC;
    const int nc = min(PC, nrhs - c0), mn = min(m, n);
    double x[PC][RPT], v[RPT], nv[RPT];
#pragma unroll
    for (int c = 0; c < PC; ++c)
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            x[c][s] = (c < nc && r < m) ? B[r + (size_t)(c0 + c) * ldb] : 0.0;
        }
    auto axis = [&](double (&d)[RPT], int j) {
        const double *src = QR + (size_t)j * lda;
#pragma unroll
        for (int s = 0; s < RPT; ++s) d[s] = src[min(t + PT * s, m - 1)];
    };
    axis(v, REVERSE ? mn - 1 : 0);
    for (int k = 0; k < mn; ++k) {
        const int j = REVERSE ? mn - 1 - k : k;
        const double sign = signum_rs(diag[j]);
        if (k + 1 < mn) axis(nv, REVERSE ? j - 1 : j + 1);
        reflect<double, RPT, PC, 0>(x, v, sign, j, m, nc, prod, fac);
#pragma unroll
        for (int s = 0; s < RPT; ++s) v[s] = nv[s];
    }
#pragma unroll
    for (int c = 0; c < PC; ++c)
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int r = t + PT * s;
            if (c < nc && r < m) B[r + (size_t)(c0 + c) * ldb] = x[c][s];
        }
}

// QR::q_tr_mul / Q B on one workgroup, B in memory: more rows than the
// registers of qr_apply_kernel hold.
template <bool REVERSE>
__global__ __launch_bounds__(256) void qr_apply_tall_kernel(const double *QR, int m, int n, int lda,
                                                            const double *diag, double *B, int ldb, int nrhs)
{
    __shared__ double scratch[256];
    const int mn = m < n ? m : n;
    for (int k = 0; k < mn; ++k) {
        const int i = REVERSE ? mn - 1 - k : k;
        reflect_cols<double>(QR + i + (size_t)i * lda, m - i, B + i, ldb, 0, nrhs, signum_rs(diag[i]), scratch);
        __syncthreads();
    }
}

// B (n x nrhs) <- R B with R the n x n upper triangle of QR::r (qr.rs:81-89:
// |diag| on the diagonal), in the reference BLAS TRMM order (side left,
// upper, no transpose): row i is ((b_i r_ii + b_{i+1} r_{i,i+1}) + ...) over
// the input values, a zero b_k contributing nothing.  One thread per row; the
// input column is read from B0 (a copy), the result written to B.
__global__ __launch_bounds__(256) void rmul_kernel(const double *QR, int n, int lda, const double *diag,
                                                   const double *B0, double *B, int ldb, int nrhs)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    for (int c = blockIdx.y; c < nrhs; c += gridDim.y) {
        if (i >= n) continue;
        const double *b0 = B0 + (size_t)c * n;
        const double bi = b0[i];
        double acc = (bi != 0.0) ? bi * fabs(diag[i]) : bi;
        const double *rrow = QR + i;
        for (int k = i + 1; k < n; ++k) {
            const double bk = b0[k];
            if (bk != 0.0) acc = acc + bk * rrow[(size_t)k * lda];
        }
        B[i + (size_t)c * ldb] = acc;
    }
}

// Most rows of the kernels that hold columns in registers.
constexpr int QR_COLUMNS_MAX = 32 * PT;

template <typename T, int RPT, int PC>
int geqrf_columns(nrocm_handle h, int m, int n, T *a, int lda, T *diag)
{
    typedef typename Word<T>::U U;
    const unsigned groups = nrocm_cdiv(n, PC);
    int *ticket = nullptr;
    U *V = nullptr, *H = nullptr;
    if (groups > 1) {
        const int mn = std::min(m, n);
        const size_t words = (size_t)mn * m + mn;
        void *ws = nullptr;
        const int s = nrocm_workspace(h, 256 + words * sizeof(U), &ws);
        if (s != NROCM_OK) return s;
        ticket = (int *)ws;
        V = (U *)((char *)ws + 256);
        H = V + (size_t)mn * m;
        hipLaunchKernelGGL((qr_prep_kernel<U>), dim3(std::min(2048u, nrocm_cdiv(words, 512))), dim3(256), 0, h->stream,
                           V, words, Word<T>::EMPTY, ticket);
    }
    nrocm_allow_lds<geqrf_columns_kernel<T, RPT, PC>>(h->device);
    hipLaunchKernelGGL((geqrf_columns_kernel<T, RPT, PC>), dim3(groups), dim3(PT),
                       qr_lds_elements(m, PC) * sizeof(T), h->stream, a, m, n, lda, diag, V, H, ticket,
                       nrocm_wait_limit(h, QR_SPIN_LIMIT));
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}

// Matrices whose columns take less time than the pipeline's hand-overs and the
// filling of its buffer (f64, us, one workgroup and pipeline: 2 x 2 4.2 and 5.8, 4 x 4 8.4
// and 9.6, 8 x 4 9.9 and 9.7, 5 x 5 10.8 and 15.3, 20 x 20 48.7 and 50.6, 24 x 24 61.0 and 60.4;
// f32: 5 x 5 10.2 and 12.7, 12 x 12 24.8 and 25.6, 16 x 16 34.8 and 33.1).  Up to four columns
// are one group and need no buffer.
bool qr_is_tiny(int m, int n, bool f64)
{
    if (n <= 4) return n > 1 && m <= 4;
    return std::max(m, n) <= (f64 ? 20 : 12);
}

// The column pipeline takes its hand-over buffer from the handle's workspace;
// on a stream under capture, where that may not grow and must not be baked in,
// and above the rows that registers hold, one workgroup walks the columns.
template <typename T>
int geqrf(nrocm_handle h, int m, int n, T *a, int lda, T *diag)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(h->stream, &cap) != hipSuccess) {
        (void)hipGetLastError();  // the legacy stream beside a capture
        cap = hipStreamCaptureStatusActive;
    }
    if (cap != hipStreamCaptureStatusNone || m > QR_COLUMNS_MAX || qr_is_tiny(m, n, sizeof(T) == 8)) {
        hipLaunchKernelGGL((geqrf_exact_kernel<T>), dim3(1), dim3(256), 0, h->stream, a, m, n, lda, diag);
        NROCM_CHECK_LAUNCH(h);
        return NROCM_OK;
    }
    if (m <= PT) return geqrf_columns<T, 1, 4>(h, m, n, a, lda, diag);
    if (m <= 2 * PT) return geqrf_columns<T, 2, 4>(h, m, n, a, lda, diag);
    if (m <= 4 * PT) return geqrf_columns<T, 4, 4>(h, m, n, a, lda, diag);
    if (m <= 8 * PT) return geqrf_columns<T, 8, 4>(h, m, n, a, lda, diag);
    if (m <= 16 * PT) return geqrf_columns<T, 16, 2>(h, m, n, a, lda, diag);
    return geqrf_columns<T, 32, 1>(h, m, n, a, lda, diag);
}

template <int RPT, int PC, bool REVERSE>
int qr_apply_columns(nrocm_handle h, int m, int n, const double *qr, int lda, const double *diag, int nrhs, double *b,
                     int ldb)
{
    nrocm_allow_lds<qr_apply_kernel<RPT, PC, REVERSE>>(h->device);
    hipLaunchKernelGGL((qr_apply_kernel<RPT, PC, REVERSE>), dim3(nrocm_cdiv(nrhs, PC)), dim3(PT),
                       qr_lds_elements(m, PC) * sizeof(double), h->stream, qr, m, n, lda, diag, b, ldb, nrhs);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}

// One column per workgroup while that leaves CUs free (it is the shorter
// chain), four when the chip is full.
template <bool REVERSE>
int qr_apply(nrocm_handle h, int m, int n, const double *qr, int lda, const double *diag, int nrhs, double *b, int ldb)
{
    const bool one = nrhs <= h->num_cus;
#define NROCM_APPLY(RPT, PC)                                                                                  \
    (one || PC == 1 ? qr_apply_columns<RPT, 1, REVERSE>(h, m, n, qr, lda, diag, nrhs, b, ldb)                 \
                    : qr_apply_columns<RPT, PC, REVERSE>(h, m, n, qr, lda, diag, nrhs, b, ldb))
    if (m <= PT) return NROCM_APPLY(1, 4);
    if (m <= 2 * PT) return NROCM_APPLY(2, 4);
    if (m <= 4 * PT) return NROCM_APPLY(4, 4);
    if (m <= 8 * PT) return NROCM_APPLY(8, 4);
    if (m <= 16 * PT) return NROCM_APPLY(16, 2);
    if (m <= QR_COLUMNS_MAX) return NROCM_APPLY(32, 1);
#undef NROCM_APPLY
    hipLaunchKernelGGL((qr_apply_tall_kernel<REVERSE>), dim3(1), dim3(256), 0, h->stream, qr, m, n, lda, diag, b, ldb,
                       nrhs);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}

__global__ void copy_cols_kernel(const double *B, int ldb, int n, int nrhs, double *B0)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < (size_t)n * nrhs) B0[e] = B[(e % n) + (e / n) * (size_t)ldb];
}

}  // namespace

// ---------------------------------------------------------------- batched tall least squares
#include "qr_batched.inc"

extern "C" {

int nrocm_dgeqrf(nrocm_handle h, int m, int n, double *a, int lda, double *diag)
{
    if (!h) return -1;
    if (m < 0) return -2;
    if (n < 0) return -3;
    if (!a && m > 0 && n > 0) return -4;
    if (lda < std::max(1, m)) return -5;
    if (!diag && std::min(m, n) > 0) return -6;
    if (std::min(m, n) == 0) return NROCM_OK;
    return geqrf<double>(h, m, n, a, lda, diag);
}

int nrocm_sgeqrf(nrocm_handle h, int m, int n, float *a, int lda, float *diag)
{
    if (!h) return -1;
    if (m < 0) return -2;
    if (n < 0) return -3;
    if (!a && m > 0 && n > 0) return -4;
    if (lda < std::max(1, m)) return -5;
    if (!diag && std::min(m, n) > 0) return -6;
    if (std::min(m, n) == 0) return NROCM_OK;
    return geqrf<float>(h, m, n, a, lda, diag);
}

int nrocm_dqr_qtmul(nrocm_handle h, int m, int n, const double *qr, int lda, const double *diag, int nrhs,
                    double *b, int ldb)
{
    if (!h) return -1;
    if (m < 0) return -2;
    if (n < 0) return -3;
    if (!qr && m > 0 && n > 0) return -4;
    if (lda < std::max(1, m)) return -5;
    if (!diag && std::min(m, n) > 0) return -6;
    if (nrhs < 0) return -7;
    if (!b && m > 0 && nrhs > 0) return -8;
    if (ldb < std::max(1, m)) return -9;
    if (std::min(m, n) == 0 || nrhs == 0) return NROCM_OK;
    return qr_apply<false>(h, m, n, qr, lda, diag, nrhs, b, ldb);
}

int nrocm_dqr_qmul(nrocm_handle h, int m, int n, const double *qr, int lda, const double *diag, int nrhs, double *b,
                   int ldb)
{
    if (!h) return -1;
    if (m < 0) return -2;
    if (n < 0) return -3;
    if (!qr && m > 0 && n > 0) return -4;
    if (lda < std::max(1, m)) return -5;
    if (!diag && std::min(m, n) > 0) return -6;
    if (nrhs < 0) return -7;
    if (!b && m > 0 && nrhs > 0) return -8;
    if (ldb < std::max(1, m)) return -9;
    if (std::min(m, n) == 0 || nrhs == 0) return NROCM_OK;
    return qr_apply<true>(h, m, n, qr, lda, diag, nrhs, b, ldb);
}

int nrocm_dqr_rmul(nrocm_handle h, int m, int n, const double *qr, int lda, const double *diag, int nrhs, double *b,
                   int ldb)
{
    if (!h) return -1;
    if (m < 0) return -2;
    if (n < 0 || n > m) return -3;
    if (!qr && n > 0) return -4;
    if (lda < std::max(1, m)) return -5;
    if (!diag && n > 0) return -6;
    if (nrhs < 0) return -7;
    if (!b && n > 0 && nrhs > 0) return -8;
    if (ldb < std::max(1, n)) return -9;
    if (n == 0 || nrhs == 0) return NROCM_OK;
    void *ws = nullptr;
    const int s = nrocm_workspace(h, (size_t)n * nrhs * sizeof(double), &ws);
    if (s != NROCM_OK) return s;
    double *b0 = (double *)ws;
    const size_t tot = (size_t)n * nrhs;
    hipLaunchKernelGGL(copy_cols_kernel, dim3(nrocm_cdiv(tot, 256)), dim3(256), 0, h->stream, b, ldb, n, nrhs, b0);
    hipLaunchKernelGGL(rmul_kernel, dim3(nrocm_cdiv(n, 256), std::min(nrhs, 65535)), dim3(256), 0, h->stream, qr, n,
                       lda, diag, b0, b, ldb, nrhs);
    NROCM_CHECK_LAUNCH(h);
    return NROCM_OK;
}

int nrocm_dqr_rsolve(nrocm_handle h, int n, const double *qr, int lda, const double *diag, int nrhs, double *b,
                     int ldb, int *info)
{
    if (!h) return -1;
    if (n < 0) return -2;
    if (!qr && n > 0) return -3;
    if (lda < std::max(1, n)) return -4;
    if (!diag && n > 0) return -5;
    if (nrhs < 0) return -6;
    if (!b && n > 0 && nrhs > 0) return -7;
    if (ldb < std::max(1, n)) return -8;
    if (!info) return -9;
    return nrocm_qr_rsolve(h, n, nrhs, qr, lda, diag, b, ldb, info);
}

}  // extern "C"
