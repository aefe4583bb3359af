// Substitutions of the batched adjoints, eight lanes to a member.
#pragma once
#include "nrocm_internal.hpp"

namespace nrocm_adjoint {

// x of lane T of the eight-lane group, in lane J (T, J static)
template <int J, int T>
__device__ __forceinline__ double from_lane(double x)
{
    if constexpr (J == T) {
        return x;
    } else {
        constexpr int CTRL = J > T ? 0x110 + (J - T) : 0x100 + (T - J);  // row_shr, row_shl
        const long long v = __double_as_longlong(x);
        const int lo = __builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), CTRL, 0xf, 0xf, true);
        return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
    }
}

// res + x of lanes FROM, FROM + STEP, ... (COUNT of them), in that order, in lane J
template <int J, int FROM, int STEP, int COUNT>
__device__ __forceinline__ double add_lanes(double res, double x)
{
    if constexpr (COUNT > 0) {
        res += from_lane<J, FROM>(x);
        res = add_lanes<J, FROM + STEP, STEP, COUNT - 1>(res, x);
    }
    return res;
}

// Members per wavefront of a batch: as few as fill the chip with one wavefront per
// SIMD.  A step takes as long for one member as for eight, but its columns come
// sooner, and the outer product is the whole wavefront's, member after member.
// (Cholesky's adjoint, us, 8 in each wavefront, now, and with two per SIMD: 8 members
// of 64, 4 right-hand sides 236 / 107 / 107, 512 of 64 246 / 113 / 112, 2048 of 16, one
// 15.4 / 11.4 / 16.2, 4096 of 32 40.0 / 30.7 / 35.4.)
inline int members_per_wave(int num_cus, int count)
{
    for (int per = 1; per < 8; per *= 2)
        if ((long)count <= (long)per * 4 * num_cus) return per;
    return 8;
}

// The adjoint's two substitutions read a matrix column by column; a group of
// eight lanes holds one member, lane c the solved values of index c modulo 8:
// the eight interleaved accumulators of dotx (src/base/blas.rs:93-167) are the
// eight lanes.  The columns are fetched AHEAD steps before their use.
constexpr int AHEAD = 4;

// A member's matrix; in the global address space, because a flat load (of an
// address that comes from memory) is waited for with all the others.
typedef const __attribute__((address_space(1))) double *Matrix;

template <int KM>
struct Column {
    double x[KM];  // the elements that meet solved blocks 0, 1, ...
    double cur;    // those of the block in work
};

// ---- U^T y = g, i = 8 kb + J ascending: the products of whole blocks of 8
// before i in the lanes' accumulators, those of i's own block one after another.
template <int KM, int CH, int J>
__device__ __forceinline__ void upper_step(int kb, int c, const Column<KM> &u, const double (&z)[CH][KM],
                                           double (&cur)[CH], const double (&gv)[CH])
{
#pragma unroll
    for (int q = 0; q < CH; ++q) {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < KM; ++k) {
            const double p = u.x[k] * z[q][k];
            acc += k < kb ? p : 0.0;
        }
        const double tail = u.cur * cur[q];
        const double pair = acc + from_lane<0, 4>(acc);  // in lanes 0..3
        double res = add_lanes<J, 0, 1, 4>(0.0, pair);
        res = add_lanes<J, 0, 1, J>(res, tail);
        const double y = (gv[q] - res) / u.cur;  // in lane J
        cur[q] = c == J ? y : cur[q];
    }
}

// accumulators 0..3 (each with its pair) of step J of the descending pass: T = 0..3
template <int J, int T>
__device__ __forceinline__ double add_pairs(double res, double pair)
{
    if constexpr (T < 4) {
        res += from_lane<J, (J + 7 - T) & 3>(pair);
        res = add_pairs<J, T + 1>(res, pair);
    }
    return res;
}

// ---- L^T z = y, i = n - 1 - s descending, s = 8 kb + J: counted from the end
// (e = n - 1 - row), the dot runs over e = s - 1 down to 0, so its whole blocks
// of 8 end at e = J and the tail is e = J - 1 .. 0.  Accumulator t holds the e
// with e = J - 1 - t modulo 8.
template <bool UNIT, int KM, int CH, int J>
__device__ __forceinline__ void lower_step(int kb, int c, const Column<KM> &l, const double (&z)[CH][KM],
                                           double (&cur)[CH], const double (&yv)[CH])
{
#pragma unroll
    for (int q = 0; q < CH; ++q) {
        const double pc = l.cur * cur[q];
        double acc = 0.0;
        acc += (kb > 0 && c < J) ? pc : 0.0;
        double p0 = 0.0;
#pragma unroll
        for (int k = KM - 1; k >= 0; --k) {
            const double p = l.x[k] * z[q][k];
            acc += (k < kb && (k > 0 || c >= J)) ? p : 0.0;
            if (k == 0) p0 = p;
        }
        const double tail = kb > 0 ? p0 : pc;
        const double pair = acc + from_lane<0, 4>(acc);  // in lanes 0..3
        double res = add_pairs<J, 0>(0.0, pair);
        res = add_lanes<J, J - 1, -1, J>(res, tail);
        double y = yv[q] - res;  // the unit diagonal divides by one
        if constexpr (!UNIT) y = y / l.cur;
        cur[q] = c == J ? y : cur[q];
    }
}

template <int KM>
__device__ __forceinline__ void fetch_upper(Column<KM> &u, Matrix M, int n, int i, int c)
{
    i = min(i, n - 1);
    Matrix col = M + (size_t)i * n;
#pragma unroll
    for (int k = 0; k < KM; ++k) u.x[k] = col[min(8 * k + c, i)];
    u.cur = col[min((i & ~7) + c, i)];
}

template <bool UNIT, int KM>
__device__ __forceinline__ void fetch_lower(Column<KM> &l, Matrix M, int n, int s, int c)
{
    s = min(s, n - 1);
    const int i = n - 1 - s, top = UNIT ? min(i + 1, n - 1) : i;
    Matrix col = M + (size_t)i * n;
#pragma unroll
    for (int k = 0; k < KM; ++k) l.x[k] = col[max(n - 1 - 8 * k - c, top)];
    l.cur = col[max(n - 1 - (s & ~7) - c, top)];
}

// ---- L y = g, i = 8 kb + J ascending: y_i = b_i / L_ii goes to the whole group,
// b_r -= y_i L_ri for the rows below (axpy's order, the negation on y_i).
template <int J>
__device__ __forceinline__ double group_lane(double x)
{
    const long long v = __double_as_longlong(x);
    // lane J of each 16-lane row to its lanes 0..7, lane J + 8 to lanes 8..15
    int lo = __builtin_amdgcn_update_dpp(0, (int)v, 0x150 + J, 0xf, 0xf, true);
    int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), 0x150 + J, 0xf, 0xf, true);
    lo = __builtin_amdgcn_update_dpp(lo, (int)v, 0x158 + J, 0xf, 0xc, false);
    hi = __builtin_amdgcn_update_dpp(hi, (int)(v >> 32), 0x158 + J, 0xf, 0xc, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int KM, int CH, int J>
__device__ __forceinline__ void forward_step(int kb, int c, const Column<KM> &l, double (&b)[CH][KM], double (&cur)[CH])
{
#pragma unroll
    for (int q = 0; q < CH; ++q) {
        const double y = group_lane<J>(cur[q] / l.cur);
        const double below = cur[q] + (-y) * l.cur;
        cur[q] = c == J ? y : c > J ? below : cur[q];
#pragma unroll
        for (int k = 1; k < KM; ++k) {
            const double r = b[q][k] + (-y) * l.x[k];
            b[q][k] = k > kb ? r : b[q][k];
        }
    }
}

template <int KM>
__device__ __forceinline__ void fetch_forward(Column<KM> &l, Matrix M, int n, int i, int c)
{
    i = min(i, n - 1);
    Matrix col = M + (size_t)i * n;
#pragma unroll
    for (int k = 1; k < KM; ++k) l.x[k] = col[min(max(8 * k + c, i), n - 1)];
    l.cur = col[min(max((i & ~7) + c, i), n - 1)];
}

// U^T y = g; L^T y = g with a unit diagonal; the same with L's own; L y = g.
enum Kind { UPPER, UNIT_LOWER, LOWER, FORWARD };

template <Kind K, int KM>
__device__ __forceinline__ void fetch(Column<KM> &u, Matrix M, int n, int s, int c)
{
    if constexpr (K == UPPER) fetch_upper<KM>(u, M, n, s, c);
    else if constexpr (K == FORWARD) fetch_forward<KM>(u, M, n, s, c);
    else fetch_lower<K == UNIT_LOWER, KM>(u, M, n, s, c);
}

template <Kind K, int KM, int CH, int J>
__device__ __forceinline__ void block_steps(int kb, int c, Column<KM> (&ring)[AHEAD], Matrix M, int n,
                                            double (&z)[CH][KM], double (&cur)[CH], const double (&gv)[CH])
{
    if constexpr (J < 8) {
        if constexpr (K == UPPER) upper_step<KM, CH, J>(kb, c, ring[J % AHEAD], z, cur, gv);
        else if constexpr (K == FORWARD) forward_step<KM, CH, J>(kb, c, ring[J % AHEAD], z, cur);
        else lower_step<K == UNIT_LOWER, KM, CH, J>(kb, c, ring[J % AHEAD], z, cur, gv);
        fetch<K, KM>(ring[J % AHEAD], M, n, 8 * kb + J + AHEAD, c);
        // one step at a time: interleaved, the steps of the adjoint of Cholesky
        // run out of registers
        if constexpr (K == FORWARD || K == LOWER) __builtin_amdgcn_sched_barrier(0);
        block_steps<K, KM, CH, J + 1>(kb, c, ring, M, n, z, cur, gv);
    }
}

// One substitution over v (the group's values by row, overwritten by the result).
template <Kind K, int KM, int CH, int LD>
__device__ __forceinline__ void substitute(Matrix M, int n, int blocks, int c, double (*v)[LD])
{
    constexpr bool DOWN = K == UPPER || K == FORWARD;
    Column<KM> ring[AHEAD];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) fetch<K, KM>(ring[s], M, n, s, c);
    double z[CH][KM];
#pragma unroll
    for (int q = 0; q < CH; ++q)
#pragma unroll
        for (int k = 0; k < KM; ++k) z[q][k] = K == FORWARD ? v[q][8 * k + c] : 0.0;
#pragma unroll 1
    for (int kb = 0; kb < blocks; ++kb) {
        const int e = 8 * kb + c, row = DOWN ? e : n - 1 - e;
        double gv[CH], cur[CH];
#pragma unroll
        for (int q = 0; q < CH; ++q) {
            gv[q] = K == FORWARD ? 0.0 : v[q][max(row, 0)];
            cur[q] = 0.0;
            if constexpr (K == FORWARD)
#pragma unroll
                for (int k = 0; k < KM; ++k) cur[q] = k == kb ? z[q][k] : cur[q];
        }
        block_steps<K, KM, CH, 0>(kb, c, ring, M, n, z, cur, gv);
#pragma unroll
        for (int q = 0; q < CH; ++q) {
            if constexpr (K != FORWARD)
#pragma unroll
                for (int k = 0; k < KM; ++k) z[q][k] = k == kb ? cur[q] : z[q][k];
            if (e < n) v[q][row] = cur[q];
        }
    }
}

}  // namespace nrocm_adjoint
