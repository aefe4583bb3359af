// Index rules of kernels whose loads run past what they use: plain functions, so
// that they can be checked exhaustively without a GPU.
#pragma once

#ifdef __HIPCC__
#define NROCM_RULE __host__ __device__ constexpr
#else
#define NROCM_RULE constexpr
#endif

namespace nrocm_rules {

// gemm_cm_kernel: may the slice of columns [k0, k0 + bk) of A (m x k, column
// stride lda) be fetched for the rows [bm, bm + tile) with wide loads?  Rows past
// m are not used; they are read if every load ends inside A's last column.  With
// lda < m (columns that overlap, or lie in decreasing order) the last column is
// not the last in memory.
NROCM_RULE bool gemm_wide_slice(long m, long k, long lda, long bm, long tile, long k0, long bk)
{
    return k0 + bk <= k && (bm + tile <= m || (lda >= m && bm + tile + (k0 + bk - 1) * lda <= m + (k - 1) * lda));
}

// chol_dot_backward: the loading wavefronts make the products of phase p (row
// n - 1 - p, elements x[n - p + e], e < p) for p = 0 .. dot_last_phase(n), whole
// rounds of DOT_AHEAD phases that begin two phases ahead.  Element e reads row
// dot_first_row + min(e, dot_last_element), a row of x also where the phase has no
// such element (e >= p), none at all (p = 0) or is past the last row (p >= n).
constexpr int DOT_AHEAD = 4;
NROCM_RULE int dot_last_phase(int n) { return (n + DOT_AHEAD - 1) / DOT_AHEAD * DOT_AHEAD + 1; }
NROCM_RULE int dot_first_row(int n, int p) { return p < n ? n - p : 0; }
NROCM_RULE int dot_last_element(int n, int p) { return n - 1 - dot_first_row(n, p); }

}  // namespace nrocm_rules
