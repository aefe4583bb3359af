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

}  // namespace nrocm_rules
