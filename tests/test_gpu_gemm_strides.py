"""Matrix::gemm with columns in decreasing order and overlapping columns (element
strides are signed, src/base/blas_uninit.rs:276-313), from products of a few
tiles to those of the wide-load kernel, ragged edges included."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,k,n", [(5, 7, 3), (100, 100, 100), (368, 40, 371), (370, 128, 370), (1100, 96, 1031)])
@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("rev", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)])
def test_gemm_columns_in_decreasing_order(nl, dtype, m, k, n, pad, rev):
    from nalgebra_amd._lib import lib
    from nalgebra_amd.linalg import handle
    rng = np.random.default_rng(m + k + n + pad)
    mats, ptrs, strides, keep = [], [], [], []
    for (rows, cols), r in zip(((m, k), (k, n), (m, n)), rev):
        M = rng.integers(-4, 5, (rows, cols)).astype(dtype)
        ld = rows + pad
        buf = np.full(ld * (cols - 1) + rows, np.nan, dtype=dtype)  # ends with the last column
        for j in range(cols):
            buf[j * ld: j * ld + rows] = M[:, cols - 1 - j if r else j]
        t = torch.from_numpy(buf).cuda()
        keep.append((t, ld, r))
        ptrs.append(C.c_void_p(t.data_ptr() + (ld * (cols - 1) * t.element_size() if r else 0)))
        strides.append(-ld if r else ld)
        mats.append(M.astype(np.float64))
    print(f"gemm {m} {k} {n} pad {pad} reversed {rev}", flush=True)
    fn = lib().nrocm_dgemm if dtype == np.float64 else lib().nrocm_sgemm
    assert fn(handle(), m, k, n, 2.0, ptrs[0], 1, strides[0], ptrs[1], 1, strides[1], -1.0, ptrs[2], 1, strides[2]) == 0
    want = 2.0 * (mats[0] @ mats[1]) - mats[2]
    t, ld, r = keep[2]
    got = t.cpu().numpy()
    for j in range(n):
        at = (n - 1 - j if r else j) * ld
        assert np.array_equal(got[at: at + m], want[:, j].astype(dtype))


@pytest.mark.parametrize("lda", [0, 1, 7])
def test_gemm_overlapping_columns(nl, lda):
    """Columns lda apart, less than their length: a Hankel matrix, or one column repeated."""
    from nalgebra_amd._lib import lib
    from nalgebra_amd.linalg import handle
    m, k, n = 400, 100, 400
    rng = np.random.default_rng(lda)
    buf = rng.integers(-4, 5, m + lda * (k - 1)).astype(np.float64)
    A = np.stack([buf[j * lda: j * lda + m] for j in range(k)], axis=1)
    B = rng.integers(-4, 5, (k, n)).astype(np.float64)
    a, b = torch.from_numpy(buf).cuda(), torch.from_numpy(B.ravel(order="F").copy()).cuda()
    c = torch.zeros(m * n, dtype=torch.float64, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    assert lib().nrocm_dgemm(handle(), m, k, n, 1.0, p(a), 1, lda, p(b), 1, k, 0.0, p(c), 1, m) == 0
    assert np.array_equal(c.cpu().numpy().reshape(n, m).T, A @ B)
