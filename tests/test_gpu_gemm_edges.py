"""Matrix::gemm on column-major operands of any leading dimension and base, from
products of a few tiles to those that fill the chip: the
16-byte loads that run past a tile's rows must neither leave the operands nor let
what lies there reach C (the rows below a view hold NaN here)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _view(rng, rows, cols, ld, off, dt):
    buf = np.full(off + ld * cols, np.nan, dtype=dt)
    M = rng.integers(-4, 5, (rows, cols)).astype(dt)
    for j in range(cols):
        buf[off + j * ld: off + j * ld + rows] = M[:, j]
    # the last column ends the buffer: a load past it would leave the allocation
    return M, torch.from_numpy(buf[: off + (cols - 1) * ld + rows].copy()).cuda()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (3, 5, 2), (31, 64, 33), (32, 128, 32), (33, 65, 100), (100, 100, 100),
                                   (127, 33, 129), (129, 16, 2300), (2047, 47, 300), (1100, 130, 1100),
                                   (17, 257, 15), (16, 1000, 48), (360, 48, 352), (368, 20, 368)])
@pytest.mark.parametrize("pad,off", [(0, 0), (1, 1), (3, 2)])
def test_gemm_any_leading_dimension(nl, dtype, m, k, n, pad, off):
    from nalgebra_amd._lib import lib
    from nalgebra_amd.linalg import handle
    rng = np.random.default_rng(m * 7 + k + n + pad)
    A, a = _view(rng, m, k, m + pad, off, dtype)
    B, b = _view(rng, k, n, k + pad, off, dtype)
    Cm, c = _view(rng, m, n, m + pad, off, dtype)
    es = a.element_size()
    p = lambda t: C.c_void_p(t.data_ptr() + off * es)  # noqa: E731
    fn = lib().nrocm_dgemm if dtype == np.float64 else lib().nrocm_sgemm
    st = fn(handle(), m, k, n, 2.0, p(a), 1, m + pad, p(b), 1, k + pad, -1.0, p(c), 1, m + pad)
    assert st == 0
    got = c.cpu().numpy()
    want = 2.0 * (A.astype(np.float64) @ B.astype(np.float64)) - Cm
    for j in range(n):  # small integers: exact
        assert np.array_equal(got[off + j * (m + pad): off + j * (m + pad) + m], want[:, j].astype(dtype))
        if pad and j + 1 < n:
            assert np.isnan(got[off + j * (m + pad) + m: off + (j + 1) * (m + pad)]).all()
