"""Adjoint of the batched LU solve with eight members to a wavefront: every
member bit for bit against the oracle's transposed solves, where members of
different sizes (and empty ones) share a wavefront, the last one is not full,
and the batch lies on either side of the 32-row limit."""
import numpy as np
import pytest
import torch

import gen
from test_gpu_lu_batched import _bits, make_batch, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrhs", [1, 2, 3, 5])
@pytest.mark.parametrize("ns", [[1], [32] * 9, [33, 1, 0, 8], [0, 5, 0, 3, 9, 17, 24, 25, 31, 32, 16, 15, 2, 1],
                                list(range(64, 0, -1)) + [64] * 5, [64, 8, 8, 8, 8, 8, 8, 8, 7]])
@pytest.mark.parametrize("special", [False, True])
def test_adjoint_bitwise(nl, orc, ns, nrhs, special):
    ns, A, offA, B, offB = make_batch(ns, nrhs, 17 + nrhs)
    bt, Ag, Bg, Pg, info = run(nl, ns, A, B, nrhs, nl.EXACT)
    assert not info.any()
    dX = np.zeros_like(B)
    for j, n in enumerate(ns):
        dX[offB[j]:offB[j] + n * nrhs] = gen.normal(900 + j, (n * nrhs,))
    if special and dX.size:  # infinities and NaNs stay inside their own dots
        dX[:: 7] = np.inf
        dX[3:: 11] = np.nan
        dX[5:: 13] = -0.0
    dA, dB = bt.backward(*(torch.from_numpy(x).cuda() for x in (Ag, Pg, Bg, dX)))
    dA = dA.cpu().numpy(); dB = dB.cpu().numpy()

    def same(x, y):  # NaNs compare as NaNs (the sign of a NaN made from two NaNs is left open)
        return np.array_equal(np.isnan(x), np.isnan(y)) and np.array_equal(_bits(x[~np.isnan(y)]), _bits(y[~np.isnan(y)]))

    with np.errstate(all="ignore"):
        for j, n in enumerate(ns):
            if n == 0:
                continue
            LU = Ag[offA[j]:offA[j] + n * n].reshape(n, n, order="F")
            X = Bg[offB[j]:offB[j] + n * nrhs].reshape(n, nrhs, order="F")
            G = dX[offB[j]:offB[j] + n * nrhs].reshape(n, nrhs, order="F")
            dAr, dBr, ok = orc.getrs_adjoint(LU, Pg[bt.offP[j]:bt.offP[j] + n], X, G)
            assert ok
            assert same(dB[offB[j]:offB[j] + n * nrhs], dBr.ravel(order="F")), (j, n)
            assert same(dA[offA[j]:offA[j] + n * n], dAr.ravel(order="F")), (j, n)
