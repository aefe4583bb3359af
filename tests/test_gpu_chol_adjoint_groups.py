"""Adjoint of the batched Cholesky solve with eight members to a wavefront: every
member bit for bit against the oracle's, where members of different sizes (and
empty ones) share a wavefront, the last one is not full, and the batch lies on
either side of the 32-row limit."""
import numpy as np
import pytest
import torch

import gen

pytestmark = pytest.mark.gpu


def _same(x, y):  # NaNs compare as NaNs
    ok = ~np.isnan(y)
    return np.array_equal(np.isnan(x), ~ok) and np.array_equal(x[ok].view(np.uint64), y[ok].view(np.uint64))


@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("ns", [[1], [32] * 9, [33, 1, 0, 8], [0, 5, 0, 3, 9, 17, 24, 25, 31, 32, 16, 15, 2, 1],
                                list(range(64, 0, -1)) + [64] * 5, [64, 8, 8, 8, 8, 8, 8, 8, 7]])
@pytest.mark.parametrize("special", [False, True])
def test_adjoint_bitwise(nl, orc, ns, nrhs, special):
    A, offA, B, offB = gen.spd_batch(61 + nrhs, ns, nrhs)
    bt = nl.CholeskyBatch(ns, nrhs)
    Ad, Bd = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    assert not bt.solve(Ad, Bd, nl.EXACT).cpu().numpy().any()
    dX = np.zeros_like(B)
    for j, n in enumerate(ns):
        dX[offB[j]:offB[j] + n * nrhs] = gen.normal(700 + j, (n * nrhs,))
    if special:  # infinities and NaNs stay inside their own member
        dX[::97] = np.inf
        dX[3::101] = np.nan
        dX[5::13] = -0.0
    dA, dB = bt.backward(Ad, Bd, torch.from_numpy(dX).cuda())
    dA, dB, Lh, Xh = dA.cpu().numpy(), dB.cpu().numpy(), Ad.cpu().numpy(), Bd.cpu().numpy()
    with np.errstate(all="ignore"):
        for j, n in enumerate(ns):
            if n == 0:
                continue
            L = Lh[offA[j]:offA[j] + n * n].reshape(n, n, order="F")
            X = Xh[offB[j]:offB[j] + n * nrhs].reshape(n, nrhs, order="F")
            G = dX[offB[j]:offB[j] + n * nrhs].reshape(n, nrhs, order="F")
            got = dB[offB[j]:offB[j] + n * nrhs].reshape(n, nrhs, order="F")
            total = None
            for q in range(nrhs):
                dAq, dBq = orc.potrs_adjoint(L, X[:, q], G[:, q])
                assert _same(got[:, q].copy(), np.ascontiguousarray(dBq).ravel()), (j, n, q)
                total = dAq if total is None else total + dAq
            assert _same(dA[offA[j]:offA[j] + n * n], total.ravel(order="F")), (j, n)
