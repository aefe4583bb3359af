"""Solves of up to eight rows, a right-hand side per thread: bit for bit the oracle's
(nalgebra's order), swaps, zero diagonals, NaN and more right-hand sides than a
wavefront included, on both sides of the size where the sweeps begin."""
import numpy as np
import pytest

from test_gpu_solve_sweeps import EXACT, FAST, _call, _same, factors, rhs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 8, 9])
@pytest.mark.parametrize("nrhs", [1, 3, 64, 65, 200])
def test_tiny(nl, orc, n, nrhs):
    M, ipiv = factors(n, 30 + n)
    B = rhs(n, nrhs, n + nrhs)
    x, info = _call(nl, "lu", M, B, EXACT, ipiv=ipiv)
    assert info == 0 and _same(x, orc.getrs(M, ipiv, B)[0])
    x, info = _call(nl, "qr", M, B, EXACT, diag=M.diagonal().copy())
    assert info == 0 and _same(x, orc.qr_rsolve(M, M.diagonal().copy(), B)[0])
    L = M.copy()
    L[np.arange(n), np.arange(n)] = np.abs(M.diagonal())
    assert _same(_call(nl, "chol", L, B, EXACT)[0], orc.potrs(L, B))
    for kind, ref in (("lu", orc.getrs(M, ipiv, B)[0]), ("chol", orc.potrs(L, B))):
        x, _ = _call(nl, kind, M if kind == "lu" else L, B, FAST, ipiv=ipiv)
        assert np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [2, 6, 8])
def test_tiny_special(nl, orc, n):
    M, ipiv = factors(n, 50 + n)
    B = rhs(n, 4, n)
    B[0, 1], B[n - 1, 2], B[n // 2, 3] = np.nan, np.inf, -0.0
    with np.errstate(all="ignore"):
        assert _same(_call(nl, "lu", M, B, EXACT, ipiv=ipiv)[0], orc.getrs(M, ipiv, B)[0])
        L = M.copy()
        L[np.arange(n), np.arange(n)] = np.abs(M.diagonal())
        assert _same(_call(nl, "chol", L, B, EXACT)[0], orc.potrs(L, B))
    M[0, 0] = 0.0
    assert _call(nl, "lu", M, B, EXACT, ipiv=ipiv)[1] == 1
    M[n - 1, n - 1] = -0.0
    assert _call(nl, "lu", M, B, EXACT, ipiv=ipiv)[1] == n
    assert _call(nl, "qr", M, B, EXACT, diag=M.diagonal().copy())[1] == n
    assert _call(nl, "lu", M, np.ones((n, 0)), EXACT, ipiv=ipiv)[1] == 0
