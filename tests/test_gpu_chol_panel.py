"""Cholesky::new above 64 rows (src/linalg/cholesky.rs:196-272): panels and their
trailing update at the edges of blocks, of the panel's workgroups and of the
update's tiles; pivots and quotients outside the short division's range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spd(n, seed):
    G = np.random.default_rng(seed).standard_normal((n, n))
    return np.asfortranarray(G @ G.T + n * np.eye(n))


def _same(x, xr):
    return np.array_equal(np.ascontiguousarray(x).view(np.uint64), np.ascontiguousarray(xr).view(np.uint64))


@pytest.mark.parametrize("n", [65, 127, 128, 129, 192, 319, 320, 321, 577, 700])
def test_panels_exact(nl, orc, n):
    A = _spd(n, n)
    A[0, n - 1] = 7e7  # the strict upper triangle is not read
    ch = nl.DMatrix.from_numpy(A).cholesky(nl.EXACT)
    Lr, info = orc.potrf(A)
    assert ch is not None and info == 0 and _same(ch.l_dirty().numpy(), Lr)


@pytest.mark.parametrize("scale", [1e-70, 1e70, 1e-290])
def test_panels_extreme_scales(nl, orc, scale):
    """Rows and columns scaled together keep the matrix positive definite while roots and numerators
    leave the range of the three-instruction division."""
    n = 200
    s = np.ones(n)
    s[3::7] = scale ** 0.5
    s[70::31] = scale
    A = np.asfortranarray(_spd(n, 5) * s[:, None] * s[None, :])
    ch = nl.DMatrix.from_numpy(A).cholesky(nl.EXACT)
    Lr, info = orc.potrf(A)
    assert (ch is not None) == (info == 0)
    if info == 0:
        assert _same(np.tril(ch.l_dirty().numpy()), np.tril(Lr))


@pytest.mark.parametrize("n,bad", [(130, 0), (130, 70), (400, 399)])
def test_panels_not_positive_definite(nl, orc, n, bad):
    A = _spd(n, 9)
    A[bad, bad] = -1.0
    assert nl.DMatrix.from_numpy(A).cholesky(nl.EXACT) is None
    sub = nl.Cholesky.new_with_substitute(nl.DMatrix.from_numpy(A), 2.5, nl.EXACT)
    Lr, info = orc.potrf(A, 2.5)
    assert sub is not None and info == 0 and _same(np.tril(sub.l_dirty().numpy()), np.tril(Lr))


def test_panels_fast(nl, orc):
    n = 450
    A = _spd(n, 3)
    L = np.tril(nl.DMatrix.from_numpy(A).cholesky(nl.FAST).l_dirty().numpy())
    assert np.linalg.norm(L @ L.T - A) <= 1e-14 * np.linalg.norm(A)
