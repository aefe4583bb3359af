"""The triangular sweeps behind LU::solve_mut, Cholesky::solve_mut and
QR::solve_mut (src/linalg/solve.rs:106-182, 488-519, 697-755; qr.rs:224-256) at
the sizes where their blocking changes: one row block, block and workgroup
edges, every number of right-hand sides per workgroup (1, 2 and 4), and
operands outside the short division's range.  EXACT is bitwise against the
oracle on the same synthetic factors, FAST within 1e-12 relative."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EXACT, FAST = 0, 1


def factors(n, seed, extreme=False):
    """A packed, well-conditioned factor (both triangles filled) and pivots; extreme: a few rows
    scaled so that quotients leave 2^-900..2^600 and divisors leave 2^-100..2^100."""
    rng = np.random.default_rng(seed)
    M = np.asfortranarray(rng.uniform(-0.5, 0.5, (n, n)) / np.sqrt(n))
    d = rng.uniform(1.0, 2.0, n) * np.where(rng.random(n) < 0.5, -1.0, 1.0)
    if extreme:
        d[:: 7] *= 1e-40
        d[3:: 11] *= 1e45
    M[np.arange(n), np.arange(n)] = d
    ipiv = np.array([rng.integers(i, n) if rng.random() < 0.7 else i for i in range(n)], dtype=np.int32)
    return M, ipiv


def rhs(n, nrhs, seed, extreme=False):
    B = np.random.default_rng(seed).standard_normal((n, nrhs))
    if extreme:
        B[::5] *= 1e-290
        B[1::9] = 0.0
        B[2::13] = -0.0
    return B


def _dev(a):
    return torch.from_numpy(np.asfortranarray(a).ravel(order="F").copy()).cuda()


def _p(t):
    return C.c_void_p(t.data_ptr())


def _call(nl, op, M, B, mode, ipiv=None, diag=None):
    from nalgebra_amd._lib import lib
    from nalgebra_amd.linalg import handle
    n, nrhs = B.shape
    m, b = _dev(M), _dev(B)
    info = torch.full((1,), 77, dtype=torch.int32, device="cuda")
    if op == "lu":
        piv = torch.from_numpy(ipiv).cuda()
        st = lib().nrocm_dgetrs(handle(), n, nrhs, _p(m), n, _p(piv), _p(b), n, _p(info), mode)
    elif op == "noalloc":
        piv = torch.from_numpy(ipiv).cuda()
        st = lib().nrocm_dgetrs_noalloc(handle(), n, nrhs, _p(m), n, _p(piv), _p(b), n, _p(info), mode)
    elif op == "chol":
        st = lib().nrocm_dpotrs(handle(), n, nrhs, _p(m), n, _p(b), n, mode)
    else:
        dg = torch.from_numpy(diag).cuda()
        st = lib().nrocm_dqr_rsolve(handle(), n, _p(m), n, _p(dg), nrhs, _p(b), n, _p(info))
    assert st == 0, st
    torch.cuda.synchronize()
    return b.cpu().numpy().reshape(nrhs, n).T, int(info.item())


def _same(x, xr):
    """Equal bits; NaNs at the same places (the sign of a NaN made of two NaN operands is left open)."""
    nan = np.isnan(xr)
    return bool(np.array_equal(np.isnan(x), nan) and np.array_equal(x[~nan].view(np.uint64), xr[~nan].view(np.uint64)))


@pytest.mark.parametrize("extreme", [False, True])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (3, 2), (63, 1), (64, 3), (65, 1), (128, 2), (257, 5), (449, 1), (1023, 3),
                                    (100, 300), (70, 600), (1024, 5), (1500, 60), (1100, 140)])
def test_sweeps_exact(nl, orc, n, nrhs, extreme):
    print(f"sweeps n={n} nrhs={nrhs} extreme={extreme}", flush=True)
    M, ipiv = factors(n, 40 + n, extreme)
    B = rhs(n, nrhs, n + nrhs, extreme)
    x, info = _call(nl, "lu", M, B, EXACT, ipiv=ipiv)
    xr, ok = orc.getrs(M, ipiv, B)
    assert ok and info == 0 and _same(x, xr)
    Lm = M.copy()
    Lm[np.arange(n), np.arange(n)] = np.abs(M.diagonal())
    assert _same(_call(nl, "chol", Lm, B, EXACT)[0], orc.potrs(Lm, B))
    diag = M.diagonal().copy()
    x, info = _call(nl, "qr", M, B, EXACT, diag=diag)
    xr, ok = orc.qr_rsolve(M, diag, B)
    assert ok and info == 0 and _same(x, xr)


@pytest.mark.parametrize("n,nrhs", [(64, 1), (200, 2), (1030, 1), (80, 600)])
def test_sweeps_row_scaling(nl, orc, n, nrhs):
    """Rows of the factor and of b scaled together: every x stays ordinary while numerators and
    divisors leave the short division's range."""
    M, _ = factors(n, 20 + n)
    ipiv = np.arange(n, dtype=np.int32)
    s = np.ones(n)
    s[::7], s[3::11], s[5::13] = 1e-40, 1e-290, 1e200
    U = np.asfortranarray(np.triu(M) * s[:, None])
    B = rhs(n, nrhs, n) * s[:, None]
    x, info = _call(nl, "lu", U, B, EXACT, ipiv=ipiv)
    xr, ok = orc.getrs(U, ipiv, B)
    assert ok and info == 0 and np.isfinite(xr).all() and _same(x, xr)
    x, _ = _call(nl, "qr", U, B, EXACT, diag=U.diagonal().copy())
    assert _same(x, orc.qr_rsolve(U, U.diagonal().copy(), B)[0])


@pytest.mark.parametrize("n,nrhs", [(1, 1), (64, 1), (65, 2), (300, 4), (1023, 1), (90, 520), (1025, 2), (1300, 90)])
def test_sweeps_fast(nl, orc, n, nrhs):
    M, ipiv = factors(n, 60 + n)
    B = rhs(n, nrhs, n + nrhs)
    x, info = _call(nl, "lu", M, B, FAST, ipiv=ipiv)
    xr, _ = orc.getrs(M, ipiv, B)
    assert info == 0 and np.linalg.norm(x - xr) <= 1e-12 * np.linalg.norm(xr)
    Lm = M.copy()
    Lm[np.arange(n), np.arange(n)] = np.abs(M.diagonal())
    x, _ = _call(nl, "chol", Lm, B, FAST)
    xr = orc.potrs(Lm, B)
    assert np.linalg.norm(x - xr) <= 1e-12 * np.linalg.norm(xr)


@pytest.mark.parametrize("n,nrhs", [(200, 9), (3000, 7), (7000, 3)])
def test_noalloc_chunks(nl, orc, n, nrhs):
    """The static scratch takes several right-hand sides at a time while it holds their tags."""
    M, ipiv = factors(n, 80 + n)
    B = rhs(n, nrhs, n)
    x, info = _call(nl, "noalloc", M, B, EXACT, ipiv=ipiv)
    xr, _ = orc.getrs(M, ipiv, B)
    assert info == 0 and _same(x, xr)


def test_zero_diagonal_and_empty(nl, orc):
    n = 500
    M, ipiv = factors(n, 5)
    M[70, 70], M[400, 400] = 0.0, -0.0
    assert _call(nl, "lu", M, np.ones((n, 2)), EXACT, ipiv=ipiv)[1] == 401
    assert _call(nl, "qr", M, np.ones((n, 1)), EXACT, diag=M.diagonal().copy())[1] == 401
    assert _call(nl, "lu", M, np.ones((n, 0)), EXACT, ipiv=ipiv)[1] == 0


def test_qr_rsolve_beyond_one_workgroup(nl, orc):
    """x no longer fits one workgroup's LDS: the solve moves to many workgroups."""
    n = 12200
    M, _ = factors(n, 7)
    diag = M.diagonal().copy()
    B = rhs(n, 1, 8)
    print("qr rsolve n=12200", flush=True)
    x, info = _call(nl, "qr", M, B, EXACT, diag=diag)
    xr, ok = orc.qr_rsolve(M, diag, B)
    assert ok and info == 0 and _same(x, xr)
