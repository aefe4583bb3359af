"""Waits between workgroups that run out (a bound of one poll, which every kernel
leaves normally) are reported: info = -1, or NaN where there is no info.  The
next call of the handle with the usual bounds is unaffected."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.fixture()
def own(nl):
    """A handle of its own on the null stream, and its library."""
    from nalgebra_amd._lib import lib
    L, h = lib(), C.c_void_p()
    assert L.nrocm_create(C.byref(h)) == 0
    yield L, h
    assert L.nrocm_destroy(h) == 0


def _twice(own, call):
    """call() with one poll per wait, then with the usual bounds."""
    L, h = own
    res = []
    for polls in (1, 0):
        assert L.nrocm_set_wait_limit(h, polls) == 0
        torch.cuda.synchronize()
        res.append(call())
        torch.cuda.synchronize()
    return res


def _i32(n):
    return torch.zeros(n, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("m,n,mode", [(500, 500, 0), (1000, 120, 0), (1500, 300, 0), (1500, 300, 1), (2100, 60, 0)])
def test_lu(own, orc, m, n, mode):
    L, h = own
    A = np.asfortranarray(np.random.default_rng(m + n).uniform(-1, 1, (m, n)))
    print(f"lu {m} x {n} mode {mode}", flush=True)

    def call():
        a = torch.from_numpy(A.ravel(order="F").copy()).cuda()
        piv, info = _i32(n), _i32(1)
        torch.cuda.synchronize()
        assert L.nrocm_dgetrf(h, m, n, _ptr(a), m, _ptr(piv), _ptr(info), mode) == 0
        torch.cuda.synchronize()
        return a.cpu().numpy().reshape(n, m).T, piv.cpu().numpy(), int(info.item())
    (_, piv, info), (lu, piv2, info2) = _twice(own, call)
    assert info == -1
    assert (piv >= 0).all() and (piv < m).all()
    ref, pivr, infor = orc.getrf(A)
    assert info2 == infor and np.array_equal(piv2, pivr)
    if mode == 0:
        assert np.array_equal(np.ascontiguousarray(lu).view(np.uint64), np.ascontiguousarray(ref).view(np.uint64))


@pytest.mark.parametrize("m,n,dtype", [(600, 64, np.float64), (1500, 30, np.float64), (700, 50, np.float32)])
def test_qr(own, m, n, dtype):
    L, h = own
    A = np.random.default_rng(m + n).uniform(-1, 1, m * n).astype(dtype)
    print(f"qr {m} x {n}", flush=True)

    def call():
        a = torch.from_numpy(A.copy()).cuda()
        d = torch.zeros(n, dtype=a.dtype, device="cuda")
        torch.cuda.synchronize()
        fn = L.nrocm_dgeqrf if dtype == np.float64 else L.nrocm_sgeqrf
        assert fn(h, m, n, _ptr(a), m, _ptr(d)) == 0
        torch.cuda.synchronize()
        return d.cpu().numpy()
    lost, d = _twice(own, call)
    assert np.isnan(lost[-1])
    R = np.linalg.qr(A.reshape(n, m).T.astype(np.float64), mode="r")
    assert np.allclose(np.abs(d), np.abs(R.diagonal()), rtol=1e-10 if dtype == np.float64 else 1e-4)


@pytest.mark.parametrize("kind", ["lu", "chol"])
@pytest.mark.parametrize("n,nrhs,mode", [(1100, 1, 0), (1100, 3, 1), (3000, 2, 1)])
def test_solves(own, orc, kind, n, nrhs, mode):
    L, h = own
    rng = np.random.default_rng(n + nrhs)
    M = np.asfortranarray(rng.uniform(-1, 1, (n, n)) / n)
    M[np.arange(n), np.arange(n)] = 1.0 + rng.uniform(0, 1, n)
    B = np.asfortranarray(rng.uniform(-1, 1, (n, nrhs)))
    a, piv = torch.from_numpy(M.ravel(order="F").copy()).cuda(), torch.arange(n, dtype=torch.int32, device="cuda")
    print(f"solve {kind} {n} x {nrhs} mode {mode}", flush=True)

    def call():
        b, info = torch.from_numpy(B.ravel(order="F").copy()).cuda(), _i32(1)
        torch.cuda.synchronize()
        if kind == "lu":
            assert L.nrocm_dgetrs(h, n, nrhs, _ptr(a), n, _ptr(piv), _ptr(b), n, _ptr(info), mode) == 0
        else:
            assert L.nrocm_dpotrs(h, n, nrhs, _ptr(a), n, _ptr(b), n, mode) == 0
        torch.cuda.synchronize()
        return b.cpu().numpy().reshape(nrhs, n).T, int(info.item())
    (lost, info), (x, info2) = _twice(own, call)
    assert np.isnan(lost).any(axis=0).all()
    assert info == (-1 if kind == "lu" else 0) and info2 == 0
    ref = orc.getrs(M, np.arange(n, dtype=np.int32), B)[0] if kind == "lu" else orc.potrs(M, B)
    assert np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref)


def test_arguments(own):
    L, h = own
    assert L.nrocm_set_wait_limit(None, 1) == -1
    assert L.nrocm_set_wait_limit(h, -1) == -2
