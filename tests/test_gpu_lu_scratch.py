"""LU's scratch is two panels of the matrix, not a second matrix."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,mode", [(6000, 6000, 1), (16384, 1000, 0), (2100, 12000, 1)])
def test_scratch_is_bounded(nl, m, n, mode):
    from nalgebra_amd._lib import lib
    L, h = lib(), C.c_void_p()
    assert L.nrocm_create(C.byref(h)) == 0
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    a = torch.rand(m * n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A = a.clone()
    k = min(m, n)
    piv, info = torch.zeros(k, dtype=torch.int32, device="cuda"), torch.ones(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    # the library's code and streams are loaded first
    assert L.nrocm_dgetrf(h, 1100, 70, p(a.clone()), 1100, p(piv), p(info), mode) == 0
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    assert L.nrocm_dgetrf(h, m, n, p(a), m, p(piv), p(info), mode) == 0
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    print(f"lu {m} x {n}: {used >> 20} MiB", flush=True)
    assert int(info.item()) == 0
    # two panels, a quarter more for the next call, and 16 MiB for the graph
    assert used <= 1.25 * 2 * 64 * (m + 1) * 8 + (16 << 20)
    # P A = L U on a vector
    LU = a.view(n, m).t()
    x = torch.rand(n, 1, dtype=torch.float64, device="cuda", generator=g)
    y = torch.triu(LU[:k]) @ x
    y = torch.tril(LU[:, :k], -1) @ y + torch.cat([y, torch.zeros(m - k, 1, dtype=torch.float64, device="cuda")])
    z = (A.view(n, m).t() @ x).cpu().numpy()
    for i, q in enumerate(piv.cpu().numpy()):
        z[[i, q]] = z[[q, i]]
    err = np.abs(z - y.cpu().numpy()).max() / np.abs(z).max()
    assert err <= 1e-11
    assert L.nrocm_destroy(h) == 0
