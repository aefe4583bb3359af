"""QR::solve_mut's upper solve on both sides of the size where x no longer fits the
LDS of one workgroup and the sweep moves to many, bit for bit the oracle's."""
import numpy as np
import pytest

from test_gpu_solve_sweeps import EXACT, _call, _same, factors, rhs

pytestmark = pytest.mark.gpu

# a workgroup's 160 KB less a few words, two staged 64 x 64 blocks, x in rows of 64
MOST = ((160 * 1024 - 64) // 8 - 2 * 64 * 64) // 64 * 64


def test_bound():
    assert MOST == 12224


@pytest.mark.parametrize("n,nrhs", [(MOST, 1), (MOST + 1, 1), (12300, 3)])
def test_either_side(nl, orc, n, nrhs):
    M, _ = factors(n, 7)
    diag = M.diagonal().copy()
    B = rhs(n, nrhs, 8)
    print(f"qr rsolve n={n} nrhs={nrhs}", flush=True)
    x, info = _call(nl, "qr", M, B, EXACT, diag=diag)
    xr, ok = orc.qr_rsolve(M, diag, B)
    assert ok and info == 0 and _same(x, xr)
    # a zero on the diagonal, in a workgroup that others wait for: the largest index
    diag[[4000, n - 700]] = 0.0
    assert _call(nl, "qr", M, B, EXACT, diag=diag)[1] == n - 700 + 1
