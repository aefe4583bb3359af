"""LU::new (src/linalg/lu.rs:93-122) as a pipeline of column groups: bitwise and
with identical pivots against the oracle at the edges of the rows per thread and
of the columns per group, wide and tall, with ties, zero columns and NaN, and
above the rows where 64-column panels take over."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _same(x, xr):
    nan = np.isnan(xr)
    x, xr = np.ascontiguousarray(x), np.ascontiguousarray(xr)
    return bool(np.array_equal(np.isnan(x), nan) and np.array_equal(x[~nan].view(np.uint64), xr[~nan].view(np.uint64)))


def _check(nl, orc, A, mode=0):
    lu = nl.DMatrix.from_numpy(A).lu(mode)
    LUr, ipr, infor = orc.getrf(A)
    k = min(A.shape)
    assert np.array_equal(lu.ipiv[:k].cpu().numpy(), ipr), "pivots"
    assert lu.info == infor
    assert _same(lu.lu.numpy(), LUr), "factors"


SHAPES = [(1, 1), (1, 5), (5, 1), (7, 8), (8, 8), (9, 9), (16, 17), (63, 64), (65, 40), (40, 65), (511, 30), (512, 40),
          (513, 41), (300, 700), (1024, 20), (1025, 33), (2048, 24), (2049, 70), (2060, 200), (4097, 66), (8193, 9)]


@pytest.mark.parametrize("m,n", SHAPES)
def test_getrf_shapes(nl, orc, m, n):
    print(f"lu {m} x {n}", flush=True)
    _check(nl, orc, np.asfortranarray(np.random.default_rng(m + n).uniform(-1, 1, (m, n))))


@pytest.mark.parametrize("m,n", [(96, 96), (700, 130), (2100, 90)])
@pytest.mark.parametrize("kind", ["ties", "zerocols", "nan", "permutation"])
def test_getrf_special(nl, orc, kind, m, n):
    rng = np.random.default_rng(m)
    A = rng.uniform(-1, 1, (m, n))
    if kind == "ties":
        A = rng.integers(-2, 3, (m, n)).astype(np.float64)
    elif kind == "zerocols":
        A[:, [0, 9, n // 2, n - 1]] = 0.0
    elif kind == "nan":
        A[m // 2, 3] = np.nan
        A[20, 20] = np.nan
    else:
        A = np.zeros((m, n))
        A[rng.permutation(m)[:n], np.arange(n)] = rng.uniform(1, 2, n)
    _check(nl, orc, np.asfortranarray(A))


def test_getrf_fast_panels(nl, orc):
    """FAST above the one-pipeline size: rank-64 MFMA updates, pivots as EXACT's on random data."""
    n = 2300
    A = np.asfortranarray(np.random.default_rng(1).uniform(-1, 1, (n, n)))
    ex, fa = nl.DMatrix.from_numpy(A).lu(nl.EXACT), nl.DMatrix.from_numpy(A).lu(nl.FAST)
    assert np.array_equal(ex.ipiv.cpu().numpy(), fa.ipiv.cpu().numpy())
    E, F = ex.lu.data, fa.lu.data
    assert float((E - F).norm() / E.norm()) <= 1e-11


def test_getrf_on_two_streams_and_captured(nl, orc):
    mats = [np.random.default_rng(k).uniform(-1, 1, (300, 300)) for k in range(2)]
    ref = [orc.getrf(a) for a in mats]
    dev = [nl.DMatrix.from_numpy(a) for a in mats]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    out = []
    for _ in range(3):
        for a, s in zip(dev, streams):
            with torch.cuda.stream(s):
                out.append(a.lu())
    torch.cuda.synchronize()
    for k, lu in enumerate(out):
        assert _same(lu.lu.numpy(), ref[k % 2][0])
    # a captured factorisation keeps its scratch, whatever is factored later
    buf = nl.DMatrix(torch.empty_like(dev[0].data), 300, 300)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        buf.data.copy_(dev[0].data)
        lu = nl.LU(buf)
    for r in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert _same(lu.lu.numpy(), ref[0][0])
        nl.DMatrix.from_numpy(np.random.default_rng(9).uniform(-1, 1, (1500 + 300 * r, 1500))).lu()
