"""QR::new and its products as a pipeline of columns (src/linalg/qr.rs:55-76,
108-129, 157-171; householder.rs:19-85): bitwise against the oracle at the
edges of the rows per thread and of the columns per workgroup, wide and tall,
in f64 and f32, with columns that need no reflection."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _same(x, xr):
    nan = np.isnan(xr)
    w = np.uint64 if xr.dtype == np.float64 else np.uint32
    x, xr = np.ascontiguousarray(x), np.ascontiguousarray(xr)
    return bool(np.array_equal(np.isnan(x), nan) and np.array_equal(x[~nan].view(w), xr[~nan].view(w)))


SHAPES = [(1, 1), (5, 3), (8, 4), (9, 5), (16, 16), (40, 90), (511, 7), (512, 33), (513, 9), (700, 300), (1025, 6),
          (2049, 5), (4097, 3), (8200, 2)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", SHAPES)
def test_geqrf_bitwise(nl, orc, m, n, dtype):
    print(f"qr {m} x {n} {dtype.__name__}", flush=True)
    A = np.asfortranarray(np.random.default_rng(m + n).uniform(-1, 1, (m, n)).astype(dtype))
    qr = nl.DMatrix.from_numpy(A).qr()
    QRr, dr = orc.geqrf(A)
    assert _same(qr.diag.cpu().numpy()[:min(m, n)], dr)
    assert _same(qr.qr.numpy(), QRr)


@pytest.mark.parametrize("kind", ["zerocols", "tiny", "nan"])
def test_geqrf_special_columns(nl, orc, kind):
    """A zero column makes no reflector; norms outside the short division's range; a NaN column."""
    m, n = 600, 13
    A = np.random.default_rng(3).uniform(-1, 1, (m, n))
    if kind == "zerocols":
        A[:, [2, 3, 9]] = 0.0
    elif kind == "tiny":
        A[:, 1] *= 1e-150
        A[:, 6] *= 1e120
    else:
        A[40, 5] = np.nan
    qr = nl.DMatrix.from_numpy(A).qr()
    QRr, dr = orc.geqrf(A)
    assert _same(qr.diag.cpu().numpy(), dr) and _same(qr.qr.numpy(), QRr)


@pytest.mark.parametrize("m,n,nrhs", [(1, 1, 1), (17, 9, 3), (513, 20, 2), (1030, 12, 300), (2050, 7, 5), (9000, 3, 2)])
def test_qr_products(nl, orc, m, n, nrhs):
    rng = np.random.default_rng(m + nrhs)
    A = np.asfortranarray(rng.uniform(-1, 1, (m, n)))
    B = rng.uniform(-1, 1, (m, nrhs))
    QRr, dr = orc.geqrf(A)
    qr = nl.DMatrix.from_numpy(A).qr()
    y = nl.DMatrix.from_numpy(B)
    qr.q_tr_mul(y)
    assert _same(y.numpy(), orc.qr_qtmul(QRr, dr, B))
    z = nl.DMatrix.from_numpy(B)
    qr.q_mul(z)
    assert _same(z.numpy(), orc.qr_qmul(QRr, dr, B))


def test_qr_on_two_streams(nl, orc):
    """Calls on two streams share the handle's workspace one after the other."""
    mats = [np.random.default_rng(k).uniform(-1, 1, (700, 60)) for k in range(2)]
    dev = [nl.DMatrix.from_numpy(a) for a in mats]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    out = []
    for rep in range(3):
        for a, s in zip(dev, streams):
            with torch.cuda.stream(s):
                out.append(a.qr())
    torch.cuda.synchronize()
    for k, qr in enumerate(out):
        QRr, dr = orc.geqrf(mats[k % 2])
        assert _same(qr.qr.numpy(), QRr) and _same(qr.diag.cpu().numpy(), dr)


def test_qr_under_capture(nl, orc):
    """A captured QR uses no workspace: replays agree with the eager result."""
    A = np.random.default_rng(9).uniform(-1, 1, (150, 20))
    QRr, _ = orc.geqrf(A)
    src = nl.DMatrix.from_numpy(A)
    buf = nl.DMatrix(torch.empty_like(src.data), 150, 20)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        buf.data.copy_(src.data)
        qr = nl.QR(buf)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert _same(qr.qr.numpy(), QRr)
        nl.DMatrix.from_numpy(np.random.default_rng(1).uniform(-1, 1, (900, 200))).qr()
