"""Batched least squares: accuracy of long systems after a refinement, columns and
rows whose squares leave the range of a float, zero columns, NaN and infinities."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _solve(nl, mats, bs, refine):
    ms = [M.shape[0] for M in mats]
    bt = nl.LeastSquaresBatch(ms, mats[0].shape[1])
    A = torch.from_numpy(np.concatenate([M.ravel(order="F") for M in mats])).cuda()
    x, info = bt.solve(A, torch.from_numpy(np.concatenate(bs)).cuda(), refine)
    return x.cpu().numpy(), info.cpu().numpy()


@pytest.mark.parametrize("count", [64, 700, 2100])  # four, two and one wavefront to a system
def test_long_systems_accuracy(nl, count):
    """With a residual of standard deviation s, the error that a refinement leaves is
    that of the factors: entries N(0, 1) rounded once per update of a column, 3.5
    times in the mean for n = 8, give 0.58 * 2^-24 * sqrt(3.5) * s / sqrt(m) relative to
    x.  Twice that."""
    n, lo, hi, s, sample = 8, 1900, 2048, 1e-2, 64
    ms = np.random.RandomState(count).randint(lo, hi + 1, count).astype(np.int32)
    g = torch.Generator(device="cuda")
    g.manual_seed(count)
    A = torch.randn(int(ms.sum()) * n, generator=g, device="cuda")
    noise = torch.randn(int(ms.sum()), generator=g, device="cuda").cpu().numpy() * s
    Ah, off = A.cpu().numpy().astype(np.float64), np.concatenate([[0], np.cumsum(ms.astype(np.int64))])
    b = np.empty(len(noise), dtype=np.float32)
    rng, mats = np.random.default_rng(count), []
    for j in range(count):
        M = Ah[off[j] * n: off[j + 1] * n].reshape(n, ms[j]).T
        b[off[j]: off[j + 1]] = M @ rng.standard_normal(n) + noise[off[j]: off[j + 1]]
        mats.append(M)
    x, info = nl.LeastSquaresBatch(ms, n).solve(A, torch.from_numpy(b).cuda(), 1)
    assert not info.cpu().numpy().any()
    x, err = x.cpu().numpy(), []
    for j in range(0, count, count // sample):
        want = np.linalg.lstsq(mats[j], b[off[j]: off[j + 1]].astype(np.float64), rcond=None)[0]
        err.append(np.linalg.norm(x[j] - want) / np.linalg.norm(want))
    rms = float(np.sqrt(np.mean(np.square(err))))
    print(f"count {count}: rms error {rms:.2e}", flush=True)
    assert rms <= 2 * 0.58 * 2.0 ** -24 * np.sqrt(3.5) * s / np.sqrt((lo + hi) / 2)


@pytest.mark.parametrize("value", [1e-25, 1e-38, -1e-30, 1e25, 3.0])
def test_one_by_one(nl, value):
    x, info = _solve(nl, [np.array([[value]], dtype=np.float32)], [np.array([2.0], dtype=np.float32)], 1)
    want = 2.0 / float(np.float32(value))
    assert info[0] == 0 and abs(x[0, 0] - want) <= 1e-7 * abs(want)


@pytest.mark.parametrize("n,extra", [(7, 0), (20, 30), (40, 300)])
def test_graded_triangle(nl, n, extra):
    """Rows from 1 down to 1e-25, zero rows below: x is determined by rows whose squares vanish."""
    rng = np.random.default_rng(n)
    U = np.triu(rng.uniform(0.5, 1.0, (n, n))) * np.logspace(0, -25, n)[:, None]
    U[np.arange(n), np.arange(n)] *= 4.0
    A = np.vstack([U, np.zeros((extra, n))]).astype(np.float32)
    b = (A.astype(np.float64) @ rng.uniform(1, 2, n)).astype(np.float32)
    want = np.linalg.solve(A[:n].astype(np.float64), b[:n].astype(np.float64))
    for refine, bound in ((0, 1e-4), (1, 1e-7)):
        x, info = _solve(nl, [A], [b], refine)
        assert info[0] == 0
        assert np.linalg.norm(x[0] - want) <= bound * np.linalg.norm(want), refine


@pytest.mark.parametrize("m,n", [(60, 6), (300, 24), (700, 64)])
def test_columns_of_any_scale(nl, m, n):
    rng = np.random.default_rng(m)
    k = rng.permutation(np.linspace(-90, 90, n).round()).astype(int)
    A = (rng.standard_normal((m, n)) * 2.0 ** k).astype(np.float32)
    b = (A.astype(np.float64) @ (rng.standard_normal(n) * 2.0 ** -k) + 1e-3 * rng.standard_normal(m)).astype(np.float32)
    want = np.linalg.lstsq(A.astype(np.float64) * 2.0 ** -k, b.astype(np.float64), rcond=None)[0]
    for refine, bound in ((0, 1e-4), (1, 1e-7)):
        x, info = _solve(nl, [A], [b], refine)
        assert info[0] == 0
        assert np.linalg.norm(x[0] * 2.0 ** k - want) <= bound * np.linalg.norm(want), refine


@pytest.mark.parametrize("n", [1, 5, 33])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_not_finite(nl, n, value):
    """The system has no finite solution and says so by NaN, not by info; its neighbours are unaffected."""
    rng = np.random.default_rng(n)
    mats = [rng.standard_normal((m, n)).astype(np.float32) for m in (90, 300, 90)]
    bs = [rng.standard_normal(M.shape[0]).astype(np.float32) for M in mats]
    want, _ = _solve(nl, mats, bs, 1)
    mats[1][200, n // 2] = value
    x, info = _solve(nl, mats, bs, 1)
    assert np.isnan(x[1]).any() and not info.any()
    assert np.array_equal(x[[0, 2]], want[[0, 2]])


@pytest.mark.parametrize("n,zero", [(1, [0]), (6, [2]), (40, [3, 17, 31])])
def test_zero_columns(nl, n, zero):
    A = np.random.default_rng(n).standard_normal((200, n)).astype(np.float32)
    A[:, zero] = 0.0
    _, info = _solve(nl, [A], [np.ones(200, dtype=np.float32)], 1)
    assert info[0] == zero[-1] + 1
