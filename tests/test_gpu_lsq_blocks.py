"""Batched least squares at the edges of its blocks of 128 rows, panels of 16
columns and splits of a system over wavefronts, against FP64 lstsq."""
import numpy as np
import pytest
import torch

import gen

pytestmark = pytest.mark.gpu

# FP32 Householder QR of well-conditioned systems, and one refinement step in
# FP64 with a residual of 1e-3 (the bounds of the tests of single batches)
BOUND = (1e-4, 1e-7)


def _check(nl, ms, n, scale, sample):
    total = int(ms.sum())
    A = (gen.normal(41 * n, (total * n,)) * scale).astype(np.float32)
    offa = np.concatenate([[0], np.cumsum(ms.astype(np.int64) * n)])
    offb = np.concatenate([[0], np.cumsum(ms.astype(np.int64))])
    noise, x = gen.normal(41 * n + 1, (total,)), gen.normal(41 * n + 2, (len(ms), n))
    mats = [A[offa[j]:offa[j + 1]].reshape(ms[j], n, order="F").astype(np.float64) for j in range(len(ms))]
    b = np.concatenate([M @ x[j] for j, M in enumerate(mats)]) + 1e-3 * scale * noise
    b = b.astype(np.float32)
    bt = nl.LeastSquaresBatch(ms, n)
    Ad, bd = torch.from_numpy(A).cuda(), torch.from_numpy(b).cuda()
    for refine, bound in enumerate(BOUND):
        got, info = bt.solve(Ad, bd, refine)
        got = got.cpu().numpy()
        assert not info.cpu().numpy().any()
        assert np.isfinite(got).all()
        for j in sample:
            want = np.linalg.lstsq(mats[j], b[offb[j]:offb[j + 1]].astype(np.float64), rcond=None)[0]
            err = np.linalg.norm(got[j] - want) / np.linalg.norm(want)
            assert err <= bound, (refine, ms[j], n, err)
    assert np.array_equal(Ad.cpu().numpy(), A) and np.array_equal(bd.cpu().numpy(), b)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 48, 63, 64])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -62, 2.0 ** 50])
def test_block_edges(nl, n, scale):
    ms = np.array([n + 40, 127, 128, 129, 193, 256, 257, 511, 640, 641, 1025, 2047, 2048], dtype=np.int32)
    _check(nl, ms, n, scale, range(len(ms)))


@pytest.mark.parametrize("count", [512, 513, 700, 2047, 2048, 2051])
@pytest.mark.parametrize("n", [5, 40])
def test_splits(nl, n, count):
    ms = np.random.RandomState(count).randint(n + 40, 420, count).astype(np.int32)
    ms[:3] = [2 * n + 60, 128, 300]
    order = np.argsort(-ms, kind="stable")
    _check(nl, ms, n, 1.0, sorted({0, 1, 2, *order[:4].tolist(), *order[-4:].tolist()}))


def test_more_systems_than_one_launch_holds(nl):
    """The records of 250,000 systems exceed what one launch takes."""
    ms = np.full(250000, 3, dtype=np.int32)
    ms[[0, 123456, 249999]] = [300, 200, 129]
    _check(nl, ms, 1, 1.0, [0, 1, 2, 123455, 123456, 123457, 200000, 233000, 234000, 249998, 249999])
