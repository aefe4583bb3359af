"""Batched adjoints with one, two, four and eight members to a wavefront (by the
count): every member bit for bit as in a batch of a few."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1023, 1024, 1025, 2049, 4097, 8193, 9000])
@pytest.mark.parametrize("kind", ["chol", "lu"])
@pytest.mark.parametrize("hi,nrhs", [(9, 1), (9, 3), (34, 2)])
def test_members_per_wavefront(nl, kind, count, hi, nrhs):
    rng = np.random.default_rng(count + hi + nrhs)
    ns = rng.integers(0, hi, count).astype(np.int32)
    ns[[0, count // 2, count - 1]] = [hi, 1, hi - 1]
    cls = nl.CholeskyBatch if kind == "chol" else nl.LUBatch
    bt = cls(ns, nrhs)
    L = rng.uniform(-1, 1, bt.sizeA)
    X, dX = rng.uniform(-1, 1, (2, bt.sizeB))
    P = np.zeros(int(ns.sum()), dtype=np.int32)
    at = 0
    for j, n in enumerate(ns.tolist()):
        L[bt.offA[j] + np.arange(n) * (n + 1)] += 3.0
        P[at: at + n] = [rng.integers(i, n) for i in range(n)]
        at += n
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731

    def adjoint(batch, l, p, x, dx):
        r = batch.backward(d(l), d(x), d(dx)) if kind == "chol" else batch.backward(d(l), d(p), d(x), d(dx))
        return [t.cpu().numpy() for t in r]
    dA, dB = adjoint(bt, L, P, X, dX)
    offP = np.concatenate([[0], np.cumsum(ns)])
    picks = np.unique(np.concatenate([[0, count // 2, count - 1], rng.integers(0, count, 40)]))
    few = cls(ns[picks], nrhs)
    part = lambda a, off, size: np.concatenate([a[off[j]: off[j] + size(int(ns[j]))] for j in picks])  # noqa: E731
    sA, sB = (lambda n: n * n), (lambda n: n * nrhs)
    want = adjoint(few, part(L, bt.offA, sA), part(P, offP, lambda n: n), part(X, bt.offB, sB), part(dX, bt.offB, sB))
    assert np.array_equal(part(dA, bt.offA, sA).view(np.uint64), want[0].view(np.uint64))
    assert np.array_equal(part(dB, bt.offB, sB).view(np.uint64), want[1].view(np.uint64))
    assert np.isfinite(want[0]).all()
