"""Calls of one handle on two streams run side by side: a call on one stream does
not wait for the other stream's work, and results are those of each call alone."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _long_wait(stream):
    """Keeps `stream` busy for some tenths of a second, with one workgroup."""
    with torch.cuda.stream(stream):
        torch.cuda._sleep(_long_wait.cycles)


def _calibrate():
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1000)
    a.record()
    torch.cuda._sleep(1000000)
    b.record()
    torch.cuda.synchronize()
    _long_wait.cycles = int(1000000 * 400.0 / max(a.elapsed_time(b), 1e-3))


@pytest.fixture(scope="module")
def streams(nl):
    """Two streams that the hardware runs side by side."""
    _calibrate()
    s = [torch.cuda.Stream() for _ in range(6)]
    t = torch.zeros(64, device="cuda")
    torch.cuda.synchronize()
    for other in s[1:]:
        _long_wait(s[0])
        ea, eb = torch.cuda.Event(), torch.cuda.Event()
        ea.record(s[0])
        with torch.cuda.stream(other):
            t.add_(1)
        eb.record(other)
        eb.synchronize()
        apart = not ea.query()
        torch.cuda.synchronize()
        if apart:
            return s[0], other
    pytest.skip("no two streams of this process run side by side")


def _call(kind, n, seed):
    from nalgebra_amd._lib import lib
    from nalgebra_amd.linalg import handle
    rng = np.random.default_rng(seed)
    M = rng.uniform(-1, 1, (n, n))
    if kind == "chol":
        M = M @ M.T + n * np.eye(n)
    elif kind == "solve":
        M = M / n + np.eye(n)
    src = torch.from_numpy(np.asfortranarray(M).ravel(order="F").copy()).cuda()
    a, b = torch.empty_like(src), torch.from_numpy(rng.uniform(-1, 1, n)).cuda()
    x, ints = torch.empty_like(b), torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    piv = torch.arange(n, dtype=torch.int32, device="cuda")
    info = C.c_void_p(ints.data_ptr() + 4 * n)

    def run():
        a.copy_(src)
        x.copy_(b)
        h, L = handle(), lib()
        st = (L.nrocm_dgetrf(h, n, n, _ptr(a), n, _ptr(ints), info, 0) if kind == "lu" else
              L.nrocm_dgeqrf(h, n, n, _ptr(a), n, _ptr(x)) if kind == "qr" else
              L.nrocm_dpotrf(h, n, _ptr(a), n, info, 0) if kind == "chol" else
              L.nrocm_dgetrs(h, n, 1, _ptr(a), n, _ptr(piv), _ptr(x), n, info, 0))
        assert st == 0
    return run, (a, x, ints)


@pytest.mark.parametrize("kind,n", [("lu", 50), ("lu", 300), ("qr", 100), ("chol", 400), ("solve", 1100)])
def test_side_by_side(nl, streams, kind, n):
    jobs = [_call(kind, n, k) for k in range(2)]
    want = []
    for (run, out), s in zip(jobs, streams):  # alone, which also makes the scratch
        with torch.cuda.stream(s):
            run()
        torch.cuda.synchronize()
        want.append([t.clone() for t in out])
    torch.cuda.synchronize()
    _long_wait(streams[0])
    events = []
    for (run, _), s in zip(jobs, streams):
        with torch.cuda.stream(s):
            run()
        events.append(torch.cuda.Event())
        events[-1].record(s)
    events[1].synchronize()
    assert not events[0].query(), "the second stream waited for the first"
    torch.cuda.synchronize()
    for (_, out), ref in zip(jobs, want):
        for got, r in zip(out, ref):
            assert torch.equal(got, r)


def test_more_streams_than_scratch(nl):
    """Nine streams in turn, without a wait: each gets its own result."""
    from collections import deque
    ss = [torch.cuda.Stream() for _ in range(9)]
    jobs = [_call("lu", 120 + 7 * k, k) for k in range(9)]
    want = []
    for run, out in jobs:
        run()
        torch.cuda.synchronize()
        want.append([t.clone() for t in out])
    for _ in range(3):
        order = deque(range(9))
        for turn in range(9):
            order.rotate(4)
            with torch.cuda.stream(ss[order[0]]):
                jobs[order[0]][0]()
        torch.cuda.synchronize()
        for (_, out), ref in zip(jobs, want):
            for got, r in zip(out, ref):
                assert torch.equal(got, r)
