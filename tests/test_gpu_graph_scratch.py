"""Captured calls own their scratch: graphs replayed on several streams beside
each other and beside eager calls of the same handle give what each call gives
alone."""
import ctypes as C
import gc

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _problem(kind, n, seed):
    """(inputs, run): run(out) queues one call on torch's current stream."""
    from nalgebra_amd._lib import lib
    from nalgebra_amd.linalg import handle
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1, 1, (n, n))
    if kind == "chol":
        a = a @ a.T / n + np.eye(n)
    elif kind == "solve":
        a = a / n + np.eye(n)
    a = torch.from_numpy(np.asfortranarray(a).ravel(order="F").copy()).cuda()
    b = torch.from_numpy(rng.uniform(-1, 1, n)).cuda()
    piv = torch.arange(n, dtype=torch.int32, device="cuda").flip(0).contiguous()

    def run(out):
        x, ints = out
        h = handle()
        if kind == "solve":
            x.copy_(b)
            st = lib().nrocm_dgetrs(h, n, 1, _ptr(a), n, _ptr(piv), _ptr(x), n, _ptr(ints), 0)
        else:
            x.copy_(a)
            if kind == "lu":
                st = lib().nrocm_dgetrf(h, n, n, _ptr(x), n, _ptr(ints), C.c_void_p(ints.data_ptr() + 4 * n), 0)
            else:
                st = lib().nrocm_dpotrf(h, n, _ptr(x), n, _ptr(ints), 0)
        assert st == 0
    size = n if kind == "solve" else n * n
    return run, (torch.empty(size, dtype=torch.float64, device="cuda"), torch.zeros(n + 1, dtype=torch.int32, device="cuda"))


@pytest.mark.parametrize("kind,n", [("lu", 60), ("lu", 300), ("chol", 400), ("solve", 1100)])
def test_replays_beside_each_other_and_eager_calls(nl, kind, n):
    jobs = [_problem(kind, n, s) for s in range(3)]
    want = []
    for run, out in jobs:
        run(out)
        torch.cuda.synchronize()
        want.append([t.clone() for t in out])
    torch.cuda.synchronize()
    graphs = []
    for run, out in jobs[:2]:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            run(out)
        graphs.append(g)
    streams = [torch.cuda.Stream() for _ in range(3)]
    for round_ in range(6):
        for _, out in jobs:
            for t in out:
                t.zero_()
        torch.cuda.synchronize()
        for _ in range(4):
            for k in range(2):
                with torch.cuda.stream(streams[k]):
                    graphs[k].replay()
            with torch.cuda.stream(streams[2]):
                jobs[2][0](jobs[2][1])
        torch.cuda.synchronize()
        for k in range(3):
            for got, ref in zip(jobs[k][1], want[k]):
                assert torch.equal(got, ref), (kind, round_, k)


def test_graph_scratch_is_given_back(nl):
    """What captured calls took is free again after nrocm_free_graph_scratch."""
    from nalgebra_amd._lib import lib
    L = lib()
    h = C.c_void_p()
    assert L.nrocm_create(C.byref(h)) == 0
    n, calls = 1000, 40
    s = torch.cuda.Stream()
    assert L.nrocm_set_stream(h, s.cuda_stream) == 0
    a = torch.rand(n * n, dtype=torch.float64, device="cuda")
    ints = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    free0 = torch.cuda.mem_get_info()[0]
    for _ in range(calls):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            assert L.nrocm_dgetrf(h, n, n, _ptr(a), n, _ptr(ints), C.c_void_p(ints.data_ptr() + 4 * n), 0) == 0
        del g
    torch.cuda.synchronize()
    assert free0 - torch.cuda.mem_get_info()[0] >= calls * n * n * 8
    assert L.nrocm_free_graph_scratch(h) == 0
    assert free0 - torch.cuda.mem_get_info()[0] < calls * n * n * 4
    assert L.nrocm_free_graph_scratch(None) == -1
    assert L.nrocm_destroy(h) == 0


@pytest.mark.parametrize("n,mode", [(1100, 0), (2300, 1)])
def test_captured_lu_of_panels(nl, n, mode):
    """Above 1024 rows the factorisation is many launches on two streams."""
    a = nl.DMatrix(torch.rand(n * n, dtype=torch.float64, device="cuda").sub_(0.5), n, n)
    ref = a.lu(mode)
    buf = nl.DMatrix(torch.empty_like(a.data), n, n)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        buf.data.copy_(a.data)
        lu = nl.LU(buf, mode)
    for _ in range(3):
        buf.data.zero_()
        lu.ipiv.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(lu.lu.data, ref.lu.data) and torch.equal(lu.ipiv, ref.ipiv) and lu.info == 0
        other = a.lu(mode)  # eager, between the replays
        torch.cuda.synchronize()
        assert torch.equal(other.lu.data, ref.lu.data)


def test_captured_batches(nl):
    """The batched Cholesky replays a graph of its own when it is not captured."""
    import gen
    ns = [4, 17, 33, 64, 9, 30, 50] * 20
    A, _, B, _ = gen.spd_batch(5, ns, 2)
    bt = nl.CholeskyBatch(ns, 2)
    A0, B0 = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    a, b = A0.clone(), B0.clone()
    ptrs = bt.pointers(a, b)
    info = torch.ones(len(ns), dtype=torch.int32, device="cuda")
    bt.solve_ptrs(*ptrs, info)  # eager
    torch.cuda.synchronize()
    want = [a.clone(), b.clone()]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.copy_(A0)
        b.copy_(B0)
        bt.solve_ptrs(*ptrs, info)
    for _ in range(3):
        a.zero_(), b.zero_(), info.fill_(1)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(a, want[0]) and torch.equal(b, want[1]) and not info.any()
        a.copy_(A0), b.copy_(B0)
        bt.solve_ptrs(*ptrs, info)
        torch.cuda.synchronize()
        assert torch.equal(b, want[1])
