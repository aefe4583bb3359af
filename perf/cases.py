"""Performance cases of the dense hot path, through its public entry points.

Every case is a dict of plain values whose "kind" names a use:

  gemm        C = alpha A B + beta C (Matrix::gemm) or A * B
  lu          a.lu(mode), then solve
  inverse     a.lu(mode).try_inverse()
  cholesky    a.cholesky(mode), then solve
  qr          a.qr(), then solve_least_squares
  chol_batch  uneven batch, Cholesky + solve, buffers and pointers kept
  chol_train  uneven batch, forward solve and its adjoint, loss = sum |x|^2
  lu_train    uneven batch, LU + solve and its adjoint, loss = sum |x|^2
  lsq_batch   tall f32 least-squares systems, solved in a batch
  mixed       one large system, low-precision factors + FP64 refinement

prepare() makes the inputs on the GPU and the plan a program keeps; run() is
one pass; exact() gives the same results with plain torch in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import nalgebra_amd as na

DEV = "cuda"
MODES = {"exact": na.EXACT, "fast": na.FAST}
PRECISIONS = {"fp64": na.PREC_FP64, "fp32": na.PREC_FP32, "bf16x3": na.PREC_BF16X3}
DTYPES = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # the smallest product a filter or a graph step makes: call latency
        {"name": "gemm_f64_100", "kind": "gemm", "dtype": "f64", "m": 100, "k": 100, "n": 100, "form": "update"},
        # a large product of matrices of no special size (odd leading dimensions)
        {"name": "gemm_f32_large", "kind": "gemm", "dtype": "f32", "m": 4095, "k": 3001, "n": 2047, "form": "mul"},
        # one dense system of ordinary size, the reference's own arithmetic
        {"name": "lu_exact_500", "kind": "lu", "mode": "exact", "n": 500, "nrhs": 1},
        # LU::try_inverse: as many right-hand sides as rows
        {"name": "inverse_exact_300", "kind": "inverse", "mode": "exact", "n": 300},
        # a large dense system with partial pivoting, several loads
        {"name": "lu_fast_4096", "kind": "lu", "mode": "fast", "n": 4096, "nrhs": 8},
        # a covariance matrix: factor and solve in the reference's arithmetic
        {"name": "cholesky_exact_1500", "kind": "cholesky", "mode": "exact", "n": 1500, "nrhs": 2},
        # a regression: tall QR and least squares
        {"name": "qr_1500x200", "kind": "qr", "m": 1500, "n": 200, "nrhs": 1},
        # the benchmark batch: 65,536 uneven SPD systems
        {"name": "chol_batch_65536", "kind": "chol_batch", "mode": "exact", "count": 65536, "lo": 4, "hi": 64, "nrhs": 4},
        # the differentiated solve: forward and backward
        {"name": "chol_train_4096", "kind": "chol_train", "mode": "exact", "count": 4096, "lo": 32, "hi": 32, "nrhs": 1},
        # the same for general systems of uneven sizes
        {"name": "lu_train_16384", "kind": "lu_train", "mode": "exact", "count": 16384, "lo": 4, "hi": 64, "nrhs": 2},
        # the benchmark's tall least-squares batch
        {"name": "lsq_batch_2048", "kind": "lsq_batch", "count": 2048, "lo": 256, "hi": 2048, "n": 64, "refine": 1},
        # the benchmark's large system, kappa = 1e4, mixed precision
        {"name": "mixed_fp32_8192", "kind": "mixed", "precision": "fp32", "n": 8192},
    ]


def draw(rng):
    def size(lo, hi):  # log-uniform; half of them odd or otherwise unaligned by themselves
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["gemm", "gemm", "lu", "lu", "inverse", "cholesky", "qr", "chol_batch", "chol_train", "lu_train",
                       "lsq_batch", "mixed"])
    if kind == "gemm":
        return {"kind": kind, "dtype": rng.choice(["f64", "f32"]), "m": size(24, 4095), "k": size(24, 3001),
                "n": size(24, 2047), "form": rng.choice(["update", "mul"])}
    if kind == "lu":
        mode = rng.choice(["exact", "fast"])
        return {"kind": kind, "mode": mode, "n": size(16, 1024 if mode == "exact" else 4096), "nrhs": rng.randint(1, 8)}
    if kind == "inverse":
        return {"kind": kind, "mode": rng.choice(["exact", "fast"]), "n": size(8, 300)}
    if kind == "cholesky":
        return {"kind": kind, "mode": rng.choice(["exact", "fast"]), "n": size(16, 1500), "nrhs": rng.randint(1, 4)}
    if kind == "qr":
        n = size(6, 200)
        return {"kind": kind, "m": size(max(n, 16), 1500), "n": n, "nrhs": rng.randint(1, 3)}
    if kind == "lsq_batch":
        n = rng.randint(8, 64)
        lo = size(2 * n, 512)
        return {"kind": kind, "count": size(16, 2048), "lo": lo, "hi": size(lo, 2048), "n": n,
                "refine": rng.randint(1, 2)}
    if kind == "mixed":
        return {"kind": kind, "precision": rng.choice(["fp32", "fp32", "fp64", "bf16x3"]), "n": size(700, 8000)}
    lo = size(2, 32)
    most = {"chol_batch": 65536, "chol_train": 16384, "lu_train": 16384}[kind]
    return {"kind": kind, "mode": rng.choice(["exact", "exact", "fast"]), "count": size(32, most), "lo": lo,
            "hi": size(lo, 64), "nrhs": rng.randint(1, 4 if kind == "chol_batch" else 2)}


# ---------------------------------------------------------------- inputs


def _rng(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, count, dtype=torch.float64):
    return torch.rand(count, generator=g, device=DEV, dtype=dtype).mul_(2).sub_(1)


def _sizes(case):
    """The batch's member sizes: part of the plan, the same for every seed."""
    return np.random.RandomState(case["count"]).randint(case["lo"], case["hi"] + 1, case["count"]).astype(np.int32)


def _groups(ns, per_member):
    """(n, first elements of the members of size n) of packed members of per_member(n) elements each."""
    lengths = per_member(ns.astype(np.int64))
    off = np.concatenate([[0], np.cumsum(lengths)[:-1]])
    return [(int(n), torch.from_numpy(off[ns == n]).to(DEV)) for n in np.unique(ns)], int(lengths.sum())


def _at(off, length):
    return off[:, None] + torch.arange(length, device=DEV)


def _batch_inputs(case, seed, spd):
    """Packed A (column-major members) and B of an uneven batch."""
    g, ns, nrhs = _rng(seed), _sizes(case), case["nrhs"]
    groups, total = _groups(ns, lambda n: n * n)
    A = torch.empty(total, dtype=torch.float64, device=DEV)
    for n, off in groups:
        if spd:
            G = torch.randn(len(off), n, n, generator=g, device=DEV, dtype=torch.float64)
            M = torch.bmm(G, G.transpose(1, 2).contiguous())
            M.diagonal(dim1=1, dim2=2).add_(n)
        else:
            M = _uniform(g, len(off) * n * n)
        A[_at(off, n * n)] = M.view(len(off), n * n)
    B = torch.randn(int(ns.sum()) * nrhs, generator=g, device=DEV, dtype=torch.float64)
    return ns, A, B


def _lsq_inputs(case, seed):
    """b = A x + 1e-3 N(0, 1), the entries of A and x N(0, 1)."""
    g, ms, n = _rng(seed), _sizes(case), case["n"]
    A = torch.randn(int(ms.sum()) * n, generator=g, device=DEV, dtype=torch.float32)
    b = torch.randn(int(ms.sum()), generator=g, device=DEV, dtype=torch.float32).mul_(1e-3)
    x = torch.randn(len(ms), n, generator=g, device=DEV, dtype=torch.float32)
    r0 = 0
    for j, m in enumerate(ms.tolist()):
        b[r0:r0 + m] += x[j] @ A[r0 * n:(r0 + m) * n].view(n, m)
        r0 += m
    return ms, A, b


def _gemm_inputs(case, seed):
    g, dt = _rng(seed), DTYPES[case["dtype"]]
    m, k, n = case["m"], case["k"], case["n"]
    return _uniform(g, m * k, dt), _uniform(g, k * n, dt), _uniform(g, m * n, dt)


def _dense_inputs(case, seed):
    """A general matrix and its right-hand sides, entries uniform in [-1, 1]."""
    g, n = _rng(seed), case["n"]
    return _uniform(g, case.get("m", n) * n), _uniform(g, case.get("m", n) * case.get("nrhs", 1))


def _spd_inputs(case, seed):
    g, n = _rng(seed), case["n"]
    G = torch.randn(n, n, generator=g, device=DEV, dtype=torch.float64)
    A = G @ G.T.contiguous()
    A.diagonal().add_(n)
    return A.view(-1), torch.randn(n * case["nrhs"], generator=g, device=DEV, dtype=torch.float64)


def _mix(X, g):
    """A random dense orthogonal matrix times X: random signs and Hartley transforms."""
    n = X.shape[0]
    for _ in range(2):
        s = torch.randint(0, 2, (n, 1), generator=g, device=DEV).to(torch.float64).mul_(2).sub_(1)
        F = torch.fft.fft(X * s, dim=0)
        X = (F.real - F.imag) / math.sqrt(n)
    return X


def _mixed_inputs(case, seed):
    """A = U diag(sigma) V^T with sigma log-spaced from 1 to 1e-4, and b ~ N(0, 1)."""
    g, n = _rng(seed), case["n"]
    sigma = torch.logspace(0, -4, n, dtype=torch.float64, device=DEV)
    A = _mix(_mix(torch.diag(sigma), g).T.contiguous(), g)
    return A.contiguous().view(-1), torch.randn(n, generator=g, device=DEV, dtype=torch.float64)


# ---------------------------------------------------------------- the passes


def prepare(case, seed):
    s, kind = {"case": case}, case["kind"]
    if kind == "gemm":
        a, b, c = _gemm_inputs(case, seed)
        s["a"], s["b"] = na.DMatrix(a, case["m"], case["k"]), na.DMatrix(b, case["k"], case["n"])
        s["c"] = na.DMatrix(c, case["m"], case["n"])
    elif kind in ("lu", "inverse", "qr", "cholesky", "mixed"):
        make = {"cholesky": _spd_inputs, "mixed": _mixed_inputs}.get(kind, _dense_inputs)
        a, b = make(case, seed)
        m = case.get("m", case["n"])
        s["a"], s["b"] = na.DMatrix(a, m, case["n"]), na.DMatrix(b, m, case.get("nrhs", 1))
    elif kind == "lsq_batch":
        ms, s["A"], s["b"] = _lsq_inputs(case, seed)
        s["batch"] = na.LeastSquaresBatch(ms, case["n"])
    else:
        ns, s["A0"], s["B0"] = _batch_inputs(case, seed, kind != "lu_train")
        s["A"], s["B"] = torch.empty_like(s["A0"]), torch.empty_like(s["B0"])
        if kind == "lu_train":
            s["batch"] = na.LUBatch(ns, case["nrhs"])
        else:
            bt = s["batch"] = na.CholeskyBatch(ns, case["nrhs"])
            bt.autotune(MODES[case["mode"]])
            s["ptrs"] = bt.pointers(s["A"], s["B"])
            if kind == "chol_train":
                s["dX"], s["dA"], s["dB"] = (torch.empty_like(s[k]) for k in ("B", "A", "B"))
                s["grad_ptrs"] = (*bt.pointers(s["dA"], s["dX"]), bt.pointers(s["A"], s["dB"])[1])
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "gemm":
        if case["form"] == "mul":
            return (s["a"] @ s["b"]).data
        c = s["c"].clone()
        c.gemm(0.5, s["a"], s["b"], 1.0)
        return c.data
    if kind == "lu":
        lu = s["a"].lu(MODES[case["mode"]])
        x = lu.solve(s["b"])
        return [lu.lu.data, lu.ipiv, x.data]
    if kind == "inverse":
        return s["a"].lu(MODES[case["mode"]]).try_inverse().data
    if kind == "cholesky":
        ch = s["a"].cholesky(MODES[case["mode"]])
        return [ch.l_dirty().data, ch.solve(s["b"]).data]
    if kind == "qr":
        qr = s["a"].qr()
        x = qr.solve_least_squares(s["b"])
        return [qr.qr.data, qr.diag, x.data]
    if kind == "mixed":
        # the number of refinement steps and the reached error are not results
        x, _, _, ok = na.solve_mixed_ir(s["a"], s["b"], PRECISIONS[case["precision"]] | na.PREC_WINDOW)
        return [x.data, ok]
    bt = s["batch"]
    if kind == "lsq_batch":
        x, info = bt.solve(s["A"], s["b"], case["refine"])
        return [x, info]
    A, B, mode = s["A"].copy_(s["A0"]), s["B"].copy_(s["B0"]), MODES[case["mode"]]
    if kind == "lu_train":
        P, info = bt.solve(A, B, mode)
        dA, dB = bt.backward(A, P, B, 2.0 * B)
        return [A, B, P, info, dA, dB]
    info = bt.solve(A, B, mode, ptrs=s["ptrs"])
    if kind == "chol_train":
        torch.mul(B, 2.0, out=s["dX"])
        pdA, pdX, pdB = s["grad_ptrs"]
        bt.backward_raw(s["ptrs"][0], s["ptrs"][1], pdX, pdA, pdB)
        return [A, B, info, s["dA"], s["dB"]]
    return [A, B, info]


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        c = 2 if case["form"] == "update" else 1
        return {"bytes": (8 if case["dtype"] == "f64" else 4) * (m * k + k * n + c * m * n), "flops": 2.0 * m * n * k}
    if kind in ("lu", "inverse", "cholesky", "mixed"):
        n = float(case["n"])
        r = n if kind == "inverse" else float(case.get("nrhs", 1))
        factor = n ** 3 / 3 if kind == "cholesky" else 2 * n ** 3 / 3
        read = n * n + (0 if kind == "inverse" else n * r)
        written = n * r + (0 if kind in ("inverse", "mixed") else n * n)
        return {"bytes": 8 * (read + written), "flops": factor + 2 * n * n * r}
    if kind == "qr":
        m, n, r = float(case["m"]), float(case["n"]), float(case["nrhs"])
        return {"bytes": 8 * (2 * m * n + m * r + n * r + n),
                "flops": 2 * m * n * n - 2 * n ** 3 / 3 + (4 * m * n - n * n) * r}
    ns = _sizes(case).astype(np.float64)
    if kind == "lsq_batch":
        n, ref = float(case["n"]), case["refine"]
        return {"bytes": float((4 * ns * (n + 1) + 8 * n + 4).sum()),
                "flops": float((2 * ns * n * n - 2 * n ** 3 / 3 + (1 + ref) * (4 * ns * n) + ref * 2 * ns * n).sum())}
    r = case["nrhs"]
    if kind == "lu_train":  # A read, L\U and dA written; B read, X and dB written; the pivots
        return {"bytes": float((8 * (3 * ns * ns + 3 * ns * r) + 4 * ns).sum()),
                "flops": float((2 * ns ** 3 / 3 + 6 * ns * ns * r).sum())}
    # Cholesky: the lower triangle read and written, B read, X written
    b, f = 8 * (ns * (ns + 1) + 2 * ns * r), ns ** 3 / 3 + 2 * ns * ns * r
    if kind == "chol_train":  # and dA, dB written
        b, f = b + 8 * (ns * ns + ns * r), f + 4 * ns * ns * r
    return {"bytes": float(b.sum()), "flops": float(f.sum())}


# ---------------------------------------------------------------- the results in 64 bits


def _cols(flat, m, n):
    """The m x n matrix that `flat` holds column by column."""
    return flat.view(n, m).T


def _flat(M):
    return M.T.contiguous().view(-1)


def _householder(A, B):
    """Householder QR of A with unit axes: (axes below and R above the diagonal, signed norms, Q^T B)."""
    A, B = A.contiguous().clone(), B.contiguous().clone()
    diag = torch.zeros(min(A.shape), dtype=A.dtype, device=A.device)
    for i in range(len(diag)):
        x = A[i:, i].clone()
        norm = x.norm()
        sign = torch.where(x[0] >= 0, 1.0, -1.0)
        x[0] += sign * norm
        x /= x.norm()
        for M in (A[i:, i + 1:], B[i:]):
            M.copy_(-sign * (M - 2 * torch.outer(x, x @ M)))
        A[i:, i] = x
        diag[i] = -sign * norm
    return A, diag, B


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        a, b, c = (t.double() for t in _gemm_inputs(case, seed))
        m, k, n = case["m"], case["k"], case["n"]
        ab = _cols(a, m, k) @ _cols(b, k, n)
        return _flat(ab if case["form"] == "mul" else 0.5 * ab + _cols(c, m, n))
    if kind in ("lu", "inverse"):
        a, b = (t.cpu() for t in _dense_inputs(case, seed))
        A = _cols(a, case["n"], case["n"])
        if kind == "inverse":
            return _flat(torch.linalg.inv(A))
        LU, piv = torch.linalg.lu_factor(A)
        x = torch.linalg.lu_solve(LU, piv, _cols(b, case["n"], case["nrhs"]).contiguous())
        return [_flat(LU), None, _flat(x)]
    if kind == "cholesky":
        a, b = (t.cpu() for t in _spd_inputs(case, seed))
        A = _cols(a, case["n"], case["n"])
        L = torch.linalg.cholesky(A)
        x = torch.cholesky_solve(_cols(b, case["n"], case["nrhs"]).contiguous(), L)
        return [_flat(L.tril() + A.triu(1)), _flat(x)]
    if kind == "qr":
        a, b = (t.cpu() for t in _dense_inputs(case, seed))
        m, n, r = case["m"], case["n"], case["nrhs"]
        QR, diag, QtB = _householder(_cols(a, m, n), _cols(b, m, r))
        R = QR[:n].triu(1) + torch.diag(diag.abs())
        x = torch.linalg.solve_triangular(R, QtB[:n], upper=True)
        return [_flat(QR), diag, _flat(x)]
    if kind == "mixed":
        a, b = (t.cpu() for t in _mixed_inputs(case, seed))
        return [torch.linalg.solve(_cols(a, case["n"], case["n"]), b), None]
    if kind == "lsq_batch":  # well conditioned: the normal equations
        ms, A, b = _lsq_inputs(case, seed)
        n, r0, G, y = case["n"], 0, [], []
        for m in ms.tolist():
            M = A[r0 * n:(r0 + m) * n].double().view(n, m)
            G.append(M @ M.T.contiguous())
            y.append(M @ b[r0:r0 + m].double())
            r0 += m
        x = torch.cholesky_solve(torch.stack(y).cpu()[:, :, None], torch.linalg.cholesky(torch.stack(G).cpu()))
        return [x[:, :, 0].contiguous(), None]
    ns, A, B = _batch_inputs(case, seed, kind != "lu_train")
    A, B, r = A.cpu(), B.cpu(), case["nrhs"]
    F, X = torch.empty_like(A), torch.empty_like(B)
    dA, dB = torch.empty_like(A), torch.empty_like(B)
    ga, gb = _groups(ns, lambda n: n * n)[0], _groups(ns, lambda n: n * r)[0]
    for (n, oa), (_, ob) in zip(ga, gb):
        ia, ib = _at(oa, n * n).cpu(), _at(ob, n * r).cpu()
        M = A[ia].view(-1, n, n).transpose(1, 2).contiguous()
        Y = B[ib].view(-1, r, n).transpose(1, 2).contiguous()
        train = kind != "chol_batch"
        lam = grad = None
        if kind == "lu_train":
            factor, piv = torch.linalg.lu_factor(M)
            x = torch.linalg.lu_solve(factor, piv, Y)
            lam = torch.linalg.solve(M.transpose(1, 2).contiguous(), 2.0 * x)
            grad = -torch.bmm(lam, x.transpose(1, 2).contiguous())
        else:
            L = torch.linalg.cholesky(M)
            x = torch.cholesky_solve(Y, L)
            factor = L.tril() + M.triu(1)
            if train:
                lam = torch.cholesky_solve(2.0 * x, L)
                half = -0.5 * torch.bmm(lam, x.transpose(1, 2).contiguous())
                grad = half + half.transpose(1, 2)
        F[ia] = factor.transpose(1, 2).reshape(-1, n * n)
        X[ib] = x.transpose(1, 2).reshape(-1, n * r)
        if train:
            dA[ia] = grad.transpose(1, 2).reshape(-1, n * n)
            dB[ib] = lam.transpose(1, 2).reshape(-1, n * r)
    if kind == "chol_batch":
        return [F, X, None]
    if kind == "chol_train":
        return [F, X, None, dA, dB]
    return [F, X, None, None, dA, dB]
