"""Performance cases: what a user of mustard_amd runs, over the sizes and options it is used with.

A case is a dict of plain values with one of these paths:

  tile         one eager tile operation (dgemm, dsyrk, dtrsm) on its own matrices
  factor       a recorded tiled factorization (LU or Cholesky), lowered once and replayed on a
               restored matrix, as the command lines and bench.py do: one hipGraph ("tiled") or one
               persistent scheduler launch ("subgraph")
  solve        recorded forward and back substitution with finished factors, replayed on new
               right-hand sides
  ir           solve_ir: factorization with reduced-precision updates and FP64 refinement, whole call
  grad         autograd.cholesky and its backward, whole calls
  batch        one launch of a batch of uneven factorizations on restored matrices
  batch_solve  BatchSolve.solve: batched factorization, solves and refinement

Matrices are column-major as mustard_amd.to_device makes them: tensor T holds A with T[j, i] = A(i, j).
"""
from __future__ import annotations

import numpy as np
import torch

import mustard_amd as mu
from mustard_amd import autograd, autotune
from mustard_amd.batch import Batch, BatchSolve

DEV = "cuda"
F64 = torch.float64


def listed():
    return [
        # the smallest call: one eager tile product, where launch latency and host work are all
        dict(name="gemm_tile_250", path="tile", op="gemm", m=250, n=250, k=250, ta="N", tb="N"),
        # an eager panel solve of the tile size the benchmark uses (1000), L from a Cholesky tile
        dict(name="trsm_tile_1000", path="tile", op="trsm", m=1000, n=1000, k=0, ta="T", tb="N"),
        # the smallest factorization in use: the verification configuration, 600 in 2 x 2 tiles
        dict(name="lu_600", path="factor", kind="lu", n=600, t=2, mode="tiled"),
        # an ordinary Cholesky with an odd tile size and leading dimension: nothing is aligned
        dict(name="chol_7007", path="factor", kind="chol", n=7007, t=7, mode="tiled"),
        # the headline configuration, N = 24000 in 24 x 24 tiles: LU (the largest case) and Cholesky
        dict(name="lu_24000", path="factor", kind="lu", n=24000, t=24, mode="tiled"),
        dict(name="chol_24000", path="factor", kind="chol", n=24000, t=24, mode="tiled"),
        # the persistent device scheduler (the reference's --subgraph mode) on an ordinary LU
        dict(name="lu_sched_6000", path="factor", kind="lu", n=6000, t=6, mode="subgraph"),
        # substitution with finished LU factors, 16 right-hand sides: a solve server's repeated call
        dict(name="solve_lu_12000", path="solve", kind="lu", n=12000, t=12, nrhs=16),
        # a whole mixed-precision solve, BF16 updates and FP64 refinement
        dict(name="ir_chol_bf16_12000", path="ir", kind="chol", n=12000, t=12, nrhs=16, prec="bf16"),
        # Cholesky inside a differentiated loss: forward and backward (the gradient test's largest size)
        dict(name="grad_4096", path="grad", n=4096, t=16, prec="fp64"),
        # the benchmark's batch: 4096 SPD problems of 32..512 and 512 LU problems of 64..1024
        dict(name="batch_4608", path="batch", nchol=4096, nlu=512, orders=420, prec="fp64"),
        # batched solves with FP32 updates and refinement of all problems together
        dict(name="batch_solve_fp32_288", path="batch_solve", nchol=256, nlu=32, orders=420, prec="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _tiled_order(rng, lo, hi):
    """(n, t): n about log-uniform in [lo, hi] and cut in tiles of about 100 to 1100, odd ones too."""
    n = _log_int(rng, lo, hi)
    b = min(n, _log_int(rng, 100, 1100))
    t = max(1, min(24, n // b))
    return n // t * t, t


def draw(rng):
    path = rng.choice(["tile", "factor", "factor", "factor", "solve", "ir", "grad", "batch", "batch_solve"])
    if path == "tile":
        op = rng.choice(["gemm", "syrk", "trsm"])
        c = dict(path=path, op=op, m=_log_int(rng, 32, 3000), n=_log_int(rng, 17, 3000),
                 k=_log_int(rng, 16, 3000), ta=rng.choice("NT"), tb=rng.choice("NT"))
        if op != "gemm":  # one transposition only: SYRK has none, a solve the triangle's
            c.update(k=c["k"] if op == "syrk" else 0, ta="N" if op == "syrk" else c["ta"], tb="N")
        return c
    kind = rng.choice(["lu", "chol"])
    if path == "factor":
        mode = rng.choice(["tiled", "tiled", "subgraph"])
        n, t = _tiled_order(rng, 200, 20000 if mode == "tiled" else 9000)
        return dict(path=path, kind=kind, n=n, t=t, mode=mode)
    if path == "solve":
        n, t = _tiled_order(rng, 500, 14000)
        return dict(path=path, kind=kind, n=n, t=t, nrhs=rng.randint(1, 16))
    if path == "ir":
        n, t = _tiled_order(rng, 1000, 12000)
        return dict(path=path, kind=kind, n=n, t=t, nrhs=rng.randint(1, 20), prec=rng.choice(["fp32", "bf16"]))
    if path == "grad":
        n, t = _tiled_order(rng, 256, 5000)
        return dict(path=path, n=n, t=t, prec="fp64")
    count = _log_int(rng, 36, 4000 if path == "batch" else 500)
    nlu = rng.randint(count // 16, count // 4)
    return dict(path=path, nchol=count - nlu, nlu=nlu, orders=rng.randrange(1 << 30),
                prec="fp64" if path == "batch" else rng.choice(["fp64", "fp32", "bf16"]))


# ------------------------------------------------------------------------------------------------------
# inputs, from the seed alone
# ------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, *shape):
    return torch.rand(shape, dtype=F64, device=DEV, generator=g)


def _dominant(g, n):
    """Symmetric, uniform [0, 1) off the diagonal, n added to it (the reference generator's matrix)."""
    A = _rand(g, n, n).tril_()
    A += A.tril(-1).t()
    A.diagonal().add_(float(n))
    return A


def _conditioned(g, n, kappa=1e3):
    """Q diag(kappa^(-i/(n-1))) Q^T with Q four Householder reflectors: symmetric, cond_2 = kappa."""
    A = torch.diag(kappa ** (-torch.arange(n, dtype=F64, device=DEV) / max(1, n - 1)))
    for _ in range(4):
        v = 2.0 * _rand(g, n) - 1.0
        v /= v.norm()
        w = A @ v
        S = torch.outer(v, w)
        A -= 2.0 * (S + S.t())
        A += (4.0 * torch.dot(v, w)) * torch.outer(v, v)
    return A


def _batch_orders(case):
    """Kinds and orders of a batch; they belong to the case, the matrices to the seed."""
    r = np.random.default_rng(case["orders"])
    kinds = ["chol"] * case["nchol"] + ["lu"] * case["nlu"]
    ns = [int(x) for x in r.integers(32, 513, case["nchol"])] + [int(x) for x in r.integers(64, 1025, case["nlu"])]
    return kinds, ns


def _batch_inputs(case, seed):
    """Packed matrices (uniform [0, 1), n added to the diagonal; a Cholesky problem is its lower triangle)
    and packed right-hand sides."""
    kinds, ns = _batch_orders(case)
    g = _gen(seed)
    off = np.concatenate([[0], np.cumsum([n * n for n in ns])]).astype(np.int64)
    A = _rand(g, int(off[-1]))
    diag = np.concatenate([o + np.arange(n, dtype=np.int64) * (n + 1) for o, n in zip(off, ns)])
    A[torch.from_numpy(diag).to(DEV)] += torch.from_numpy(np.repeat(np.asarray(ns, dtype=np.float64), ns)).to(DEV)
    b = 2.0 * _rand(g, int(sum(ns))) - 1.0
    if case["path"] == "batch_solve":  # a residual reads whole matrices: make the Cholesky ones symmetric
        for p, n in enumerate(ns[:case["nchol"]]):
            T = A[int(off[p]):int(off[p + 1])].view(n, n)
            T.copy_(T.triu() + T.triu(1).t())
    return kinds, ns, off, A, b


def _tile_inputs(case, seed):
    g = _gen(seed)
    m, n, k = case["m"], case["n"], case["k"]
    if case["op"] == "gemm":
        A = _rand(g, *((k, m) if case["ta"] == "N" else (m, k)))
        B = _rand(g, *((n, k) if case["tb"] == "N" else (k, n)))
        return A, B, _rand(g, n, m)
    if case["op"] == "syrk":
        return _rand(g, k, n), None, _rand(g, n, n)
    # right, lower: B (m x n) <- B op(L)^-1, L a Cholesky factor's tile
    L = _rand(g, n, n).triu_()
    L.diagonal().add_(float(n))
    return L, None, _rand(g, n, m)


def prepare(case, seed):
    p = case["path"]
    if p == "tile":
        A, B, C = _tile_inputs(case, seed)
        return dict(case=case, A=A, B=B, C0=C, C=C.clone())
    if p == "factor":
        n, t = case["n"], case["t"]
        A0 = _dominant(_gen(seed), n)
        F, info = torch.empty_like(A0), mu.info_cell()
        dag = mu.Dag()
        (dag.record_lu if case["kind"] == "lu" else dag.record_cholesky)(mu.ptr(F), n, t, None, mu.ptr(info))
        return dict(case=case, A0=A0, F=F, info=info, ex=mu.Exec(dag, case["mode"]))
    if p == "solve":
        n, t, g = case["n"], case["t"], _gen(seed)
        F = _dominant(g, n)
        B = 2.0 * _rand(g, case["nrhs"], n) - 1.0
        mu.factorize(case["kind"], F, n, t)
        X = torch.empty_like(B)
        dag = mu.Dag().record_solve(mu.ptr(F), n, t, case["kind"], mu.ptr(X), case["nrhs"])
        return dict(case=case, F=F, B=B, X=X, ex=mu.Exec(dag, "tiled"))
    if p == "ir":
        g = _gen(seed)
        A = _conditioned(g, case["n"])
        return dict(case=case, A=A, B=2.0 * _rand(g, case["nrhs"], case["n"]) - 1.0)
    if p == "grad":
        g = _gen(seed)
        A = _dominant(g, case["n"])
        return dict(case=case, A=A, gL=(2.0 * _rand(g, case["n"], case["n"]) - 1.0).tril_())
    kinds, ns, _, A, b = _batch_inputs(case, seed)
    table = autotune.load()
    tiles = [autotune.choose(k, n, table) for k, n in zip(kinds, ns)]
    if p == "batch":
        return dict(case=case, A0=A, bt=Batch(kinds, ns, tiles, prec=case["prec"]))
    bs = BatchSolve(kinds, ns, tiles, prec=case["prec"])
    bs.A0.copy_(A)
    bs.Bv.copy_(b)
    return dict(case=case, bs=bs)


def run(s):
    case = s["case"]
    p = case["path"]
    if p == "tile":
        m, n, k, C = case["m"], case["n"], case["k"], s["C"]
        C.copy_(s["C0"])
        if case["op"] == "gemm":
            mu.dgemm(case["ta"], case["tb"], m, n, k, -1.0, mu.ptr(s["A"]), s["A"].shape[1], mu.ptr(s["B"]),
                     s["B"].shape[1], 1.0, mu.ptr(C), m)
        elif case["op"] == "syrk":
            mu.dsyrk("L", "N", n, k, -1.0, mu.ptr(s["A"]), n, 1.0, mu.ptr(C), n)
        else:
            mu.dtrsm("R", "L", case["ta"], "N", m, n, 1.0, mu.ptr(s["A"]), n, mu.ptr(C), m)
        return C
    if p == "factor":
        s["F"].copy_(s["A0"])
        s["ex"].launch()
        return [s["F"], s["info"]]
    if p == "solve":
        s["X"].copy_(s["B"])
        s["ex"].launch()
        return s["X"]
    if p == "ir":
        X, _ = mu.solve_ir(case["kind"], s["A"], s["B"], case["n"], case["nrhs"], case["t"], prec=case["prec"])
        return X
    if p == "grad":
        A = s["A"].detach().requires_grad_(True)
        L = autograd.cholesky(A, case["t"], case["prec"])
        (G,) = torch.autograd.grad(L, A, s["gL"])
        return [L, G]
    if p == "batch":
        s["bt"].buf.copy_(s["A0"])
        s["bt"].launch()
        return [s["bt"].buf, s["bt"].info]
    s["bs"].solve()
    return s["bs"].X


def _factor_cost(kind, n):
    """(bytes, flops): a Cholesky reads and writes the lower triangle."""
    if kind == "lu":
        return 16.0 * n * n, 2.0 * n ** 3 / 3.0
    return 8.0 * n * (n + 1), n ** 3 / 3.0


def work(case):
    p = case["path"]
    if p == "tile":
        m, n, k = case["m"], case["n"], case["k"]
        if case["op"] == "gemm":
            return dict(bytes=8.0 * (m * k + k * n + 2 * m * n), flops=2.0 * m * n * k)
        if case["op"] == "syrk":
            return dict(bytes=8.0 * (n * k + n * (n + 1)), flops=1.0 * n * (n + 1) * k)
        return dict(bytes=8.0 * (n * (n + 1) / 2 + 2 * m * n), flops=1.0 * m * n * n)
    if p in ("batch", "batch_solve"):
        kinds, ns = _batch_orders(case)
        by = sum(_factor_cost(k, n)[0] for k, n in zip(kinds, ns))
        fl = sum(_factor_cost(k, n)[1] for k, n in zip(kinds, ns))
        if p == "batch_solve":  # the matrices in, the solutions out
            by = sum(8.0 * n * n if k == "lu" else 4.0 * n * (n + 1) for k, n in zip(kinds, ns)) + 16.0 * sum(ns)
            fl += sum(2.0 * n * n for n in ns)
        return dict(bytes=by, flops=fl)
    n = case["n"]
    if p == "factor":
        by, fl = _factor_cost(case["kind"], n)
    elif p == "solve":
        by = (8.0 * n * n if case["kind"] == "lu" else 4.0 * n * (n + 1)) + 16.0 * n * case["nrhs"]
        fl = 2.0 * n * n * case["nrhs"]
    elif p == "ir":
        by = (8.0 * n * n if case["kind"] == "lu" else 4.0 * n * (n + 1)) + 16.0 * n * case["nrhs"]
        fl = _factor_cost(case["kind"], n)[1] + 2.0 * n * n * case["nrhs"]
    else:  # grad: A and Lbar in, L and the gradient out; n^3/3 forward, two n^3/3 products and solves back
        by, fl = 8.0 * n * (n + 1) + 4.0 * n * (n + 1) + 8.0 * n * n, n ** 3 / 3.0 + 2.0 * n ** 3 / 3.0
    return dict(bytes=by, flops=fl)


# ------------------------------------------------------------------------------------------------------
# the same results by torch in 64 bits
# ------------------------------------------------------------------------------------------------------
def _chol_out(T):
    """Lower factor over the untouched strict upper triangle, of the column-major T (its triu is A's lower)."""
    S = T.triu() + T.triu(1).t()
    return torch.linalg.cholesky(S).t() + T.tril(-1)


def _lu_out(T):
    """L and U packed; column-wise diagonally dominant, so partial pivoting keeps the rows in order."""
    return torch.linalg.lu_factor(T.t())[0].t().contiguous()


def exact(case, seed):
    p = case["path"]
    if p == "tile":
        A, B, C = _tile_inputs(case, seed)
        if case["op"] == "gemm":  # C - op(A) op(B), transposed: T(C) - T(op B) T(op A)
            a = A if case["ta"] == "N" else A.t()
            b = B if case["tb"] == "N" else B.t()
            return C - b @ a
        if case["op"] == "syrk":
            return C.tril(-1) + (C - A.t() @ A).triu()
        # column-major X op(L) = C; with T(X) = X^T: op(L)^T X^T = C^T, and the tensor A is L^T
        if case["ta"] == "N":
            return torch.linalg.solve_triangular(A, C, upper=True)
        return torch.linalg.solve_triangular(A.t(), C, upper=False)
    if p == "factor":
        T = _dominant(_gen(seed), case["n"])
        return [_lu_out(T) if case["kind"] == "lu" else _chol_out(T), None]
    if p == "solve":
        g = _gen(seed)
        A = _dominant(g, case["n"])
        B = 2.0 * _rand(g, case["nrhs"], case["n"]) - 1.0
        return torch.linalg.solve(A, B.t()).t()
    if p == "ir":
        g = _gen(seed)
        A = _conditioned(g, case["n"])
        B = 2.0 * _rand(g, case["nrhs"], case["n"]) - 1.0
        return torch.linalg.solve(A, B.t()).t()
    if p == "grad":
        g = _gen(seed)
        A = _dominant(g, case["n"]).requires_grad_(True)
        gL = (2.0 * _rand(g, case["n"], case["n"]) - 1.0).tril_()
        L = torch.linalg.cholesky(A)
        (G,) = torch.autograd.grad(L, A, gL)
        return [L.detach(), G]
    kinds, ns, off, A, b = _batch_inputs(case, seed)
    if p == "batch":
        if len(ns) > 1500:  # a loop over every problem takes too long
            return None
        out = A.cpu()
        for i, (k, n) in enumerate(zip(kinds, ns)):
            T = out[int(off[i]):int(off[i + 1])].view(n, n)
            T.copy_(_lu_out(T) if k == "lu" else _chol_out(T))
        return [out, None]
    A, b, v = A.cpu(), b.cpu(), 0
    for i, n in enumerate(ns):
        T = A[int(off[i]):int(off[i + 1])].view(n, n)
        b[v:v + n] = torch.linalg.solve(T.t(), b[v:v + n])
        v += n
    return b
