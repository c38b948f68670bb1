"""GPU tests of the one-workgroup factorizations and panel solves on squared-
exponential kernel matrices, whose diagonal blocks are as ill-conditioned as
double precision allows: the backward error has to be that of substitution,
whatever the condition, and a matrix that LAPACK factors has to be factored.

The bounds: an element of L L^T, L U or T X passes at most n + 1 roundings of
its products and sums; a 16 x 16 block solved through its inverse and one
residual correction adds three products of 17 terms and their sums (about 60
roundings) in place of its own 16, and twice that covers the reciprocals of
the pivots."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def kernel_matrix(n, nugget, seed):
    """Covariances of n sorted points in [0, 1], length scale 0.1, plus nugget * I."""
    t = np.sort(np.random.default_rng(seed).random(n))
    return np.exp(-((t[:, None] - t[None]) ** 2) / 0.02) + nugget * np.eye(n)


def bound(n, S):
    return 2 * (n + 64) * U * S


def product(A, B):
    return (A.astype(np.longdouble) @ B.astype(np.longdouble)).astype(np.longdouble)


def factor(kind, A, mode):
    """Factors of one tile: an eager call, a graph node or the persistent scheduler."""
    import mustard_amd as mu
    n, dA, info = len(A), mu.to_device(np.asfortranarray(A)), mu.info_cell()
    if mode == "eager":
        if kind == "lu":
            mu.dgetrf_nopiv(n, mu.ptr(dA), n, mu.ptr(info))
        else:
            mu.dpotrf("L", n, mu.ptr(dA), n, mu.ptr(info))
    else:
        dag = mu.Dag()
        (dag.record_lu if kind == "lu" else dag.record_cholesky)(mu.ptr(dA), n, 1, None, mu.ptr(info))
        ex = mu.Exec(dag, mode)
        ex.launch()
    F = mu.to_host(dA)
    assert mu.info_value(info) == 0
    return F


@pytest.mark.parametrize("mode", ["eager", "tiled", "subgraph"])
@pytest.mark.parametrize("nugget", [1e-6, 1e-8, 1e-10, 1e-12, 1e-13])
@pytest.mark.parametrize("n", [17, 33, 64, 100, 125, 128])
def test_cholesky_tile(torch_gpu, n, nugget, mode):
    for seed in range(5):
        A = kernel_matrix(n, nugget, seed)
        np.linalg.cholesky(A)
        L = np.tril(factor("chol", A, mode))
        assert np.all(np.abs(product(L, L.T) - A) <= bound(n, np.abs(L) @ np.abs(L).T))


@pytest.mark.parametrize("mode", ["eager", "tiled", "subgraph"])
@pytest.mark.parametrize("nugget", [1e-6, 1e-8, 1e-10, 1e-12, 1e-13, None])
@pytest.mark.parametrize("n", [17, 33, 64, 100, 125, 128])
def test_lu_tile(torch_gpu, n, nugget, mode):
    """Kernel matrices, and (None) uniform ones without any dominance, whose pivots and multipliers vary wildly."""
    for seed in range(5):
        A = np.random.default_rng(seed).uniform(-1, 1, (n, n)) if nugget is None else kernel_matrix(n, nugget, seed)
        F = factor("lu", A, mode)
        L, R = np.tril(F, -1) + np.eye(n), np.triu(F)
        assert np.all(np.abs(product(L, R) - A) <= bound(n, np.abs(L) @ np.abs(R)))


def lu_nopiv(A):
    F = A.copy()
    for c in range(len(F)):
        F[c + 1:, c] /= F[c, c]
        F[c + 1:, c + 1:] -= np.outer(F[c + 1:, c], F[c, c + 1:])
    return F


# the factors a tile solve meets: (side, uplo, trans, diag) and the kind of factor
SOLVES = [("R", "L", "T", "N", "chol"), ("L", "L", "N", "N", "chol"), ("L", "L", "T", "N", "chol"),
          ("L", "L", "N", "U", "lu"), ("R", "U", "N", "N", "lu"), ("L", "U", "N", "N", "lu")]


@pytest.mark.parametrize("side,uplo,trans,diag,kind", SOLVES)
@pytest.mark.parametrize("nugget", [1e-6, 1e-10, 1e-13, None])
@pytest.mark.parametrize("n", [17, 33, 64, 100, 125, 128])
def test_panel_solve(torch_gpu, n, nugget, side, uplo, trans, diag, kind):
    """Right-hand sides whose solution is of order one (what a factorization solves for), on panels of 16 right-hand
    sides and of 64; uniform matrices (None) for LU."""
    import mustard_amd as mu
    rng = np.random.default_rng(n)
    if nugget is None and kind == "chol":
        A = rng.uniform(-1, 1, (n, n))
        T = np.linalg.cholesky(A @ A.T + 1e-10 * np.eye(n))
    else:
        A = rng.uniform(-1, 1, (n, n)) if nugget is None else kernel_matrix(n, nugget, n)
        T = np.linalg.cholesky(A) if kind == "chol" else lu_nopiv(A)
    keep = np.tril if uplo == "L" else np.triu
    dT = mu.to_device(np.asfortranarray(np.where(keep(np.ones((n, n), dtype=bool)), T, np.nan)))
    T = keep(T)
    if diag == "U":
        T[np.arange(n), np.arange(n)] = 1.0
    op = T.T if trans == "T" else T
    for nrhs in (16, 8300):
        Y = rng.uniform(-1, 1, (n, nrhs) if side == "L" else (nrhs, n))
        B = op @ Y if side == "L" else Y @ op
        dB = mu.to_device(np.asfortranarray(B))
        mu.dtrsm(side, uplo, trans, diag, *B.shape, 1.0, mu.ptr(dT), n, mu.ptr(dB), len(B))
        X = mu.to_host(dB)
        some = rng.permutation(nrhs)[:24]
        X, B = (X[:, some], B[:, some]) if side == "L" else (X[some], B[some])
        P, S = (product(op, X), np.abs(op) @ np.abs(X)) if side == "L" else (product(X, op), np.abs(X) @ np.abs(op))
        assert np.all(np.abs(P - B) <= bound(n, S))


@pytest.mark.parametrize("kind", ["chol", "lu"])
@pytest.mark.parametrize("mode", ["eager", "tiled", "subgraph"])
@pytest.mark.parametrize("n", [129, 250, 400])
def test_nested_tile(torch_gpu, n, mode, kind):
    """Tiles nested into blocks of at most 128: factorizations, panel solves and updates together."""
    for nugget in (1e-6, 1e-10, 1e-12):
        A = kernel_matrix(n, nugget, n)
        F = factor(kind, A, mode)
        L, R = (np.tril(F), np.tril(F).T) if kind == "chol" else (np.tril(F, -1) + np.eye(n), np.triu(F))
        assert np.all(np.abs(product(L, R) - A) <= bound(n, np.abs(L) @ np.abs(R)))
