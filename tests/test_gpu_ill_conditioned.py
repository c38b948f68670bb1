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
