"""GPU tests of the one-workgroup factorizations (GETRF / POTRF of order <=
128) around the edges of their 16 x 16 blocks: every block count and the
orders next to it, in a buffer filled with NaN, and the info they report for
a failing column in any block."""
import numpy as np
import pytest

from tests.util import EPS

pytestmark = pytest.mark.gpu

ORDERS = [1, 2, 15, 16, 17, 31, 33, 48, 63, 65, 80, 81, 95, 97, 112, 113, 127, 128]


def _run(kind, A, pad):
    import mustard_amd as mu
    n = A.shape[0]
    buf = np.full((n + pad, n), np.nan, order="F")
    buf[:n] = A
    dA, info = mu.to_device(buf), mu.info_cell()
    if kind == "lu":
        mu.dgetrf_nopiv(n, mu.ptr(dA), n + pad, mu.ptr(info))
    else:
        mu.dpotrf("L", n, mu.ptr(dA), n + pad, mu.ptr(info))
    got = mu.to_host(dA)
    assert np.all(np.isnan(got[n:]))
    return got[:n], mu.info_value(info)


@pytest.mark.parametrize("kind", ["lu", "chol"])
@pytest.mark.parametrize("n", ORDERS)
def test_small_factor_orders(torch_gpu, kind, n):
    """Backward error of the computed factors, elementwise: |A - L U| <= 4 n eps
    |L| |U| (the classical bound gamma_n, with room for the block inverses of a
    diagonally dominant matrix, whose condition number is below 4)."""
    rng = np.random.default_rng(n)
    A = rng.uniform(0.0, 1.0, (n, n)) + n * np.eye(n)
    if kind == "chol":
        A = np.tril(A) + np.tril(A, -1).T
    F, info = _run(kind, A, 3)
    assert info == 0
    if kind == "lu":
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
    else:
        assert np.array_equal(np.triu(F, 1), np.triu(A, 1))
        L, U = np.tril(F), np.tril(F).T
    assert np.all(np.abs(A - L @ U) <= 4 * (n + 4) * EPS * (np.abs(L) @ np.abs(U)))


@pytest.mark.parametrize("kind", ["lu", "chol"])
@pytest.mark.parametrize("n,col", [(40, 0), (40, 15), (64, 16), (100, 37), (125, 96), (128, 127)])
def test_small_factor_info(torch_gpu, kind, n, col):
    """Column `col` is the first that fails: a zero pivot (its row and column
    left of it are zero, so no update touches it) or a negative one."""
    A = np.eye(n) * 3.0
    A[col, col] = 0.0 if kind == "lu" else -1.0
    F, info = _run(kind, A, 0)
    assert info == col + 1
    assert np.allclose(np.diag(F)[:col], 3.0 if kind == "lu" else np.sqrt(3.0), rtol=4 * EPS)
