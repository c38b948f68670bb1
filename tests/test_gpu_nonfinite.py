"""GPU tests of how far a NaN, an infinity or a zero pivot spreads in the
factorizations of order <= 128 and in the panel solves of such triangles: as
with substitution, only to what depends on it.  What does not depend on it keeps
its bits, or (its own row or column) agrees to rounding with the clean run: the
matrices are diagonally dominant, so 1e-12 relative is far above n u = 1.4e-14."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def close(got, ref):
    return np.all(np.abs(got - ref) <= 1e-12 * np.abs(ref).max(initial=0.0))


# (side, uplo, trans, diag), and whether the solve runs from the first row (column) to the last
SOLVES = [("L", "L", "N", "U", True), ("R", "U", "N", "N", True), ("R", "L", "T", "N", True),
          ("L", "U", "N", "N", False), ("L", "L", "T", "N", False)]


@pytest.mark.parametrize("side,uplo,trans,diag,forward", SOLVES)
@pytest.mark.parametrize("order", [5, 16, 33, 100, 128])
def test_panel_solve(torch_gpu, order, side, uplo, trans, diag, forward):
    import mustard_amd as mu
    rng = np.random.default_rng(order)
    T = rng.uniform(-1, 1, (order, order)) / order
    T[np.arange(order), np.arange(order)] = 2.0 + rng.uniform(0, 1, order)
    dT = mu.to_device(np.asfortranarray(T))

    def solve(B):  # B: (right-hand side, row), solved in the order of the rows
        M = B if forward else B[:, ::-1]
        d = mu.to_device(np.asfortranarray(M.T if side == "L" else M))
        m, n = (order, len(B)) if side == "L" else (len(B), order)
        mu.dtrsm(side, uplo, trans, diag, m, n, 1.0, mu.ptr(dT), order, mu.ptr(d), m)
        X = mu.to_host(d)
        X = X.T if side == "L" else X
        return X if forward else X[:, ::-1]

    for nrhs in (20, 8300):
        B = rng.uniform(-1, 1, (nrhs, order))
        clean = solve(B)
        for value in (np.nan, np.inf, -np.inf):
            for r in sorted({0, 3, order // 2, order - 1}):
                for c in (3, 17):
                    C = B.copy()
                    C[c, r] = value
                    X = solve(C)
                    others = np.arange(nrhs) != c
                    assert np.array_equal(X[others], clean[others])
                    assert close(X[c, :r], clean[c, :r])
                    assert np.array_equal(X[c, r], value, equal_nan=True)
                    assert not np.any(np.isfinite(X[c, r]))
    if diag == "N":
        r = order // 2
        p = r if forward else order - 1 - r
        T[p, p] = 0.0
        dT = mu.to_device(np.asfortranarray(T))
        X = solve(B)
        assert close(X[:, :r], clean[:, :r]) and np.all(np.isinf(X[:, r]))


def factor(kind, A):
    import mustard_amd as mu
    n, dA, info = len(A), mu.to_device(np.asfortranarray(A)), mu.info_cell()
    if kind == "lu":
        mu.dgetrf_nopiv(n, mu.ptr(dA), n, mu.ptr(info))
    else:
        mu.dpotrf("L", n, mu.ptr(dA), n, mu.ptr(info))
    F = mu.to_host(dA)
    return (F if kind == "lu" else np.tril(F)), mu.info_value(info)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("kind,i,k", [("chol", 70, 37), ("chol", 127, 0), ("chol", 17, 15), ("lu", 70, 37),
                                      ("lu", 37, 70), ("lu", 127, 1), ("lu", 2, 127), ("lu", 16, 14)])
def test_factor_entry(torch_gpu, kind, i, k, value):
    """A(i, k), in another block than the diagonal's: nothing before it in its row (lower part) or column (upper),
    and no other row and column before the later of i and k.  The rows and columns of the latter's 16 x 16 block are
    solved with a triangle that holds a NaN then, by substitution, so they agree to rounding; inside that diagonal
    block the elimination multiplies the rows above a NaN pivot row by zero (not looked at)."""
    n = 128
    A = np.random.default_rng(7).uniform(0.0, 1.0, (n, n)) + n * np.eye(n)
    A = A if kind == "lu" else np.tril(A) + np.tril(A, -1).T
    clean, info = factor(kind, A)
    assert info == 0
    A[i, k] = value
    F, _ = factor(kind, A)
    line, first, last = (F[i], clean[i], i) if i > k else (F[:, k], clean[:, k], k)
    assert close(line[:min(i, k)], first[:min(i, k)]) and not np.isfinite(line[min(i, k)])
    rows = np.arange(n)
    untouched = (np.minimum(rows[:, None], rows[None]) < last) & ~((rows == last)[:, None] if i > k else
                                                                   (rows == last)[None])
    here = rows // 16 == last // 16
    solved = untouched & (here[:, None] ^ here[None]) & (np.minimum(rows[:, None], rows[None]) >= last // 16 * 16)
    untouched &= np.minimum(rows[:, None], rows[None]) < last // 16 * 16
    assert np.array_equal(F[untouched], clean[untouched])
    assert close(F[solved], clean[solved])


def test_zero_pivot(torch_gpu):
    """LU with an exactly zero pivot in column 37: info, and the blocks below and right of its diagonal block before it."""
    n, c = 128, 37
    A = np.random.default_rng(8).uniform(0.0, 1.0, (n, n)) + n * np.eye(n)
    A[c, :c + 1] = A[:c + 1, c] = 0.0
    F, info = factor("lu", A)
    A[c, c] = 1.0
    ref, _ = factor("lu", A)
    assert info == c + 1
    assert close(F[48:, :c], ref[48:, :c]) and close(F[:c, 48:], ref[:c, 48:])
