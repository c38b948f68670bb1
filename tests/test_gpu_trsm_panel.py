"""GPU tests of the register panel solves (triangles of order <= 256) around
the edges of their 16 x 16 blocks, their block-count instances and their 64
right-hand sides per item, against numpy.  The triangle's other half and the
padding of both matrices hold NaN."""
import numpy as np
import pytest
import scipy.linalg as sl

from tests.util import EPS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,uplo,trans,diag", [("L", "L", "N", "U"), ("R", "U", "N", "N"), ("R", "L", "T", "N"),
                                                  ("L", "U", "N", "N"), ("L", "L", "T", "N"), ("R", "U", "T", "U")])
@pytest.mark.parametrize("order", [1, 16, 17, 32, 33, 49, 64, 65, 96, 97, 127, 128, 129, 177, 192, 193, 241, 255, 256])
def test_panel_solve_orders(torch_gpu, side, uplo, trans, diag, order):
    import mustard_amd as mu
    rng = np.random.default_rng(order)
    for nrhs in (1, 16, 17, 63, 65, 130):
        pad_t, pad_z, alpha = order % 3, nrhs % 4, 0.5
        T = rng.uniform(-1, 1, (order, order)) / order
        T[np.arange(order), np.arange(order)] = 2.0 + rng.uniform(0, 1, order)
        keep = np.tril if uplo == "L" else np.triu
        buf = np.full((order + pad_t, order), np.nan, order="F")
        buf[:order] = np.where(keep(np.ones((order, order), dtype=bool), -1 if diag == "U" and uplo == "L" else
                                    1 if diag == "U" else 0), T, np.nan)
        m, n = (order, nrhs) if side == "L" else (nrhs, order)
        B = rng.uniform(-1, 1, (m, n))
        zb = np.full((m + pad_z, n), np.nan, order="F")
        zb[:m] = B
        dT, dB = mu.to_device(buf), mu.to_device(zb)
        mu.dtrsm(side, uplo, trans, diag, m, n, alpha, mu.ptr(dT), order + pad_t, mu.ptr(dB), m + pad_z)
        got = mu.to_host(dB)
        assert np.all(np.isnan(got[m:]))
        X = got[:m]
        Tc = keep(T)
        if diag == "U":
            Tc[np.arange(order), np.arange(order)] = 1.0
        op = Tc.T if trans == "T" else Tc
        # residual of a solve by substitution with block inverses; the blocks
        # (diagonal in [2, 3] or 1, the rest below 1 / order) have condition < 10
        R, S = (op @ X - alpha * B, np.abs(op) @ np.abs(X)) if side == "L" else \
               (X @ op - alpha * B, np.abs(X) @ np.abs(op))
        assert np.all(np.abs(R) <= 10 * (order + 4) * EPS * (S + np.abs(alpha * B)))
