"""GPU tests of the FP64 updates with fewer than 64 rows or columns, or k < 16, at
even sizes in aligned buffers, where the operands are read in pairs: against
numpy, and the same bits as from buffers with odd leading dimensions."""
import numpy as np
import pytest

from tests.util import EPS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(2, 18, 2), (62, 130, 34), (130, 62, 30), (48, 48, 48), (128, 128, 14),
                                   (66, 70, 2), (64, 20, 250), (30, 200, 16)])
def test_even_small_blocks(torch_gpu, ta, tb, m, n, k):
    import mustard_amd as mu
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    A = rng.uniform(-1, 1, (m, k) if ta == "N" else (k, m))
    B = rng.uniform(-1, 1, (k, n) if tb == "N" else (n, k))
    C = rng.uniform(-1, 1, (m, n))
    out = []
    for pad in (2, 1):  # even sizes: an even leading dimension, an odd one
        bufs = []
        for M in (A, B, C):
            b = np.full((M.shape[0] + pad, M.shape[1]), np.nan, order="F")
            b[:len(M)] = M
            bufs.append(mu.to_device(b))
        mu.dgemm(ta, tb, m, n, k, -0.5, mu.ptr(bufs[0]), len(A) + pad, mu.ptr(bufs[1]), len(B) + pad, 0.75,
                 mu.ptr(bufs[2]), m + pad)
        got = mu.to_host(bufs[2])
        assert np.all(np.isnan(got[m:]))
        out.append(got[:m])
    a, b = (A if ta == "N" else A.T), (B if tb == "N" else B.T)
    # k products and two more roundings on each side
    bound = 2 * (k + 3) * EPS * (0.5 * (np.abs(a) @ np.abs(b)) + 0.75 * np.abs(C))
    assert np.all(np.abs(out[0] - (0.75 * C - 0.5 * (a @ b))) <= bound)
    assert np.array_equal(out[0], out[1])
