"""GPU tests of the FP64 GEMM / SYRK blocks at the edges of their 64 x 64 x 16
tiling: orders around one and two blocks, k around whole slices of 16, odd
leading dimensions and offsets, against numpy.  The operands sit in buffers
filled with NaN, so a read outside them or a write outside C shows."""
import numpy as np
import pytest

from tests.util import EPS

pytestmark = pytest.mark.gpu


def _embed(M, pad, rng_off):
    """M inside a NaN-filled column-major buffer: (buffer, element offset, ld)."""
    m, n = M.shape
    ld = m + pad
    buf = np.full((ld, n + 1), np.nan, order="F")
    buf[rng_off:rng_off + m, :n] = M
    return buf, rng_off, ld


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(64, 64, 16), (65, 64, 17), (64, 65, 31), (127, 66, 32), (129, 191, 15),
                                   (63, 200, 48), (200, 63, 48), (67, 130, 100), (192, 128, 160)])
def test_gemm_block_edges(torch_gpu, ta, tb, m, n, k):
    import mustard_amd as mu
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    A = rng.uniform(-1, 1, (m, k) if ta == "N" else (k, m))
    B = rng.uniform(-1, 1, (k, n) if tb == "N" else (n, k))
    C = rng.uniform(-1, 1, (m, n))
    for pad, off, alpha, beta in ((3, 1, -1.0, 1.0), (2, 0, 0.75, -0.5), (5, 2, 1.0, 0.0)):
        bufs = [_embed(M, pad, off) for M in (A, B, C)]
        if beta == 0.0:  # C is not read then
            bufs[2][0][:] = np.nan
        dev = [mu.to_device(b) for b, _, _ in bufs]
        (_, oa, lda), (_, ob, ldb), (cb, oc, ldc) = bufs
        mu.dgemm(ta, tb, m, n, k, alpha, mu.ptr(dev[0], oa), lda, mu.ptr(dev[1], ob), ldb, beta,
                 mu.ptr(dev[2], oc), ldc)
        torch_gpu.cuda.synchronize()
        got = mu.to_host(dev[2])
        a, b = (A if ta == "N" else A.T), (B if tb == "N" else B.T)
        ref = alpha * (a @ b) + (beta * C if beta != 0.0 else 0.0)
        # k products and two more roundings on each side
        bound = 2 * (k + 3) * EPS * (abs(alpha) * (np.abs(a) @ np.abs(b)) + abs(beta) * np.abs(C))
        assert np.all(np.abs(got[oc:oc + m, :n] - ref) <= bound)
        out = np.ones(got.shape, dtype=bool)
        out[oc:oc + m, :n] = False
        assert np.array_equal(got[out], cb[out], equal_nan=True)


@pytest.mark.parametrize("n,k", [(64, 16), (65, 33), (127, 20), (130, 125), (193, 64), (63, 64)])
def test_syrk_block_edges(torch_gpu, n, k):
    """Lower triangle only: the strict upper part keeps its bits."""
    import mustard_amd as mu
    rng = np.random.default_rng(n + k)
    A, C = rng.uniform(-1, 1, (n, k)), rng.uniform(-1, 1, (n, n))
    (ab, oa, lda), (cb, oc, ldc) = _embed(A, 3, 1), _embed(C, 1, 0)
    dA, dC = mu.to_device(ab), mu.to_device(cb)
    mu.dsyrk("L", "N", n, k, -1.0, mu.ptr(dA, oa), lda, 1.0, mu.ptr(dC, oc), ldc)
    torch_gpu.cuda.synchronize()
    got = mu.to_host(dC)
    lo = np.zeros(got.shape, dtype=bool)
    lo[:n, :n] = np.tril(np.ones((n, n), dtype=bool))
    ref, bound = C - A @ A.T, 2 * (k + 3) * EPS * (np.abs(A) @ np.abs(A).T + np.abs(C))
    t = lo[:n, :n]
    assert np.all(np.abs(got[:n, :n] - ref)[t] <= bound[t])
    assert np.array_equal(got[~lo], cb[~lo], equal_nan=True)
