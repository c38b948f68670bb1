"""GPU tests of tiles whose columns lie so far apart that their elements'
offsets exceed 32 bits: the same results, to the bit, as in a compact copy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tall(torch_gpu):
    """47 GB of device memory, mostly untouched."""
    torch = torch_gpu
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 47 GB of free device memory")
    buf = torch.empty(47 << 27, dtype=torch.float64, device="cuda")
    yield buf
    del buf
    torch.cuda.empty_cache()


# the last column's offset, a 16-wide block's and a 4-wide one's past 2^32
@pytest.mark.parametrize("n,lda", [(128, 34_000_003), (128, 48_000_000), (17, 290_000_001), (4, 1_440_000_000)])
@pytest.mark.parametrize("kind", ["lu", "chol"])
def test_small_factor_tall(torch_gpu, tall, kind, n, lda):
    import mustard_amd as mu
    torch = torch_gpu
    rng = np.random.default_rng(n)
    A = rng.uniform(0.0, 1.0, (n, n)) + n * np.eye(n)
    flat = mu.to_device(np.asfortranarray(np.tril(A) + np.tril(A, -1).T if kind == "chol" else A))
    far = torch.as_strided(tall, (n, n), (lda, 1))
    far.copy_(flat)
    for p, ld in ((flat, n), (far, lda)):
        info = mu.info_cell()
        if kind == "lu":
            mu.dgetrf_nopiv(n, mu.ptr(p), ld, mu.ptr(info))
        else:
            mu.dpotrf("L", n, mu.ptr(p), ld, mu.ptr(info))
        assert mu.info_value(info) == 0
    assert torch.equal(far, flat)


# a 16 x 16 block of the triangle past 2^32 bytes, where panels of 16 right-hand
# sides and of 64 part; then right-hand sides past 2^32 elements
@pytest.mark.parametrize("order,lda,ldb", [(17, 60_000_000, 0), (58, 36_000_000, 0), (20, 0, 290_000_001)])
@pytest.mark.parametrize("side,uplo,trans,diag", [("L", "L", "N", "U"), ("R", "U", "N", "N"), ("L", "U", "N", "N"),
                                                  ("L", "L", "T", "N")])
def test_panel_solve_tall(torch_gpu, tall, side, uplo, trans, diag, order, lda, ldb):
    import mustard_amd as mu
    torch = torch_gpu
    if ldb and side == "R":
        pytest.skip("such a right-hand side is 46 GB for four rows of the triangle")
    rng = np.random.default_rng(order)
    T = rng.uniform(-1, 1, (order, order)) / order + 2.0 * np.eye(order)
    flat = mu.to_device(np.asfortranarray(T))
    for nrhs in (16, 17) if ldb else (1, 16, 17, 700):
        B = rng.uniform(-1, 1, (order, nrhs) if side == "L" else (nrhs, order))
        m, n = B.shape
        near = mu.to_device(np.asfortranarray(B))
        mu.dtrsm(side, uplo, trans, diag, m, n, 0.5, mu.ptr(flat), order, mu.ptr(near), m)
        if ldb:
            far = torch.as_strided(tall, (n, m), (ldb, 1))
            far.copy_(mu.to_device(np.asfortranarray(B)))
            mu.dtrsm(side, uplo, trans, diag, m, n, 0.5, mu.ptr(flat), order, mu.ptr(far), ldb)
        else:
            tri = torch.as_strided(tall, (order, order), (lda, 1))
            tri.copy_(flat)
            far = mu.to_device(np.asfortranarray(B))
            mu.dtrsm(side, uplo, trans, diag, m, n, 0.5, mu.ptr(tri), lda, mu.ptr(far), m)
        assert torch.equal(far, near)
