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
