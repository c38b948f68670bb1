"""GPU tests of the panel solves with 16 right-hand sides on four waves: the
same results, to the bit, as the 64-wide panels a call of many right-hand
sides runs on, at the edges of the 16-row blocks and of the rows per wave."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDE = 64 * 256 + 3  # right-hand sides that run on 64-wide panels


@pytest.mark.parametrize("side,uplo,trans,diag", [("L", "L", "N", "U"), ("R", "U", "N", "N"), ("R", "L", "T", "N"),
                                                  ("L", "U", "N", "N"), ("L", "L", "T", "N"), ("R", "U", "T", "U")])
@pytest.mark.parametrize("order", [1, 15, 16, 31, 33, 64, 65, 100, 127, 128, 129, 143, 192, 193, 209, 250, 256])
def test_split_panels_match_wide_panels(torch_gpu, side, uplo, trans, diag, order):
    import torch

    import mustard_amd as mu
    rng = np.random.default_rng(order)
    T = rng.uniform(-1, 1, (order, order)) / order
    T[np.arange(order), np.arange(order)] = 2.0 + rng.uniform(0, 1, order)
    keep = np.tril if uplo == "L" else np.triu
    dT = mu.to_device(np.where(keep(np.ones((order, order), dtype=bool)), T, np.nan))
    g = torch.Generator(device="cuda")
    g.manual_seed(order)
    # tensor B holds the column-major matrix: (right-hand sides, order) on the left, its transpose on the right
    shape = (WIDE, order) if side == "L" else (order, WIDE)
    B = 2.0 * torch.rand(shape, dtype=torch.float64, device="cuda", generator=g) - 1.0
    wide = B.clone()
    m, n = (order, WIDE) if side == "L" else (WIDE, order)
    mu.dtrsm(side, uplo, trans, diag, m, n, 0.5, mu.ptr(dT), order, mu.ptr(wide), m)
    for first, nrhs in ((0, 1), (1, 15), (16, 16), (32, 17), (49, 130)):
        cut = slice(first, first + nrhs)
        part = (B[cut] if side == "L" else B[:, cut]).contiguous()
        m, n = (order, nrhs) if side == "L" else (nrhs, order)
        mu.dtrsm(side, uplo, trans, diag, m, n, 0.5, mu.ptr(dT), order, mu.ptr(part), m)
        assert torch.equal(part, wide[cut] if side == "L" else wide[:, cut])
