"""GPU test of the batched residual kernel around its 64-row and 16-column
groups, with an order beyond one pass of its workgroups, and a NaN that has to
reach the norms."""
import numpy as np
import pytest

from tests.util import EPS

pytestmark = pytest.mark.gpu


def test_batch_residual_orders(torch_gpu):
    import mustard_amd as mu
    torch = torch_gpu
    ns = [1, 15, 16, 17, 63, 64, 65, 80, 129, 1024, 1100, 33]
    rng = np.random.default_rng(3)
    As = [np.asfortranarray(rng.uniform(-1, 1, (n, n))) for n in ns]
    xs, bs = [rng.uniform(-1, 1, n) for n in ns], [rng.uniform(-1, 1, n) for n in ns]
    xs[-1][5] = np.nan
    aoff = np.concatenate([[0], np.cumsum([n * n for n in ns])])[:-1]
    voff = np.concatenate([[0], np.cumsum(ns)])[:-1]
    dev = dict(device="cuda")
    A = torch.from_numpy(np.concatenate([a.reshape(-1, order="F") for a in As])).to("cuda")
    X, B = (torch.from_numpy(np.concatenate(v)).to("cuda") for v in (xs, bs))
    R = torch.full_like(X, np.nan)
    norms = torch.full((4 * len(ns),), np.nan, dtype=torch.float64, **dev)
    d = [torch.tensor(ns, dtype=torch.int32, **dev)] + [torch.tensor(o, dtype=torch.int64, **dev) for o in (aoff, voff)]
    mu.call("mu_batch_residual", len(ns), mu.ptr(d[0]), mu.ptr(d[1]), mu.ptr(d[2]), mu.ptr(A), mu.ptr(X), mu.ptr(B),
            mu.ptr(R), mu.ptr(norms), mu.stream_handle())
    torch.cuda.synchronize()
    r, nm = R.cpu().numpy(), norms.view(-1, 4).cpu().numpy()
    for p, n in enumerate(ns):
        got = r[voff[p]:voff[p] + n]
        if p == len(ns) - 1:
            assert np.all(np.isnan(got)) and np.isnan(nm[p, 0]) and np.isnan(nm[p, 1])
            continue
        bound = (n + 2) * EPS * (np.abs(As[p]) @ np.abs(xs[p]) + np.abs(bs[p]))
        assert np.all(np.abs(got - (bs[p] - As[p] @ xs[p])) <= bound)
        assert nm[p, 0] == np.max(np.abs(got)) and nm[p, 1] == np.max(np.abs(xs[p]))
        assert abs(nm[p, 2] - np.linalg.norm(As[p], np.inf)) <= n * EPS * nm[p, 2]
        assert nm[p, 3] == np.max(np.abs(bs[p]))
