"""GPU tests of nested factorizations lowered by whole panels, and of the
per-XCD item order of a batch: the same factors, to the bit, as the
persistent scheduler computes block by block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(kinds, ns, mode, host):
    from mustard_amd.batch import Batch
    b = Batch(kinds, ns, [1] * len(ns), mode=mode)
    b.load(host)
    b.launch()
    out, infos = b.buf.cpu().numpy(), b.infos()
    b.close()
    return out, infos


@pytest.mark.parametrize("ns", [[129], [255], [257], [385, 1], [512, 500], [1025],
                                [97 + 3 * i % 190 for i in range(70)]])
@pytest.mark.parametrize("kind", ["chol", "lu"])
def test_panels_match_blocks(torch_gpu, kind, ns):
    from mustard_amd.batch import make_problems
    kinds = [kind] * len(ns)
    host = make_problems(kinds, ns, len(ns))
    got, infos = _run(kinds, ns, "tiled", host)
    ref, _ = _run(kinds, ns, "subgraph", host)
    assert not np.any(infos)
    assert np.array_equal(got, ref)
