"""One-pass bin sorts against the oracle's, exactly: bin tables, subproblem
map, and input order inside every bin.  Sizes at the edges of the 1024- and
4096-point tiles, of the rule between them (256 CUs x 4096 points; the counts
of 1024-point tiles within M) and of digit counts (2 to 977 bins)."""
import numpy as np
import pytest

from tests import gpu_util as G
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,m", [
    (1, 520, 1), (1, 520, 1023), (1, 1500, 1024), (1, 1500, 1025), (1, 40_000, 4097),
    (1, 500_000, 1023), (1, 500_000, 5000), (1, 500_000, 1 << 20), (1, 500_000, (1 << 20) + 1),
    (2, 64, 4001), (2, 500, 300_001), (3, 30, 70_000)])
@pytest.mark.parametrize("dist", ["uniform", "clustered"])
def test_one_pass_sort(torch_dev, dim, n, m, dist):
    from cufinufft_amd import cufinufft
    pts = (G.uniform_pts(m, dim, np.float32, 5) if dist == "uniform" else
           G.clustered_pts(m, dim, np.float32, 5, ncl=2, sigma=0.01))
    plan = cufinufft(1, (n,) * dim, eps=1e-4, dtype=np.float32, gpu_method=2,
                     gpu_maxsubprobsize=100)
    # larger sets first: every table has to be written anew
    plan.set_pts(*[G.to_dev(np.concatenate([p, p])[:2 * m], torch_dev) for p in pts[::-1]])
    plan.set_pts(*[G.to_dev(p, torch_dev) for p in pts[::-1]])
    inf, got = plan.info(), plan.sort_arrays()
    ref = O.bin_sort(pts, inf["nf"][:dim], inf["binsize"][:dim], maxsub=100)
    nbins = ref["binsize"].size
    assert nbins <= 1024
    np.testing.assert_array_equal(got["binsize"], ref["binsize"])
    np.testing.assert_array_equal(got["binstart"], ref["binstart"])
    np.testing.assert_array_equal(got["s2b"], np.repeat(np.arange(nbins), ref["numsub"]))
    np.testing.assert_array_equal(got["idx"], np.argsort(ref["binof"], kind="stable"))
