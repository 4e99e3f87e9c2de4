"""Plan groups whose zero fill and FFT transposes run as one launch over all
members: 2D and 3D, both types and precisions, members of unequal, odd and tiny
sizes (less than a tile, a tile's edge, several tiles) and several transforms,
against each member's own execute.  Bounds: both run the same kernels on the same
data, apart from the order of the spread's additions, 50 eps of the largest value."""
import numpy as np
import pytest

from tests import gpu_util as G

pytestmark = pytest.mark.gpu

SIZES = {2: [(33, 31), (64, 64), (130, 5), (2, 200), (97, 161)],
         3: [(17, 20, 33), (2, 40, 3), (32, 33, 31), (5, 4, 66)]}


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("typ", [1, 2])
@pytest.mark.parametrize("dtype,tol", [(np.float32, 1e-5), (np.float64, 1e-9)])
@pytest.mark.parametrize("graph", [False, True])
def test_group_passes(torch_dev, dim, typ, dtype, tol, graph):
    import torch
    from cufinufft_amd import cufinufft
    from cufinufft_amd.cufinufft import cufinufft_group
    plans, cs, fks = [], [], []
    for k, nm in enumerate(SIZES[dim]):
        m, ntr = 500 + 1777 * k, 1 + k % 3
        plan = cufinufft(typ, nm, n_trans=ntr, eps=tol, dtype=dtype, gpu_method=2,
                         maxbatchsize=ntr)
        plan.set_pts(*[G.to_dev(p, torch_dev) for p in G.uniform_pts(m, dim, dtype, 3 + k)])
        plans.append(plan)
        cs.append(G.to_dev(G.strengths(m, dtype, k, ntr), torch_dev))
        fks.append(G.to_dev(G.modes((ntr,) + nm, dtype, k), torch_dev))
    outs = fks if typ == 1 else cs
    want = []
    for p, c, f, o in zip(plans, cs, fks, outs):
        p.execute(c, f)
        want.append(o.clone())
        o.zero_()
    group = cufinufft_group(plans, cs, fks)
    for _ in range(3):
        for o in outs:
            o.fill_(7)
        group.execute(use_graph=graph)
        torch.cuda.synchronize()
        for o, w in zip(outs, want):
            assert (o - w).abs().max() <= 50 * np.finfo(dtype).eps * w.abs().max()
