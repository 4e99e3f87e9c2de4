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


@pytest.mark.parametrize("dtype,tol,bar", [(np.float32, 1e-6, 2e-6), (np.float64, 1e-9, 1e-12)])
@pytest.mark.parametrize("graph", [False, True])
def test_group_window_spread(torch_dev, dtype, tol, bar, graph):
    """Type-1 groups whose members' points fill the windows, against each member's own
    execute (relative L2; weights and sums of either path agree to rounding), also
    after a member's points were set again."""
    import torch
    from cufinufft_amd import cufinufft
    from cufinufft_amd.cufinufft import cufinufft_group
    plans, cs, fks, sizes = [], [], [], [(33, 40), (64, 51), (97, 16), (20, 130)]
    for k, nm in enumerate(sizes):
        m, ntr = 60001 + 1777 * k, 1 + k % 3
        plan = cufinufft(1, nm, n_trans=ntr, eps=tol, dtype=dtype, gpu_method=2, maxbatchsize=ntr)
        pts = (G.uniform_pts if k % 2 else G.clustered_pts)(m, 2, dtype, 3 + k)
        plan.set_pts(*[G.to_dev(p, torch_dev) for p in pts])
        plans.append(plan)
        cs.append(G.to_dev(G.strengths(m, dtype, k, ntr), torch_dev))
        fks.append(torch.empty((ntr,) + nm, dtype=cs[-1].dtype, device=torch_dev))
    group = cufinufft_group(plans, cs, fks)
    for again in range(3):
        if again == 2:  # other points of a member
            m = cs[1].numel() // plans[1].n_trans
            plans[1].set_pts(*[G.to_dev(p, torch_dev) for p in G.uniform_pts(m, 2, dtype, 77)])
        for o in fks:
            o.fill_(7)
        group.execute(use_graph=graph)
        torch.cuda.synchronize()
        for p, c, f in zip(plans, cs, fks):
            want = torch.empty_like(f)
            p.execute(c, want)
            assert (f - want).norm() < bar * want.norm()
