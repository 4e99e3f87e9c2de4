"""Window spread and interp kernels (matrix cores; 2D and 3D) against the
oracle.  They run where the plan's width, points and density make them the
faster ones (win_sort.hip, win_pays); the shapes here lie just inside that rule,
at every kernel width they are built for.

* spread alone (gpu_spreadinterponly = 1) against the oracle's FP64 spread with
  the plan's kernel: FP32 products of three rounded weights and a strength, each
  within 2^-24, and sums of up to a window's points in FP32: 8e-7, the bar of the
  other FP32 spreads; FP64 1e-12 as they have.  A systematic scale error is held to
  3e-7 / 1e-12.
* type 2 and type 1 transforms against the oracle pipeline: tol/5, or 5e-7 (the
  FP32 FFT and deconvolution at these sizes) / 1e-13 where that is larger, as for
  the other kernels.
* points on the period's edges, beside cells and half cells, outside [-pi, pi) (up to 3 pi)
  and repeated; odd mode counts; a batch that is no multiple of the transforms
  that share weights; fewer points after more."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_util as G
from tests.conftest import rel_l2, scale_err

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64


def _tol(dtype, ns):
    return 1.5 * 10.0 ** (1 - ns)  # ceil(-log10(tol / 10)) = ns


def _pts(dim, M, dtype, nf, seed):
    """Half uniform, a quarter in two clusters, and special points: the
    period's edges, 1/1000 of a cell beside cells and cell middles (where a tap
    enters the support; nearer, the oracle's unclamped square root is NaN), copies of
    one point, and points up to 3 pi away from 0."""
    u = G.uniform_pts(M // 2, dim, dtype, seed)
    cl = G.clustered_pts(M // 4, dim, dtype, seed, ncl=2, sigma=0.2)
    rng = np.random.default_rng(seed + 5)
    n = M - M // 2 - M // 4
    out = []
    for d in range(dim):
        s = rng.uniform(-3 * np.pi, 3 * np.pi, n).astype(dtype)
        cell = rng.integers(0, 2 * nf[d], n // 4) / 2 + rng.choice([-1e-3, 1e-3], n // 4)
        s[: n // 4] = (cell / nf[d] * 2 * np.pi - np.pi).astype(dtype)
        s[n // 4: n // 2] = dtype(0.3)
        top = np.nextafter(dtype(np.pi), dtype(0))
        s[n // 2: n // 2 + 8] = [-top, top, -top, top, 0, 0, top, -top]
        out.append(np.concatenate([u[d], cl[d], s.astype(dtype)]))
    return out


SPREAD = ([(3, F32, ns, (40, 33, 28), 60000) for ns in (6, 7, 8)] +
          [(3, F64, ns, (36, 29, 26), 20000) for ns in (4, 7, 10, 11, 12, 13)] +
          [(2, F32, ns, (64, 51), 4200000 // (ns * ns // 49)) for ns in (7, 8)] +
          [(2, F64, ns, (60, 47), 1 + 100000000 // (ns * ns)) for ns in (9, 13)])


@pytest.mark.parametrize("case", SPREAD, ids=lambda c: f"{c[0]}d-{np.dtype(c[1]).name}-ns{c[2]}")
def test_window_spread_only(torch_dev, case):
    dim, dtype, ns, nm, M = case
    print(f"window spread {case}", flush=True)
    tol = _tol(dtype, ns)
    pts = _pts(dim, M, dtype, nm, 7)
    c = G.strengths(M, dtype, 7)
    fw, plan = G.run_type1(torch_dev, pts, c, nm, tol, dtype, gpu_spreadinterponly=1)
    assert plan.info()["ns"] == ns
    ref = O.spread(pts, c, list(nm), O.setup_spreader(tol, dtype == F32))
    single = dtype == F32
    assert rel_l2(fw, ref) < (8e-7 if single else 1e-12)
    assert scale_err(fw, ref) < (3e-7 if single else 1e-12)


FULL = [
    # type, dim, dtype, ns, modes, M, ntr
    (2, 3, F32, 6, (21, 16, 18), 200000, 1),
    (2, 3, F32, 8, (17, 16, 15), 200003, 3),
    (2, 3, F64, 7, (17, 15, 18), 200000, 1),
    (2, 3, F64, 10, (16, 15, 13), 200000, 2),
    (2, 3, F64, 13, (14, 13, 15), 200000, 1),
    (2, 2, F32, 6, (80, 71), 2800000, 4),
    (2, 2, F64, 10, (50, 41), 500001, 3),
    (2, 2, F64, 13, (45, 40), 600000, 1),
    (1, 2, F32, 6, (60, 77), 1200000, 5),
    (1, 2, F32, 7, (33, 40), 1400000, 3),
    (1, 3, F32, 6, (20, 24, 15), 60000, 2),
    (1, 3, F64, 9, (16, 13, 21), 20001, 3),
]


@pytest.mark.parametrize("case", FULL,
                         ids=lambda c: f"t{c[0]}-{c[1]}d-{np.dtype(c[2]).name}-ns{c[3]}-x{c[6]}")
def test_window_transforms(torch_dev, case):
    ty, dim, dtype, ns, nm, M, ntr = case
    print(f"window transform {case}", flush=True)
    tol = _tol(dtype, ns)
    single = dtype == F32
    pts = _pts(dim, M, dtype, [2 * n for n in nm], 11)
    P = O.Plan(ty, list(nm), tol, single=single)
    bar = max(tol / 5, 5e-7 if single else 1e-13)
    if ty == 1:
        c = G.strengths(M, dtype, 11, ntr)
        got, plan = G.run_type1(torch_dev, pts, c, nm, tol, dtype, ntr, maxbatchsize=0)
        for t in (0, ntr - 1):
            ref = P.type1(pts, c.reshape(ntr, M)[t])
            assert rel_l2(got.reshape(ntr, -1)[t], ref) < bar
    else:
        fk = G.modes(nm[::-1], dtype, 11, ntr)
        got, plan = G.run_type2(torch_dev, pts, fk, tol, dtype, ntr, maxbatchsize=0)
        for t in (0, ntr - 1):
            ref = P.type2(pts, fk.reshape((ntr,) + tuple(nm[::-1]))[t])
            assert rel_l2(got.reshape(ntr, M)[t], ref) < bar
    assert plan.info()["ns"] == ns


def test_window_changing_points(torch_dev):
    """One plan, new points of other counts: from the window kernels to the
    per-point ones (500 points; their accuracy has its own tests) and back, and more
    points than before."""
    import torch
    from cufinufft_amd import cufinufft
    nm, tol = (30, 24, 22), 2e-6
    plan = cufinufft(1, nm[::-1], eps=tol, dtype=F32)
    P = O.Plan(1, list(nm), tol, single=True)
    for k, M in enumerate((40000, 500, 40000, 90001)):
        print("window points", M, flush=True)
        pts = _pts(3, M, F32, [2 * n for n in nm], 20 + k)
        c = G.strengths(M, F32, 20 + k)
        plan.set_pts(*[G.to_dev(p, torch_dev) for p in pts[::-1]])
        fk = torch.zeros(nm[::-1], dtype=torch.complex64, device=torch_dev)
        plan.execute(G.to_dev(c, torch_dev), fk)
        torch.cuda.synchronize()
        if M != 500:
            assert rel_l2(fk.cpu().numpy(), P.type1(pts, c)) < 5e-7


@pytest.mark.parametrize("dtype,ns,ntr,M", [(F32, 7, 4, 1100000), (F32, 7, 7, 600000),
                                            (F32, 8, 13, 300000), (F64, 9, 6, 210000),
                                            (F64, 13, 4, 160000)])
def test_window_packed_batch(torch_dev, dtype, ns, ntr, M):
    """Packed strengths of 2D batches, whole and partly filled packs, on points that
    leave gaps of one and more windows along y (rows taken over, or all flushed)."""
    print(f"window batch {dtype} {ns} {ntr}", flush=True)
    nm, tol, single = (40, 66), _tol(dtype, ns), dtype == F32
    pts = _pts(2, M, dtype, [2 * n for n in nm], 5)
    u = pts[1].astype(np.float64) / (2 * np.pi) + 0.5  # bands of y: 0.1, a gap of 0.06, ...
    u = np.where((u > 0.1) & (u < 0.16), 0.05, np.where((u > 0.4) & (u < 0.65), 0.7, u))
    pts[1] = ((u - 0.5) * (2 * np.pi)).astype(dtype)
    P = O.Plan(1, list(nm), tol, single=single)
    c = G.strengths(M, dtype, 5, ntr)
    got, _ = G.run_type1(torch_dev, pts, c, nm, tol, dtype, ntr, maxbatchsize=ntr)
    bar = max(tol / 5, 5e-7 if single else 1e-13)
    for t in range(ntr):
        ref = P.type1(pts, c.reshape(ntr, M)[t])
        assert rel_l2(got.reshape(ntr, -1)[t], ref) < bar
