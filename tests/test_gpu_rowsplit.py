"""Deconvolve and amplify passes whose rows are split over workgroups: 1D (a
single row) and transforms of few rows, around the 256-cell pieces, and a row
long enough that its pieces are strided, against an FP64 direct sum at sampled
modes.  FP64 at tol 1e-9; bound 1e-8 (ten times tol) per axis of the largest
output."""
import numpy as np
import pytest

from tests import gpu_util as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes", [(1,), (255,), (257,), (1024,), (2_100_001,), (3, 5000),
                                   (700, 3), (5, 2, 129)])
@pytest.mark.parametrize("ntr", [1, 3])
def test_row_split(torch_dev, modes, ntr):
    dim, m, tol = len(modes), 400, 1e-9
    rng = np.random.default_rng(11 * dim + modes[0])
    x = rng.uniform(-np.pi, np.pi, (dim, m))
    # both ends, the middle, the edge of a piece and random modes of every axis
    pick = [np.unique(np.concatenate([[0, n - 1, n // 2, min(255, n - 1), min(256, n - 1)],
                                      rng.integers(0, n, 12)])) for n in modes]
    at = (slice(None),) + np.ix_(*pick)
    k = np.stack(np.meshgrid(*[p - n // 2 for p, n in zip(pick, modes)], indexing="ij"), -1)
    phase = np.exp(1j * (k @ x))  # [picked modes..., point]
    pts, shape = list(x[::-1]), modes[::-1]

    c = rng.standard_normal((ntr, m)) + 1j * rng.standard_normal((ntr, m))
    out, _ = G.run_type1(torch_dev, pts, c.ravel(), shape, tol, np.float64, ntr=ntr)
    ref = np.moveaxis(phase @ c.T, -1, 0)
    err = np.abs(out.reshape((ntr,) + modes)[at] - ref).max()
    assert err < 1e-8 * dim * np.abs(ref).max()

    # type 2 of modes that are zero but for the picked ones
    f = np.zeros((ntr,) + modes, np.complex128)
    f[at] = rng.standard_normal((ntr,) + phase.shape[:-1])
    out, _ = G.run_type2(torch_dev, pts, f if ntr > 1 else f[0], tol, np.float64, ntr=ntr)
    ref = f[at].reshape(ntr, -1) @ phase.conj().reshape(-1, m)
    assert np.abs(out.reshape(ntr, m) - ref).max() < 1e-8 * dim * np.abs(ref).max()
