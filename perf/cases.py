"""Performance cases of the NUFFT library: what a program asks of it, from one
small image to 1e8 points, through the public Python entry points.

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges,
``prepare`` / ``run`` the inputs and one pass, ``work`` the bytes and
operations a pass cannot do without, and ``exact`` the transform as an FP64
direct sum (no code of this library).

A case is a dict of plain values.  ``kind`` selects the entry point:

* ``plan``: the ``cufinufft`` class.  The plan is made once; with ``setpts``
  every pass sets new points and executes (points that change with every
  call), without it a pass is one execute (an iterative solver on fixed
  points).
* ``grad``: ``torch_nufft.nufft_type2`` forward and backward, to modes and
  point coordinates, on a trajectory that is new in every step.
* ``group``: a ``cufinufft_group`` of many small independent plans.
"""
import math

import numpy as np
import torch

from cufinufft_amd import cufinufft
from cufinufft_amd.cufinufft import cufinufft_group
from cufinufft_amd.torch_nufft import nufft_type2

_DEV = "cuda"


def _plan_case(name, type, dtype, tol, n, m, dist="uniform", ntransf=1, setpts=False, **opts):
    n = tuple(n) + (1, 1)
    return dict({"name": name, "kind": "plan", "type": type, "dtype": dtype, "tol": tol,
                 "n1": n[0], "n2": n[1], "n3": n[2], "m": m, "dist": dist, "ntransf": ntransf,
                 "setpts": setpts}, **opts)


def listed():
    return [
        # the smallest call: a thumbnail-sized image sampled at a few thousand
        # points, new points every time; latency and launches count
        _plan_case("2d2_f32_tiny", 2, "f32", 1e-4, (64, 50), 4001, setpts=True),
        # a small image gridded from new points (the benchmark's 2D workload)
        _plan_case("2d1_f32_small", 1, "f32", 1e-5, (256, 256), 100_000, setpts=True),
        # a long irregularly sampled signal, double precision
        _plan_case("1d1_f64_signal", 1, "f64", 1e-9, (100_003,), 1_000_000, setpts=True),
        # one reconstruction step of a learned 2D radial trajectory: forward
        # and gradients (the benchmark's differentiable workload)
        {"name": "2d2_f32_radial_grad", "kind": "grad", "dtype": "f32", "tol": 1e-6, "n1": 320,
         "n2": 320, "n3": 1, "spokes": 320, "samples": 640},
        # many small independent images as one group (the benchmark's group)
        {"name": "2d1_f32_group", "kind": "group", "dtype": "f32", "tol": 1e-6, "plans": 48,
         "n_lo": 64, "n_hi": 512, "m_lo": 1000, "m_hi": 1_000_000, "graph": True},
        # many coils / frames on one set of points (the benchmark's batch)
        _plan_case("2d1_f32_coils", 1, "f32", 1e-6, (512, 512), 2_000_000, ntransf=32),
        # 2D evaluation near double precision, odd sizes, new points
        _plan_case("2d2_f64_ragged", 2, "f64", 1e-12, (701, 523), 3_000_000, setpts=True),
        # 3D evaluation of a few volumes, subproblem method asked for
        _plan_case("3d2_f32_volumes", 2, "f32", 1e-5, (160, 160, 160), 4_000_000, ntransf=2,
                   gpu_method=2),
        # 3D double precision gridding of an odd-sized volume, new points
        _plan_case("3d1_f64_ragged", 1, "f64", 1e-9, (97, 128, 75), 2_000_000, setpts=True),
        # 3D single precision gridding with the faster options, new points
        _plan_case("3d1_f32_opts", 1, "f32", 1e-6, (192, 192, 192), 20_000_000, setpts=True,
                   gpu_kerevalmeth=1, tile_slots=True),
        # 3D double precision evaluation at clustered points (the benchmark's
        # type-2 workload), default options
        _plan_case("3d2_f64_clusters", 2, "f64", 1e-9, (128, 128, 128), 10_000_000, "clusters"),
        # the largest: the benchmark's headline workload, default options
        _plan_case("3d1_f32_large", 1, "f32", 1e-5, (256, 256, 256), 100_000_000, "mixed"),
    ]


# ------------------------------------------------------------------- drawing
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(tol):
    return max(2, math.ceil(-math.log10(tol / 10) - 1e-9))


def draw(rng):
    kind = rng.choice(["plan"] * 8 + ["grad", "group"])
    if kind == "grad":
        return {"kind": "grad", "dtype": rng.choice(["f32", "f32", "f64"]),
                "tol": rng.choice([1e-4, 1e-5, 1e-6]), "n1": rng.randint(96, 384),
                "n2": rng.randint(96, 384), "n3": 1, "spokes": rng.randint(48, 400),
                "samples": rng.randint(128, 768)}
    if kind == "group":
        return {"kind": "group", "dtype": "f32", "tol": rng.choice([1e-4, 1e-5, 1e-6]),
                "plans": rng.randint(4, 60), "n_lo": rng.randint(40, 90),
                "n_hi": rng.randint(128, 512), "m_lo": 1000, "m_hi": _log_int(rng, 1e4, 1e6),
                "graph": rng.random() < 0.5}
    dim = rng.choice([1, 2, 2, 3, 3, 3])
    dtype = rng.choice(["f32", "f32", "f64"])
    tol = rng.choice([1e-3, 1e-4, 1e-5, 1e-6] if dtype == "f32" else [1e-6, 1e-9, 1e-12])
    lo, hi = {1: (200, 500_000), 2: (48, 1024), 3: (16, 224)}[dim]
    n = [_log_int(rng, lo, hi) for _ in range(dim)]
    if rng.random() < 0.4:  # an equal-sided image or volume
        n = n[:1] * dim
    ntransf = rng.choice([1, 1, 1, 1, rng.randint(2, 8), rng.randint(2, 32) if dim < 3 else 2])
    # points: bounded so that no draw does more kernel taps than the largest
    # listed case (2e10 in FP32; FP64 taps cost several times as much)
    taps = (1.5e10 if dtype == "f32" else 3e9) / (_width(tol) ** dim * ntransf)
    m = _log_int(rng, 2000, max(4000, min(2e7, taps, 2e8 / ntransf)))
    type = rng.choice([1, 2])
    opts = {}
    if type == 2 and rng.random() < 0.4:
        opts["gpu_method"] = 2
    if rng.random() < 0.2:
        opts["gpu_kerevalmeth"] = 1
    if type == 1 and dim == 3 and rng.random() < 0.2:
        opts["tile_slots"] = True
    case = _plan_case("", type, dtype, tol, n, m, rng.choice(["uniform", "clusters", "mixed"]),
                      ntransf, rng.random() < 0.5, **opts)
    del case["name"]
    return case


# ------------------------------------------------------------------- inputs
def _real(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _complex(case):
    return torch.complex64 if case["dtype"] == "f32" else torch.complex128


def _modes(case):
    """(N1[, N2[, N3]]), x first."""
    return [case[k] for k in ("n1", "n2", "n3") if k == "n1" or case[k] > 1]


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(seed)


def _wrap(x):
    return torch.remainder(x + math.pi, 2 * math.pi) - math.pi


def _clip(x, dtype):
    """To the plan's precision, inside [-pi, pi) there too."""
    top = float(np.nextafter(np.float32(np.pi), np.float32(0))) if dtype == torch.float32 \
        else float(np.nextafter(np.pi, 0))
    return x.to(dtype).clamp_(-top, top)


def _points(dist, dim, m, gen, dtype):
    """One array per axis: uniform, 8 wrapped Gaussian clusters (sigma 0.3),
    or half uniform and half in 4 clusters (sigma 0.2)."""
    mu = {"uniform": m, "clusters": 0, "mixed": m // 2}[dist]
    k, sigma = (8, 0.3) if dist == "clusters" else (4, 0.2)
    cen = (torch.rand(dim, k, generator=gen, device=_DEV, dtype=torch.float64) - 0.5) * 2 * math.pi
    lab = torch.randint(0, k, (m - mu,), generator=gen, device=_DEV)
    out = []
    for d in range(dim):
        u = (torch.rand(mu, generator=gen, device=_DEV, dtype=torch.float64) - 0.5) * 2 * math.pi
        g = torch.randn(m - mu, generator=gen, device=_DEV, dtype=torch.float64) * sigma
        out.append(_clip(torch.cat([u, _wrap(cen[d][lab] + g)]), dtype))
    return out


def _normal(shape, gen, dtype):
    return torch.randn(*shape, generator=gen, device=_DEV, dtype=dtype)


def _radial(case, gen):
    """(2, spokes * samples) golden-angle radial trajectory with jitter."""
    s, n = case["spokes"], case["samples"]
    ang = torch.arange(s, device=_DEV, dtype=torch.float64) * (math.pi * 2 / (1 + math.sqrt(5)))
    rad = -math.pi + 2 * math.pi * torch.arange(n, device=_DEV, dtype=torch.float64) / n
    p = torch.stack([torch.outer(f(ang), rad).reshape(-1) for f in (torch.cos, torch.sin)])
    p = p + 1e-3 * torch.randn(2, s * n, generator=gen, device=_DEV, dtype=torch.float64)
    return _clip(_wrap(p), _real(case))


def _group_sizes(case):
    """(N1, N2, M) of every member: sizes belong to the case, not to the seed."""
    r = np.random.RandomState(7)
    out = []
    for _ in range(case["plans"]):
        n = [int(round(math.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
             for _ in range(2)]
        m = int(round(math.exp(r.uniform(math.log(case["m_lo"]), math.log(case["m_hi"])))))
        out.append((n[0], n[1], m))
    return out


def _inputs(case, seed):
    gen = _gen(seed)
    if case["kind"] == "grad":
        pts = _radial(case, gen)
        fk = _normal((case["n2"], case["n1"]), gen, _complex(case))
        return {"pts": pts, "fk": fk, "target": _normal((pts.shape[1],), gen, _complex(case))}
    if case["kind"] == "group":
        return [{"n": (n1, n2), "pts": _points("uniform", 2, m, gen, torch.float32),
                 "c": _normal((m,), gen, torch.complex64)} for n1, n2, m in _group_sizes(case)]
    n, t, m = _modes(case), case["ntransf"], case["m"]
    pts = _points(case["dist"], len(n), m, gen, _real(case))
    shape = (t, m) if case["type"] == 1 else (t, *n[::-1])
    return {"pts": pts, "in": _normal(shape, gen, _complex(case))}


_OPTIONS = ("gpu_method", "gpu_kerevalmeth", "tile_slots")


def prepare(case, seed):
    s = {"case": case}
    inp = _inputs(case, seed)
    if case["kind"] == "grad":
        s.update(inp)
    elif case["kind"] == "group":
        plans = []
        for member in inp:
            p = cufinufft(1, member["n"][::-1], eps=case["tol"], dtype=np.float32)
            p.set_pts(*member["pts"][::-1])
            plans.append(p)
        s["c"] = [member["c"] for member in inp]
        s["fk"] = [torch.empty(member["n"][::-1], dtype=torch.complex64, device=_DEV)
                   for member in inp]
        s["group"] = cufinufft_group(plans, s["c"], s["fk"])
    else:
        n, t, m = _modes(case), case["ntransf"], case["m"]
        opts = {k: case[k] for k in _OPTIONS if k in case}
        s["plan"] = cufinufft(case["type"], n[::-1], n_trans=t, eps=case["tol"],
                              dtype=np.float32 if case["dtype"] == "f32" else np.float64,
                              maxbatchsize=0, **opts)
        s["pts"], s["in"] = inp["pts"], inp["in"]
        shape = (t, *n[::-1]) if case["type"] == 1 else (t, m)
        s["out"] = torch.empty(shape, dtype=_complex(case), device=_DEV)
        if not case["setpts"]:
            s["plan"].set_pts(*s["pts"][::-1])
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "grad":
        # the trajectory comes out of the model anew in every step
        pts = s["pts"].clone().requires_grad_()
        fk = s["fk"].detach().requires_grad_()
        c = nufft_type2(pts, fk, isign=-1, eps=case["tol"])
        (c - s["target"]).abs().pow(2).sum().backward()
        return {"c": c.detach(), "grad_fk": fk.grad, "grad_pts": pts.grad}
    if case["kind"] == "group":
        s["group"].execute(use_graph=case["graph"])
        return s["fk"]
    plan = s["plan"]
    if case["setpts"]:
        plan.set_pts(*s["pts"][::-1])
    c, fk = (s["in"], s["out"]) if case["type"] == 1 else (s["out"], s["in"])
    plan.execute(c, fk)
    return s["out"]


# --------------------------------------------------------------------- work
def _transform_work(n, m, ntransf, tol, esize, setpts):
    """Bytes: coordinates (where the pass sorts), strengths and modes once
    each.  Operations: a complex multiply-add with a real weight per kernel
    tap, and the FFT of the twofold-oversampled grid's mode lines."""
    dim, ntot = len(n), math.prod(n)
    nbytes = ntransf * (m + ntot) * 2 * esize + (m * dim * esize if setpts else 0)
    flops = 4.0 * m * ntransf * _width(tol) ** dim
    lines = math.prod(2 * k for k in n)
    for k in n:  # x over every line, then only the lines that hold modes
        flops += ntransf * 5.0 * lines * math.log2(2 * k)
        lines //= 2
    return nbytes, flops


def work(case):
    e = 4 if case["dtype"] == "f32" else 8
    if case["kind"] == "grad":
        m, n = case["spokes"] * case["samples"], _modes(case)
        # forward, adjoint to the modes, one derivative per axis; points and
        # modes in, target in, values, both gradients out
        _, f = _transform_work(n, m, 2 + len(n), case["tol"], e, True)
        return {"bytes": (2 * 2 * m + 2 * 2 * m + 2 * 2 * math.prod(n)) * e, "flops": f}
    if case["kind"] == "group":
        w = [_transform_work((a, b), m, 1, case["tol"], e, False) for a, b, m in _group_sizes(case)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    b, f = _transform_work(_modes(case), case["m"], case["ntransf"], case["tol"], e,
                           case["setpts"])
    return {"bytes": b, "flops": f}


# -------------------------------------------------------------------- exact
# FP64 direct sums as matrix products: e^{i k.x} factors over the axes, and a
# long 1D axis is split as k = K * k_hi + k_lo.
_BUDGET = 3.5e13  # complex multiply-adds


def _freqs(n):
    return torch.arange(-(n // 2), (n + 1) // 2, device=_DEV, dtype=torch.float64)


def _phase(x, k, sign):
    a = torch.outer(x, k) * sign
    return torch.complex(torch.cos(a), torch.sin(a))


def _factors(pts, n, sign):
    """(E_fast, E_slow): e^{i sign k.x_j} = E_slow[j, s] * E_fast[j, f] with
    the modes in (s, f) order; the product may be longer than the modes (1D)."""
    x = [p.double() for p in pts]
    if len(n) == 1:
        big = max(1, int(math.sqrt(n[0])))
        hi = torch.arange(-(-n[0] // big), device=_DEV, dtype=torch.float64) * big - n[0] // 2
        lo = torch.arange(big, device=_DEV, dtype=torch.float64)
        return _phase(x[0], lo, sign), _phase(x[0], hi, sign)
    fast, slow = _phase(x[0], _freqs(n[0]), sign), _phase(x[1], _freqs(n[1]), sign)
    if len(n) == 3:
        z = _phase(x[2], _freqs(n[2]), sign)
        slow = (z.unsqueeze(2) * slow.unsqueeze(1)).reshape(len(x[0]), -1)
    return fast, slow


def _chunks(n, m):
    if len(n) == 1:
        wide = 2 * math.isqrt(n[0]) + 2
    else:
        wide = n[0] + math.prod(n[1:])
    step = max(64, min(m, int(6e7 / wide)))
    return [slice(i, min(m, i + step)) for i in range(0, m, step)]


def _sum1(pts, c, n, sign):
    """Type 1: modes (ntransf, N3, N2, N1) of strengths c (ntransf, M)."""
    c, total = c.to(torch.complex128), None
    for sl in _chunks(n, c.shape[1]):
        fast, slow = _factors([p[sl] for p in pts], n, sign)
        part = torch.stack([slow.t() @ (fast * ct[sl].unsqueeze(1)) for ct in c])
        total = part if total is None else total + part
    return total.reshape(c.shape[0], -1)[:, :math.prod(n)].reshape(c.shape[0], *n[::-1])


def _sum2(pts, fk, n, sign):
    """Type 2: values (ntransf, M) of modes fk (ntransf, ...)."""
    f = fk.reshape(fk.shape[0], -1).to(torch.complex128)
    m, out = pts[0].numel(), []
    for sl in _chunks(n, m):
        fast, slow = _factors([p[sl] for p in pts], n, sign)
        cells = fast.shape[1] * slow.shape[1]
        g = torch.nn.functional.pad(f, (0, cells - f.shape[1]))
        g = g.reshape(-1, slow.shape[1], fast.shape[1])
        out.append(torch.stack([((slow @ gt) * fast).sum(1) for gt in g]))
    return torch.cat(out, 1)


def _affordable(n, m, ntransf):
    return float(m) * math.prod(n) * ntransf <= _BUDGET


def exact(case, seed):
    if case["kind"] == "group":
        if sum(float(a) * b * m for a, b, m in _group_sizes(case)) > _BUDGET:
            return None
        return [_sum1(g["pts"], g["c"][None], g["n"], 1.0)[0] for g in _inputs(case, seed)]
    if case["kind"] == "grad":
        n, m = _modes(case), case["spokes"] * case["samples"]
        if not _affordable(n, m, 2 + len(n)):
            return None
        s = _inputs(case, seed)
        pts, fk = list(s["pts"]), s["fk"][None].to(torch.complex128)
        c = _sum2(pts, fk, n, -1.0)[0]
        g = 2 * (c - s["target"].to(torch.complex128))
        kx, ky = _freqs(n[0])[None, None, :], _freqs(n[1])[None, :, None]
        dx = [_sum2(pts, fk * (-1j * k), n, -1.0)[0] for k in (kx, ky)]
        return {"c": c, "grad_fk": _sum1(pts, g[None], n, 1.0)[0],
                "grad_pts": torch.stack([(g.conj() * d).real for d in dx])}
    n = _modes(case)
    if not _affordable(n, case["m"], case["ntransf"]):
        return None
    s = _inputs(case, seed)
    if case["type"] == 1:
        return _sum1(s["pts"], s["in"], n, 1.0)
    return _sum2(s["pts"], s["in"], n, -1.0)
