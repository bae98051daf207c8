"""Timed calls: the work that a user of this package has it do.

Each case is one pass through the public entry points of ``apollofft_amd`` as
a user's program makes it: a plan is built once, the inputs lie on the GPU
(host arrays for the numpy functions), and a pass is one transform, one
forward and backward step, or one batched call.  Coordinates are in radians on
[-pi, pi) per axis (float32), strengths and modes complex64 with re, im ~
N(0, 1).

A case is a dict:
  kind    "type1" / "type2" (3D), "type1_1d" / "type2_1d", "grad_type2" /
          "grad_type1" (3D forward + backward through autograd), "batched"
          (many 3D Type-1 problems), "numpy_type1" (the numpy function)
  n, nx, ny, nz   modes per axis        M       points
  w       kernel half-width             points  "uniform", "clustered", "radial"
  grid    "reference" (power-of-two 3D grids, sigma n in 1D) or "exact" (sigma n)
A batched case has ``problems``, ``min_points``, ``max_points`` and ``mix``;
the sizes of its problems follow from ``mix`` alone, so the amount of work
does not depend on the seed of the inputs.
"""
import math
import random

import numpy as np
import torch

import apollofft_amd as A
from apollofft_amd.autograd import nufft_type1, nufft_type2

TWO_PI = 2.0 * math.pi
BATCH_MODES = (32, 48, 64, 96)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # One short 1D record at the default width: a call whose time is its
        # launches (4096 samples, 256 modes).
        dict(name="t1_1d_256", kind="type1_1d", n=256, M=4096, w=6, points="uniform",
             grid="reference"),
        # Long 1D evaluation on a prime number of modes (a Bluestein axis).
        dict(name="t2_1d_1009", kind="type2_1d", n=1009, M=1_000_000, w=6, points="uniform",
             grid="reference"),
        # A small 3D call: 16^3 modes, 2000 points, again launch-bound.
        dict(name="t1_16", kind="type1", nx=16, ny=16, nz=16, M=2000, w=6, points="uniform",
             grid="reference"),
        # Ragged axes and an odd number of points at low accuracy (w = 4),
        # mixed-radix and Bluestein axes in one grid.
        dict(name="t2_ragged", kind="type2", nx=37, ny=50, nz=29, M=200_003, w=4,
             points="uniform", grid="exact"),
        # The ordinary pair at 64^3 modes, one part in 10^6: gridding of
        # samples and its opposite.
        dict(name="t1_64", kind="type1", nx=64, ny=64, nz=64, M=2_000_000, w=7,
             points="uniform", grid="reference"),
        dict(name="t2_64", kind="type2", nx=64, ny=64, nz=64, M=2_000_000, w=7,
             points="uniform", grid="reference"),
        # Large clustered sets: low accuracy on a grid with prime axes, and
        # the widest kernel on a mixed-radix grid.
        dict(name="t1_127_clustered", kind="type1", nx=127, ny=127, nz=127, M=16_000_000, w=4,
             points="clustered", grid="exact"),
        dict(name="t2_100_clustered", kind="type2", nx=100, ny=100, nz=100, M=16_000_000, w=8,
             points="clustered", grid="exact"),
        # Fitting modes and coordinates: forward and backward of
        # ||T2(f, x) - b||^2, and of ||T1(c, x) - y||^2 on radial points.
        dict(name="grad_t2_64", kind="grad_type2", nx=64, ny=64, nz=64, M=1_000_000, w=6,
             points="uniform", grid="reference"),
        dict(name="grad_t1_48", kind="grad_type1", nx=48, ny=48, nz=48, M=400_000, w=6,
             points="radial", grid="exact"),
        # Many problems of uneven size in one call.
        dict(name="batched_64", kind="batched", problems=64, min_points=100_000,
             max_points=4_000_000, w=6, mix=8, points="radial", grid="exact"),
        # The numpy function with the reference binding's arguments: host
        # arrays in and out.
        dict(name="numpy_t1_32", kind="numpy_type1", nx=32, ny=32, nz=32, M=100_000, w=6,
             points="uniform", grid="reference"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above (``rng``: random.Random)."""
    kind = rng.choice(("type1", "type2", "type1", "type2", "type1_1d", "type2_1d",
                       "grad_type2", "grad_type1", "batched", "numpy_type1"))
    w = rng.choice((4, 5, 6, 6, 7, 8))
    points = rng.choice(("uniform", "clustered", "radial"))
    grid = rng.choice(("reference", "exact"))
    if kind.endswith("_1d"):
        return dict(kind=kind, n=_log_int(rng, 64, 1024), M=_log_int(rng, 1000, 1_000_000), w=w,
                    points=rng.choice(("uniform", "clustered")), grid=grid)
    if kind == "batched":
        lo = _log_int(rng, 2000, 100_000)
        return dict(kind=kind, problems=_log_int(rng, 2, 64), min_points=lo,
                    max_points=_log_int(rng, 2 * lo, 2_000_000), w=rng.choice((4, 6, 7)),
                    mix=rng.randrange(1, 10 ** 6), points=points, grid="exact")
    top = {"type1": 16_000_000, "type2": 16_000_000, "grad_type2": 4_000_000,
           "grad_type1": 4_000_000, "numpy_type1": 400_000}[kind]
    base = _log_int(rng, 12, 96)
    nx, ny, nz = (min(127, max(8, round(base * rng.uniform(0.75, 1.33)))) for _ in range(3))
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, M=_log_int(rng, 1500, top), w=w, points=points,
                grid="reference" if kind == "numpy_type1" else grid)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _wrap(x):
    """[-pi, pi) in FP32 (the wrap itself in FP64)."""
    x = torch.remainder(x.double() + math.pi, TWO_PI) - math.pi
    return x.float().clamp_(-3.1415925, 3.1415925)


def _points(g, M, dim, how):
    """(M, dim) float32 coordinates: uniform; 70 % in 8 Gaussian clusters of
    sigma 0.1 and 30 % uniform, shuffled; or lines of 512 points through the
    origin (density ~ 1/r^2)."""
    if how == "uniform":
        return (torch.rand((M, dim), generator=g, device="cuda") - 0.5) * 6.2831850
    if how == "clustered":
        mc = int(0.7 * M)
        centres = (torch.rand((8, dim), generator=g, device="cuda") - 0.5) * TWO_PI
        which = torch.randint(0, 8, (mc,), generator=g, device="cuda")
        pts = torch.empty((M, dim), dtype=torch.float32, device="cuda")
        pts[:mc] = _wrap(centres[which] + 0.1 * torch.randn((mc, dim), generator=g, device="cuda"))
        pts[mc:] = (torch.rand((M - mc, dim), generator=g, device="cuda") - 0.5) * 6.2831850
        return pts[torch.randperm(M, generator=g, device="cuda")].contiguous()
    lines = -(-M // 512)
    dirs = torch.randn((lines, 3), generator=g, device="cuda")
    dirs /= dirs.norm(dim=1, keepdim=True)
    r = (torch.rand((lines, 512), generator=g, device="cuda") - 0.5) * 6.2831850
    return (r[:, :, None] * dirs[:, None, :]).reshape(-1, 3)[:M].contiguous()


def _normal(g, shape):
    re_im = torch.randn(tuple(shape) + (2,), generator=g, device="cuda")
    return torch.view_as_complex(re_im)


def _shape(case):
    return (case["n"],) if "n" in case else (case["nx"], case["ny"], case["nz"])


def _plan3d(n, w, grid):
    return A.NufftPlan3D(*n, *(TWO_PI / v for v in n), 2, w, grid_policy=grid)


def _batch_sizes(case):
    r = random.Random(case["mix"])
    return [(r.choice(BATCH_MODES), r.randint(case["min_points"], case["max_points"]))
            for _ in range(case["problems"])]


def _inputs(case, seed):
    """Points and data of a case, from the seed alone."""
    g = _gen(seed)
    kind, how = case["kind"], case["points"]
    if kind == "batched":
        pos, vals = [], []
        for _, M in _batch_sizes(case):
            pos.append(_points(g, M, 3, how))
            vals.append(_normal(g, (M,)))
        return {"pos": pos, "vals": vals}
    n, M = _shape(case), case["M"]
    x = _points(g, M, len(n), how)
    if len(n) == 1:
        x = x.reshape(-1)
    s = {"x": x}
    if kind in ("type1", "type1_1d", "numpy_type1", "grad_type1"):
        s["c"] = _normal(g, (M,))
    if kind in ("type2", "type2_1d", "grad_type2"):
        s["f"] = _normal(g, n)
    if kind == "grad_type2":
        s["b"] = _normal(g, (M,))
    if kind == "grad_type1":
        # the data a fit starts from: modes of the size of the transform itself
        s["y"] = _normal(g, n) * math.sqrt(M)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"] = kind = case["kind"]
    w, grid = case["w"], case["grid"]
    if kind == "batched":
        plans = {}
        for m, _ in _batch_sizes(case):
            if m not in plans:
                plans[m] = _plan3d((m, m, m), w, grid)
        s["plans"] = [plans[m] for m, _ in _batch_sizes(case)]
    elif kind == "numpy_type1":
        # the drop-in function takes float64 positions and complex128 values
        s["x"] = s["x"].cpu().numpy().astype(np.float64)
        s["c"] = s["c"].cpu().numpy().astype(np.complex128)
        s["n"], s["w"] = _shape(case), w
    elif kind.endswith("_1d"):
        s["plan"] = A.NufftPlan1D(case["n"], TWO_PI / case["n"], 2, w, grid_policy=grid)
    else:
        s["plan"] = _plan3d(_shape(case), w, grid)
    if kind.startswith("grad_"):
        s["x"].requires_grad_(True)
        s["c" if kind == "grad_type1" else "f"].requires_grad_(True)
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind in ("type1", "type1_1d"):
        return state["plan"].type1(state["x"], state["c"])
    if kind in ("type2", "type2_1d"):
        return state["plan"].type2(state["x"], state["f"])
    if kind == "batched":
        return A.execute_type1_batched(state["plans"], state["pos"], state["vals"])
    if kind == "numpy_type1":
        n = state["n"]
        return A.nufft_type1_3d_fast(state["x"], state["c"], *n, *(TWO_PI / v for v in n),
                                     kernel_width=state["w"])
    if kind == "grad_type2":
        out = nufft_type2(state["f"], state["x"], state["plan"])
        loss = (out - state["b"]).abs().pow(2).sum()
        gf, gx = torch.autograd.grad(loss, (state["f"], state["x"]))
        return {"out": out.detach(), "grad_modes": gf, "grad_points": gx}
    out = nufft_type1(state["c"], state["x"], state["plan"])
    loss = (out - state["y"]).abs().pow(2).sum()
    gc, gx = torch.autograd.grad(loss, (state["c"], state["x"]))
    return {"out": out.detach(), "grad_values": gc, "grad_points": gx}


# ---------------------------------------------------------------- necessary work
def _over(n, grid, w, dim):
    m = max(2 * n, 2 * w + 1)
    if dim == 3 and grid == "reference":
        m = 1 << (m - 1).bit_length()
    return m


def _one_work(kind, n, M, w, grid):
    """Inputs read once, outputs written once; 4 (2w)^dim flops per point for
    spreading or interpolation (three times that for the coordinate gradient)
    and 5 G log2 G per FFT of the oversampled grid."""
    dim = len(n)
    N = math.prod(n)
    G = math.prod(_over(v, grid, w, dim) for v in n)
    point = 4.0 * dim * M          # coordinates
    taps = 4.0 * (2 * w) ** dim * M
    fft = 5.0 * G * math.log2(G)
    if kind.startswith("grad_"):
        # x, the data and the target in; the transform and both gradients out
        return (2 * point + 24.0 * M + 16.0 * N if kind == "grad_type2"
                else 2 * point + 16.0 * M + 16.0 * N), 5.0 * taps + (3.0 if kind == "grad_type2" else 2.0) * fft
    scale = 2.0 if kind == "numpy_type1" else 1.0
    return scale * (point + 8.0 * M + 8.0 * N), taps + fft


def work(case):
    w, grid = case["w"], case["grid"]
    if case["kind"] == "batched":
        parts = [_one_work("type1", (m, m, m), M, w, grid) for m, M in _batch_sizes(case)]
    else:
        parts = [_one_work(case["kind"], _shape(case), case["M"], w, grid)]
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


# ---------------------------------------------------------------- 64-bit values
def _freq(n):
    """Signed frequencies in FFT order, n/2 positive."""
    k = torch.arange(n, dtype=torch.float64, device="cuda")
    return torch.where(k <= n // 2, k, k - n)


def _phase(x, n, sign):
    """(P, n) exp(sign i k x), one axis."""
    a = x.double()[:, None] * _freq(n)[None, :]
    return torch.complex(torch.cos(a), sign * torch.sin(a))


def _chunk(n):
    return max(256, min(1 << 18, (1 << 26) // max(1, math.prod(n[1:]))))


def _direct_type1(x, c, n):
    """sum_j c_j exp(-i k.x_j) for all modes, FP64."""
    x = x.reshape(-1, len(n))
    c = c.to(torch.complex128)
    out = torch.zeros((n[0], math.prod(n[1:])), dtype=torch.complex128, device="cuda")
    step = _chunk(n)
    for a in range(0, x.shape[0], step):
        p = x[a:a + step]
        right = torch.ones((p.shape[0], 1), dtype=torch.complex128, device="cuda")
        for ax in range(1, len(n)):
            right = (right[:, :, None] * _phase(p[:, ax], n[ax], -1.0)[:, None, :]).reshape(
                p.shape[0], -1)
        left = (_phase(p[:, 0], n[0], -1.0) * c[a:a + step, None]).t().contiguous()
        out += left @ right
    return out.reshape(n)


def _direct_type2(x, f, n, grad=False):
    """sum_k f_k exp(+i k.x_j) at all points, FP64; with ``grad`` also the
    derivative along each axis, (M, dim)."""
    x = x.reshape(-1, len(n))
    f2 = f.to(torch.complex128).reshape(n[0], -1)
    kf = [(1j * _freq(n[0])[:, None]) * f2]
    if grad:
        for ax in (1, 2):
            k = _freq(n[ax])
            k = k[:, None] if ax == 1 else k[None, :]
            kf.append(1j * (k.expand(n[1], n[2]).reshape(1, -1)) * f2)
    vals, ders = [], []
    step = _chunk(n)
    for a in range(0, x.shape[0], step):
        p = x[a:a + step]
        left = _phase(p[:, 0], n[0], 1.0)
        right = torch.ones((p.shape[0], 1), dtype=torch.complex128, device="cuda")
        for ax in range(1, len(n)):
            right = (right[:, :, None] * _phase(p[:, ax], n[ax], 1.0)[:, None, :]).reshape(
                p.shape[0], -1)
        vals.append(((left @ f2) * right).sum(dim=1))
        if grad:
            ders.append(torch.stack([((left @ k) * right).sum(dim=1) for k in kf], dim=1))
    v = torch.cat(vals)
    return (v, torch.cat(ders)) if grad else v


def _direct_terms(case):
    """Complex multiply-adds of ``exact``."""
    if case["kind"] == "batched":
        return sum(float(m) ** 3 * M for m, M in _batch_sizes(case))
    return float(math.prod(_shape(case))) * case["M"] * (5 if case["kind"].startswith("grad_") else 1)


def exact(case, seed):
    if _direct_terms(case) > 4.0e13:
        return None
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "batched":
        return [_direct_type1(x, c, (m, m, m))
                for (m, _), x, c in zip(_batch_sizes(case), s["pos"], s["vals"])]
    n = _shape(case)
    if kind in ("type1", "type1_1d"):
        return _direct_type1(s["x"], s["c"], n)
    if kind == "numpy_type1":
        return _direct_type1(s["x"], s["c"], n).cpu().numpy()
    if kind in ("type2", "type2_1d"):
        return _direct_type2(s["x"], s["f"], n)
    if kind == "grad_type2":
        out, der = _direct_type2(s["x"], s["f"], n, grad=True)
        g = 2.0 * (out - s["b"].to(torch.complex128))
        return {"out": out, "grad_modes": _direct_type1(s["x"], g, n),
                "grad_points": (g.conj()[:, None] * der).real}
    out = _direct_type1(s["x"], s["c"], n)
    G = 2.0 * (out - s["y"].to(torch.complex128))
    gc, der = _direct_type2(s["x"], G, n, grad=True)
    return {"out": out, "grad_values": gc,
            "grad_points": (s["c"].to(torch.complex128).conj()[:, None] * der).real}
