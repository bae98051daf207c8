"""Matrix-core window kernels against the vector-ALU kernels at the sizes
where rounds, groups, classes, chunks and subproblems end.

Both kernel families form the same FP32 sums and share the FFT.  A point's
weight is a product of three tap values; each is a polynomial in FP32 (a few
2^-24 of the largest tap) and on the matrix cores an FP16 hi + lo pair (2^-22),
with one more such rounding for the product of two factors: at most about
4 * 2^-22 + 8 * 2^-24 = 1.4e-6 of the largest weight each, and the FP32 sums add
less than that in the L2 norm.  The two families may differ by the sum of their
errors: 4e-6.  The gradient's derivative taps are rounded the same way and its
sums cancel to about a third of their terms: 1.2e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL, TOL_GRAD = 4e-6, 1.2e-5


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda:0")


def _points(case, n, w, rng):
    """Coordinates in grid cells of the 2 n oversampled axes, mapped to the unit box."""
    m = [2 * k for k in n]
    kind, count = case
    if kind == "random":
        t = rng.uniform(0, 1, (count, 3)) * m
    elif kind == "one_cell":  # one class of one tile; subproblems and rounds that end unevenly
        t = np.array(m) // 2 + rng.uniform(0, 1, (count, 3))
    elif kind == "columns":  # both ends of every y cell: every class boundary, few points each
        y = np.repeat(np.arange(m[1]), 2) + np.tile([0.0, 0.999], m[1])
        t = np.stack([np.full_like(y, 3.25), y, np.linspace(0, m[2] - 1e-3, len(y))], 1)
    else:  # "corner": supports that wrap on every axis
        t = (rng.uniform(-2, 2, (count, 3)) + np.array(m)) % m
    return (t / np.array(m)).astype(np.float32)


# (random 3000 and 60000: few and many points a cell, wide and narrow windows;
# up to 4096 points one workgroup bins them all)
CASES = [("random", 1), ("random", 65), ("random", 3000), ("random", 4096), ("random", 60000), ("one_cell", 31), ("one_cell", 64),
         ("one_cell", 4097), ("columns", 0), ("corner", 129)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}{c[1]}")
@pytest.mark.parametrize("w", [2, 3, 4, 5, 6, 7, 8])
def test_window_kernels_match_vector_kernels(dev, w, case):
    import torch
    import apollofft_amd as A
    n = (16, 21, 17)
    rng = np.random.default_rng(1000 * w + case[1])
    xyz = _points(case, n, w, rng)
    M = len(xyz)
    x = torch.from_numpy(xyz).to(dev)
    c = torch.from_numpy((rng.standard_normal((M, 2)) @ [1, 1j]).astype(np.complex64)).to(dev)
    f = torch.from_numpy((rng.standard_normal(n + (2,)) @ [1, 1j]).astype(np.complex64)).to(dev)
    out = {}
    for method in ("mfma", "valu"):
        p = A.NufftPlan3D(*n, *[1.0 / k for k in n], 2, w, kernel_method=method)
        out[method] = (p.type1(x, c), p.type2(x, f), p.grad_points(x, c, f))
    for a, b, tol in zip(out["mfma"], out["valu"], (TOL, TOL, TOL_GRAD)):
        a, b = a.to("cpu", torch.complex128), b.to("cpu", torch.complex128)
        err = float(torch.linalg.norm(a - b) / torch.linalg.norm(b))
        assert err <= tol, (case, w, err)


def test_many_tiles(dev):
    """More tiles than the stable one-pass binning takes (9216), up to the
    tile binning's 16384: the same sums as the vector-ALU kernels."""
    import torch
    import apollofft_amd as A
    n, w, M = (120, 116, 120), 8, 20_000
    rng = np.random.default_rng(9)
    x = torch.from_numpy(rng.uniform(0, 1, (M, 3)).astype(np.float32)).to(dev)
    c = torch.from_numpy((rng.standard_normal((M, 2)) @ [1, 1j]).astype(np.complex64)).to(dev)
    f = torch.from_numpy((rng.standard_normal(n + (2,)) @ [1, 1j]).astype(np.complex64)).to(dev)
    out = {}
    for method in ("mfma", "valu"):
        p = A.NufftPlan3D(*n, *[1.0 / k for k in n], 2, w, kernel_method=method, grid_policy="exact")
        if method == "mfma":
            assert 9216 < np.prod([-(-a // b) for a, b in zip(p.meta["m"], p.meta["bin_size"])]) <= 16384
        out[method] = (p.type1(x, c), p.type2(x, f))
    for a, b in zip(out["mfma"], out["valu"]):
        a, b = a.to("cpu", torch.complex128), b.to("cpu", torch.complex128)
        assert float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) <= TOL


@pytest.mark.parametrize("w", [5, 7, 8])
def test_odd_grid_lengths(dev, w):
    """Grids of odd length along z (2 w + 1 cells): rows whose pairs of cells
    are not aligned, and windows longer than the grid."""
    import torch
    import apollofft_amd as A
    n = (9, 21, 5)
    rng = np.random.default_rng(w)
    x = torch.from_numpy(rng.uniform(0, 1, (500, 3)).astype(np.float32)).to(dev)
    c = torch.from_numpy((rng.standard_normal((500, 2)) @ [1, 1j]).astype(np.complex64)).to(dev)
    f = torch.from_numpy((rng.standard_normal(n + (2,)) @ [1, 1j]).astype(np.complex64)).to(dev)
    out = {}
    for method in ("mfma", "valu"):
        p = A.NufftPlan3D(*n, *[1.0 / k for k in n], 2, w, kernel_method=method, grid_policy="exact")
        assert p.meta["m"][2] == 2 * w + 1
        out[method] = (p.type2(x, f), p.grad_points(x, c, f))
    for a, b, tol in zip(out["mfma"], out["valu"], (TOL, TOL_GRAD)):
        a, b = a.to("cpu", torch.complex128), b.to("cpu", torch.complex128)
        assert float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) <= tol
