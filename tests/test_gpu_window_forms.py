"""Wide spreading windows at every width, and the tile binning with its class
list (more than 4096 points) on ragged and prime grids, against the vector-ALU
kernels.

Both kernel families share the FFT and form the same FP32 sums: a weight is a
product of three polynomials' values (a few 2^-24 of the largest tap each) and,
on the matrix cores, of FP16 hi + lo pairs (2^-22 each), at most about 4 * 2^-22
+ 8 * 2^-24 = 1.4e-6 of the largest; the sums add less in the L2 norm.  The two
may differ by the sum of their errors: 4e-6.  The gradient's sums cancel to
about a third of their terms: 1.2e-5.

Wide windows serve at least 8192 points, below 0.25 (w >= 6: 0.5, w = 8: 1) a
cell, where at least 256 (w = 8: 4096) windows of a class are left: the grids
of 128 cells and more here at 20,000 points.
"""
import numpy as np
import pytest

from helpers import cnormal

pytestmark = pytest.mark.gpu

TOL, TOL_GRAD = 4e-6, 1.2e-5


def _compare(dev, n, w, M, policy, seed):
    import torch
    import apollofft_amd as A
    rng = np.random.default_rng(seed)
    x = torch.from_numpy(rng.uniform(0, 1, (M, 3)).astype(np.float32)).to(dev)
    c = torch.from_numpy(cnormal(rng, M)).to(dev)
    f = torch.from_numpy(cnormal(rng, n)).to(dev)
    out = {}
    for method in ("mfma", "valu"):
        p = A.NufftPlan3D(*n, *[1.0 / k for k in n], 2, w, kernel_method=method, grid_policy=policy)
        out[method] = (p.type1(x, c), p.type2(x, f), p.grad_points(x, c, f))
    for what, a, b, tol in zip(("type1", "type2", "grad"), out["mfma"], out["valu"], (TOL, TOL, TOL_GRAD)):
        a, b = a.to("cpu", torch.complex128), b.to("cpu", torch.complex128)
        err = float(torch.linalg.norm(a - b) / torch.linalg.norm(b))
        assert err <= tol, (what, n, w, err)


@pytest.mark.parametrize("n,policy", [((64, 64, 64), "reference"), ((64, 75, 61), "exact")])
@pytest.mark.parametrize("w", [2, 3, 4, 5, 6, 7, 8])
def test_wide_windows_match_vector_kernels(dev, w, n, policy):
    _compare(dev, n, w, 20_000, policy, w)


@pytest.mark.parametrize("M", [4097, 7001])
@pytest.mark.parametrize("n,w", [((15, 9, 10), 4), ((13, 7, 11), 8), ((20, 24, 18), 5), ((127, 6, 10), 6),
                                 ((9, 31, 23), 7), ((33, 5, 40), 3), ((11, 12, 50), 2)])
def test_tile_binning_on_ragged_grids(dev, n, w, M):
    _compare(dev, n, w, M, "exact", M + w)


@pytest.mark.parametrize("n,w,M", [((160, 150, 140), 8, 500), ((160, 150, 140), 8, 8000), ((200, 150, 140), 6, 5000)])
def test_digit_passes_with_class_list(dev, n, w, M):
    """More tiles than the tile binning counts in LDS (16384)."""
    import apollofft_amd as A
    p = A.NufftPlan3D(*n, *[1.0 / k for k in n], 2, w, kernel_method="mfma", grid_policy="exact")
    assert np.prod([-(-a // b) for a, b in zip(p.meta["m"], p.meta["bin_size"])]) > 16384
    _compare(dev, n, w, M, "exact", M + w)
