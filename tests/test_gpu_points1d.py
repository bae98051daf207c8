"""1D transforms at the edges of the launch rules: fewer cells than taps, one
point, a workgroup's points more or less, the point count at which workgroups
widen, and lines of 2048 to 4096 points (mixed radix, Bluestein, the most
cells the LDS grid holds).  Against the oracle's FP64 restatement of the same
approximation, so only FP32 rounding is left: at most 4e-7 a tap, times about
5 by the deconvolution, and 5e-7 of the FFT; the suite's 1e-5 holds."""
import numpy as np
import pytest

from helpers import cnormal, rel_l2

pytestmark = pytest.mark.gpu

CASES = [(4, 1, 6), (33, 255, 2), (33, 257, 5), (128, 65536, 7), (128, 65537, 3), (1024, 2000, 6),
         (1009, 300, 6), (1500, 5000, 4), (2048, 70000, 8)]


@pytest.mark.parametrize("n,M,w", CASES)
def test_1d_launch_edges(dev, oracle_mod, n, M, w):
    import torch
    import apollofft_amd as A
    rng = np.random.default_rng(n + M + w)
    dx = 0.125
    x = rng.uniform(-n * dx, 2 * n * dx, M).astype(np.float32)
    x[:1] = 0.0  # on a cell boundary: both end taps vanish or not as the oracle's
    c, f = cnormal(rng, M), cnormal(rng, n)
    plan = A.NufftPlan1D(n, dx, 2, w)
    tx = torch.from_numpy(x).to(dev)
    t1 = plan.type1(tx, torch.from_numpy(c).to(dev)).cpu().numpy()
    t2 = plan.type2(tx, torch.from_numpy(f).to(dev)).cpu().numpy()
    x64 = x.astype(np.float64)
    r1 = oracle_mod.nufft1d_type1_fast(x64, c.astype(np.complex128), n, dx, 2, w)
    r2 = oracle_mod.nufft1d_type2_fast(f.astype(np.complex128), x64, dx, 2, w)
    assert rel_l2(t1, r1) < 1e-5
    assert rel_l2(t2, r2) < 1e-5
