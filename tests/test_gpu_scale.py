"""Matrix-core point kernels over the FP32 exponent range: strengths and modes
scaled by a power of two give the same transforms, scaled.

The scale is exact and drops out of the FP16 splits, so two runs differ only by
the order of their FP32 sums (the atomic adds): at most some 60 terms a cell
here, 60 * 2^-24 = 3.6e-6 if every rounding fell the same way; and by what
falls below the FP32 subnormals, 2^-149 against the largest values of 2^-120
and more: below 2^-29 each.  4e-6.
"""
import numpy as np
import pytest

from helpers import cnormal

pytestmark = pytest.mark.gpu

TOL = 4e-6


def _rel(a, scale, b):
    a, b = a.cpu().numpy().astype(np.complex128) / scale, b.cpu().numpy().astype(np.complex128)
    assert np.isfinite(a).all()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("w", [2, 4, 6, 7, 8])
@pytest.mark.parametrize("M", [1000, 20000])
@pytest.mark.parametrize("power", [-122, -117, 100])
def test_powers_of_two_scale_the_transforms(dev, w, M, power):
    import torch
    import apollofft_amd as A
    n = (16, 21, 17)
    rng = np.random.default_rng(w)
    x = torch.from_numpy(rng.uniform(0, 1, (M, 3)).astype(np.float32)).to(dev)
    c = torch.from_numpy(cnormal(rng, M)).to(dev)
    f = torch.from_numpy(cnormal(rng, n)).to(dev)
    plan = A.NufftPlan3D(*n, *[1.0 / k for k in n], 2, w, kernel_method="mfma")
    s = 2.0 ** power
    cs, fs = torch.view_as_complex(torch.view_as_real(c) * s), torch.view_as_complex(torch.view_as_real(f) * s)
    assert _rel(plan.type1(x, cs), s, plan.type1(x, c)) <= TOL
    assert _rel(plan.type2(x, fs), s, plan.type2(x, f)) <= TOL
    if power < 0:  # (the gradient's factors 2 pi m / L, of some 100, stay in range)
        assert _rel(plan.grad_points(x, c, fs), s, plan.grad_points(x, c, f)) <= TOL
