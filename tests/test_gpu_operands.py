"""The FP16-split operands of matrix-core spreading: the 22 bits they keep.

The grid of one point is wx(i) wy(j) wz(k) c.  Spreading forms it as one
product A B of A = wx wy and B = c wz, each rounded to FP32 (2^-24) and split
once into FP16 halves (hi to nearest, lo toward zero: below 2^-22 of an operand
of 2^-2 or more after scaling), without lo lo (at most 2^-11 each: 2^-22), in
three FP32 additions (2^-23 each if truncated).  So a cell is off by at most
(2 / 4 + 2 + 1 + 3 / 2) 2^-22 = 5 * 2^-22, wherever wx wy is at least 2^-14 (times 2^12
in A) and c wz at least 2^-17 of the largest strength (below 2^15 in B).

The exact taps need not be known: a point at the same place of its cell on all
three axes has the same FP32 taps on each, so that cells (i, j, k) and (k, j, i)
are equal but for the rounding above, with the taps i and k once in A and once
in B; and re / im of every cell is that of c.  Two cells enter either check:
10 * 2^-22.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -22


@pytest.mark.parametrize("w", [2, 4, 5, 6, 7, 8])
def test_spread_cells_keep_22_bits(dev, w):
    import torch
    import apollofft_amd as A
    import apollofft_amd._native as N
    m, step = 128, 32
    p = A.NufftPlan3D(m // 2, m // 2, m // 2, 1.0, 1.0, 1.0, 2, w, kernel_method="mfma")
    assert p.meta["m"] == (m, m, m)
    rng = np.random.default_rng(w)
    # one point in the middle of every 32^3 block, so that no cell has two
    cells = np.stack(np.meshgrid(*[np.arange(0, m, step)] * 3, indexing="ij"), -1).reshape(-1, 3) + step // 2
    cells = cells + rng.integers(-4, 5, cells.shape)
    place = rng.integers(20, 1004, (len(cells), 1)) / 1024.0  # (exact in FP32)
    xyz = ((cells + place) / 2).astype(np.float32)
    # strengths of the call's largest and 2^-14 of it
    c = rng.uniform(0.7, 0.99, (len(cells), 2)) * [1, -1]
    c = (c * np.where(np.arange(len(cells)) % 2, 2.0 ** -14, 1.0)[:, None]).astype(np.float32)
    c[0] = 1.0
    tx = torch.from_numpy(xyz).to(dev)
    tc = torch.view_as_complex(torch.from_numpy(c).to(dev))
    grid = torch.empty((m, m, m), dtype=torch.complex64, device=dev)
    ws = torch.empty(p.workspace_size(len(xyz)), dtype=torch.uint8, device=dev)
    b = tx.data_ptr()
    N.check(N.lib().anufft_debug_spread(p.handle, len(xyz), N.ptr_array([b, b + 4, b + 8]), 3, tc.data_ptr(),
                                        grid.data_ptr(), ws.data_ptr(), ws.numel(), None))
    g = grid.cpu().numpy()
    worst = [0.0, 0.0]
    for cell, v in zip(cells, c.astype(np.float64)):
        s = tuple(slice(a - w + 1, a + w + 1) for a in cell)
        re, im = g[s].real.astype(np.float64), g[s].imag.astype(np.float64)
        top = int(np.argmax(re[w, w]))  # largest tap (more than 1/2), that of every axis
        plane, line = re[:, top, :], re[top, top]
        if v[0] > 0.5:  # taps down to 2^-12 of the largest, in A and in B
            ok = line >= line[top] * 2.0 ** -12
            assert ok.sum() >= w
            p = plane[ok][:, ok]
            worst[0] = max(worst[0], np.max(np.abs(p / p.T - 1.0)))
        ok = line >= 0.75 * line[top]
        worst[1] = max(worst[1], np.max(np.abs(im[top, top][ok] / line[ok] / (v[1] / v[0]) - 1.0)))
    print(f"w={w}: axes {worst[0] / U:.2f}, re / im {worst[1] / U:.2f} units of 2^-22", flush=True)
    assert max(worst) <= 10 * U
