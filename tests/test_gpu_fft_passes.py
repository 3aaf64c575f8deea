"""Line transforms at the sizes where their passes change: one, two, three and
more passes, single stages and stage pairs of every radix, odd lengths, planes
that do not fit the fused inverse kernel."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(1, 4, 6), (5, 7, 12), (14, 16, 18), (54, 50, 28), (63, 49, 75), (98, 105, 81),
         (108, 120, 45), (216, 6, 9), (7, 125, 128), (343, 4, 8), (4, 512, 10), (1024, 4, 5),
         (10, 12, 1000), (9, 168, 196)]


@pytest.mark.parametrize("grid", GRIDS)
def test_line_transform_passes_match_float64(grid):
    """Against numpy's float64 transform: a float transform of N points in
    stages is off by a few ulp per stage (at most 10 stages of 1.2e-7 here,
    growing as their root), the bound of the transform tests, 2e-6 of the largest value."""
    import torch
    from sponge_amd import lib, systems
    s = systems.tip3p_box(216, 18.7, seed=11, cutoff=8.0)
    nb = lib.Nonbonded(s, grid=grid)
    assert nb.grid == grid
    rng = np.random.default_rng(sum(grid))
    x = rng.standard_normal(grid).astype(np.float32)
    xd = torch.as_tensor(x).cuda()
    fc = grid[2] // 2 + 1
    spec = torch.empty(grid[0] * grid[1] * fc * 2, dtype=torch.float32, device="cuda")
    lib.check(nb.L.snb_fft_r2c(nb.ctx, ctypes.c_void_p(xd.data_ptr()),
                               ctypes.c_void_p(spec.data_ptr())), "snb_fft_r2c")
    nb.sync()
    got = spec.view(grid[0], grid[1], fc, 2).cpu().numpy()
    got = got[..., 0] + 1j * got[..., 1]
    ref = np.fft.rfftn(x.astype(np.float64))
    assert np.max(np.abs(got - ref)) / np.max(np.abs(ref)) < 2e-6
    back = torch.empty(grid, dtype=torch.float32, device="cuda")
    lib.check(nb.L.snb_fft_c2r(nb.ctx, ctypes.c_void_p(spec.data_ptr()),
                               ctypes.c_void_p(back.data_ptr())), "snb_fft_c2r")
    nb.sync()
    rt = back.cpu().numpy() / (grid[0] * grid[1] * grid[2])
    assert np.max(np.abs(rt - x)) < 2e-5
    nb.close()
