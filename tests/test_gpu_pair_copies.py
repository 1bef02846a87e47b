"""The paired volume copies of the tilted Joseph and the Siddon projection at
volume widths about a workgroup's 256 columns, after a call that left another
layout in the same arrays: every guard column is written.  Against the FP64 oracle:
on white noise a Joseph sample errs by its position, three FP32 roundings of the
source's distance in voxels; the Siddon rays are set up in FP64."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2), total_views=9, views_per_turn=9)


@pytest.mark.parametrize("nx,ny", [(1, 31), (255, 4), (256, 5), (257, 3), (513, 2), (4, 256), (3, 33)])
@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_widths(ctx, oracle, kind, nx, ny):
    grid = dict(volume=(nx, ny, 7), voxel_mm=(24.0 / nx, 20.0 / ny, 2.6))
    g = small_geometry(**grid, **OFF)
    tilted = small_geometry(**grid, **OFF, tilt_rad=(0.02, 0.01, -0.03))
    P = yk.Projector(ctx, np.concatenate([g.views(), tilted.views()]), g.nu, g.nv, g.grid())
    rng = np.random.default_rng(91)
    other = torch.full(P.volume_shape, 1e6, device="cuda")
    P.forward(other, kind="joseph", first=0, count=9)  # untilted: the copies of the column kernel
    x = rng.random(P.volume_shape, dtype=np.float32)
    got = P.forward(torch.from_numpy(x).cuda(), kind=kind, first=9, count=9).cpu().numpy()
    fn = oracle.fp_joseph if kind == "joseph" else oracle.fp_siddon
    ref = fn(oracle.views_from_float(P.views)[9:], g.nu, g.nv, oracle_volume(oracle, g), x)
    tol = max(1e-5, 3.0 * 2.0**-24 * g.sid_mm / min(g.voxel_mm)) if kind == "joseph" else 1e-5
    assert rel_rmse(got, ref) < tol, rel_rmse(got, ref)
