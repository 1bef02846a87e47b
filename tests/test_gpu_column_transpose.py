"""The Joseph transpose of untilted views by detector columns against the FP64
oracle's transpose: every block of rows and z groups with remainders, more
columns than a wave's lanes, more than four rays within a voxel, detectors that
end inside the volume's projection, views of one main axis only, and pixels that
are not finite.  On zero-mean input the FP32 sums cancel, so the relative error
is that of a summand, 2e-5."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2), total_views=5, views_per_turn=5)
GEOMS = {
    "rows16": dict(volume=(521, 513, 2), voxel_mm=(0.08, 0.08, 0.5), **OFF),
    "rows8": dict(volume=(131, 129, 33), voxel_mm=(0.3, 0.31, 0.5), **OFF),
    "rows4_two_groups": dict(volume=(90, 89, 65), voxel_mm=(0.4, 0.4, 0.3), **OFF),
    "three_groups": dict(volume=(60, 58, 150), voxel_mm=(0.5, 0.5, 0.14), **OFF),
    "four_groups": dict(volume=(51, 50, 200), voxel_mm=(0.6, 0.6, 0.1), **OFF),
    "two_z_blocks": dict(volume=(46, 45, 257), voxel_mm=(0.6, 0.6, 0.1), **OFF),
    "many_columns": dict(volume=(130, 130, 31), voxel_mm=(0.5, 0.5, 1.0), channels=1500, channel_mm=0.1, **OFF),
    "many_rays": dict(volume=(100, 100, 51), voxel_mm=(0.4, 0.4, 0.6), rows=400, row_mm=0.2, **OFF),
    "truncated": dict(volume=(100, 100, 51), voxel_mm=(0.4, 0.4, 0.6), channels=13, rows=7, **OFF),
    "one_pixel": dict(volume=(100, 100, 51), voxel_mm=(0.4, 0.4, 0.6), channels=1, rows=1, **OFF),
}


def setup(ctx, name):
    g = small_geometry(**GEOMS[name])
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    return g, P, np.random.default_rng(17).standard_normal((g.total_views, g.nv, g.nu)).astype(np.float32)


def reference(oracle, g, P, y):
    return oracle.bp_joseph_adjoint(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), y.astype(np.float64))


@pytest.mark.parametrize("name", list(GEOMS))
def test_matches_oracle_transpose(ctx, oracle, name):
    g, P, y = setup(ctx, name)
    got = P.adjoint(torch.from_numpy(y).cuda(), kind="joseph").cpu().numpy()
    ref = reference(oracle, g, P, y)
    assert rel_rmse(got, ref) < 2e-5, rel_rmse(got, ref)


@pytest.mark.parametrize("first", [0, 1, 2])
def test_one_view_accumulated(ctx, oracle, first):
    """One view, of either main axis, onto a volume."""
    g, P, y = setup(ctx, "rows4_two_groups")
    base = torch.ones(P.volume_shape, device="cuda")
    got = P.adjoint(torch.from_numpy(y[first:first + 1]).cuda(), kind="joseph", first=first, out=base, accumulate=True)
    y[:first], y[first + 1:] = 0.0, 0.0
    assert rel_rmse(got.cpu().numpy(), reference(oracle, g, P, y) + 1.0) < 2e-5


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_extreme_pixel_reaches_only_its_voxels(ctx, oracle, value):
    g, P, y = setup(ctx, "rows4_two_groups")
    plain = P.adjoint(torch.from_numpy(y).cuda(), kind="joseph").cpu().numpy()
    one = np.zeros(y.shape, dtype=np.float32)
    one[3, 17, 21] = 1.0
    met = reference(oracle, g, P, one)
    y[3, 17, 21] = value
    got = P.adjoint(torch.from_numpy(y).cuda(), kind="joseph").cpu().numpy()
    assert (met > 1e-3).any() and not np.isfinite(got[met > 1e-3]).any()
    clear = met == 0.0
    # (a ray within rounding of a support's edge may or may not meet it)
    assert np.isfinite(got[clear]).mean() > 0.9999
    assert (np.abs(got[clear] - plain[clear]) <= 1e-5 * np.abs(plain).max()).mean() > 0.9999
