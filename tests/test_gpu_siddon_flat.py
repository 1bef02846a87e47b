"""The Siddon transpose of untilted views, whose rays share their x and y within
a detector column and their z within a row, against the FP64 oracle's transpose:
both lengths of z runs with remainders, dense and truncated detectors, and
pixels that are not finite.  On zero-mean input the relative error is that of a
summand: three roundings of a plane crossing at up to the source-detector
distance, over the voxel it cuts."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2), total_views=5, views_per_turn=5)
GEOMS = {
    "runs_of_two": dict(volume=(33, 17, 7), **OFF),
    "runs_of_eight": dict(volume=(250, 243, 33), voxel_mm=(0.11, 0.1, 0.5), **OFF),
    "many_pixels": dict(volume=(21, 22, 9), voxel_mm=(1.0, 1.0, 2.0), channels=300, channel_mm=0.2, rows=150, row_mm=0.4, **OFF),
    "truncated": dict(channels=13, rows=7, **OFF),
    "one_pixel": dict(channels=1, rows=1, channel_mm=3.0, row_mm=3.0, **OFF),
}


def setup(ctx, name):
    g = small_geometry(**GEOMS[name])
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    return g, P, np.random.default_rng(19).standard_normal((g.total_views, g.nv, g.nu)).astype(np.float32)


def reference(oracle, g, P, y):
    return oracle.bp_siddon_adjoint(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), y.astype(np.float64))


@pytest.mark.parametrize("name", list(GEOMS))
def test_matches_oracle_transpose(ctx, oracle, name):
    g, P, y = setup(ctx, name)
    tol = max(2e-5, 3.0 * 2.0**-24 * g.sdd_mm / min(g.voxel_mm))
    got = P.adjoint(torch.from_numpy(y).cuda(), kind="siddon").cpu().numpy()
    ref = reference(oracle, g, P, y)
    assert rel_rmse(got, ref) < tol, rel_rmse(got, ref)
    part = P.adjoint(torch.from_numpy(y[1:4]).cuda(), kind="siddon", first=1, out=torch.ones(P.volume_shape, device="cuda"),
                     accumulate=True).cpu().numpy()
    y[:1], y[4:] = 0.0, 0.0
    assert rel_rmse(part, reference(oracle, g, P, y) + 1.0) < tol


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_extreme_pixel_reaches_only_its_voxels(ctx, oracle, value):
    g, P, y = setup(ctx, "runs_of_two")
    plain = P.adjoint(torch.from_numpy(y).cuda(), kind="siddon").cpu().numpy()
    one = np.zeros(y.shape, dtype=np.float32)
    one[3, 17, 21] = 1.0
    met = reference(oracle, g, P, one)
    y[3, 17, 21] = value
    got = P.adjoint(torch.from_numpy(y).cuda(), kind="siddon").cpu().numpy()
    assert (met > 1e-3).any() and not np.isfinite(got[met > 1e-3]).any()
    clear = met == 0.0
    # (a ray within rounding of a voxel's edge may or may not meet it)
    assert np.isfinite(got[clear]).mean() > 0.999
    assert (np.abs(got[clear] - plain[clear]) <= 1e-5 * np.abs(plain).max()).mean() > 0.999


def test_rays_across_the_main_axis(ctx, oracle):
    """Tilted views with rays perpendicular to their main axis, which the general gather leaves to the search."""
    g = small_geometry(sid_mm=40.0, sdd_mm=60.0, channels=170, channel_mm=1.0, tilt_rad=(0.02, 0.01, -0.03), volume=(24, 22, 18),
                       start_angle_rad=0.78, offset_unv_mm=(0.3, 0.0, 0.2), total_views=3, views_per_turn=7)
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    y = np.random.default_rng(23).standard_normal((g.total_views, g.nv, g.nu)).astype(np.float32)
    got = P.adjoint(torch.from_numpy(y).cuda(), kind="siddon").cpu().numpy()
    tol = max(2e-5, 3.0 * 2.0**-24 * g.sdd_mm / min(g.voxel_mm))
    assert rel_rmse(got, reference(oracle, g, P, y)) < tol
