"""The gather transposes of the Joseph and Siddon projections, and the views
they leave to the per-voxel search, against the FP64 oracle's transposes:
remainders of the lane tiles and z runs, truncated detectors, voxels of many
pixels and pixels of many voxels, waves of both main axes, and pixels of
extreme values.  On zero-mean input the FP32 sums cancel, so the relative error
is that of a summand: 2e-5 for Joseph; for Siddon three roundings of a plane
crossing at up to the source-detector distance, over the voxel it cuts."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2))
GEOMS = {
    "one_voxel": dict(volume=(1, 1, 1), **OFF),
    "remainders": dict(volume=(17, 33, 9), **OFF),
    "remainders_tilted": dict(volume=(33, 17, 11), tilt_rad=(0.02, 0.01, -0.03), **OFF),
    "long_runs": dict(volume=(160, 150, 83), voxel_mm=(0.3, 0.3, 0.3), total_views=5, views_per_turn=5, **OFF),
    "truncated": dict(channels=13, rows=7, tilt_rad=(0.02, 0.01, -0.03), **OFF),
    "many_pixels": dict(volume=(5, 4, 3), voxel_mm=(4.0, 4.5, 5.0), channels=70, rows=61, channel_mm=0.7, row_mm=0.6, **OFF),
    "few_pixels": dict(channels=11, rows=9, channel_mm=6.0, row_mm=5.0, tilt_rad=(0.02, 0.01, -0.03), **OFF),
    "wide_fan": dict(sid_mm=40.0, sdd_mm=60.0, channels=100, channel_mm=0.9, **OFF),
    "detector_inside": dict(sdd_mm=123.0, **OFF),
    "source_near": dict(sid_mm=16.0, sdd_mm=60.0, channels=100, **OFF),
    "one_pixel": dict(channels=1, rows=1, channel_mm=3.0, row_mm=3.0, **OFF),
}


def tolerance(kind, g):
    return 2e-5 if kind == "joseph" else max(2e-5, 3.0 * 2.0**-24 * g.sdd_mm / min(g.voxel_mm))


@pytest.mark.parametrize("name", list(GEOMS))
@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_matches_oracle_transpose(ctx, oracle, kind, name):
    g = small_geometry(**GEOMS[name])
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    y = np.random.default_rng(13).standard_normal((g.total_views, g.nv, g.nu)).astype(np.float32)
    got = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    fn = oracle.bp_joseph_adjoint if kind == "joseph" else oracle.bp_siddon_adjoint
    ref = fn(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), y.astype(np.float64))
    assert rel_rmse(got, ref) < tolerance(kind, g), rel_rmse(got, ref)
    # a view range, accumulated onto a volume, of the same rays
    part = P.adjoint(torch.from_numpy(y[2:5]).cuda(), kind=kind, first=2, out=torch.ones(P.volume_shape, device="cuda"),
                     accumulate=True).cpu().numpy()
    y[:2], y[5:] = 0.0, 0.0
    ref = fn(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), y.astype(np.float64))
    assert rel_rmse(part, ref + 1.0) < tolerance(kind, g)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_extreme_pixel_reaches_only_its_voxels(ctx, oracle, kind, value):
    """One pixel that is not finite changes the voxels its ray meets and no other."""
    g = small_geometry(tilt_rad=(0.02, 0.01, -0.03), **OFF)
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    y = np.random.default_rng(3).random((g.total_views, g.nv, g.nu)).astype(np.float32)
    plain = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    fn = oracle.bp_joseph_adjoint if kind == "joseph" else oracle.bp_siddon_adjoint
    one = np.zeros(y.shape)
    one[7, 17, 21] = 1.0
    met = fn(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), one)
    y[7, 17, 21] = value
    got = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    assert (met > 1e-3).any() and not np.isfinite(got[met > 1e-3]).any()
    clear = met == 0.0
    # (a ray within rounding of a support's edge may or may not meet it)
    assert np.isfinite(got[clear]).mean() > 0.9999
    same = np.abs(got[clear] - plain[clear]) <= 1e-5 * plain.max()
    assert same.mean() > 0.9999
