"""The slab form of the Siddon projection and the rays it hands to the walk,
against the FP64 oracle: remainders of the 64-ray segments and eight-view
groups, waves holding rays of both main axes, rays steepest along Z, a
detector or source inside the volume, and volumes with values only the walk
can carry.  rel-RMSE 1e-5 and 1e-4 of the peak, the projectors' FP32 gates."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import max_abs, oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

GEOMS = {
    "odd": dict(channels=131, rows=7, total_views=17, views_per_turn=17, start_angle_rad=0.1,
                offset_unv_mm=(0.3, 0.0, 0.2), channel_mm=0.4),
    "wide_fan": dict(sid_mm=40.0, sdd_mm=60.0, channels=100, channel_mm=0.9, start_angle_rad=0.3,
                     offset_unv_mm=(0.3, 0.0, 0.2)),
    "steep": dict(sid_mm=40.0, sdd_mm=60.0, rows=150, row_mm=1.1, volume=(16, 15, 33), voxel_mm=(1.0, 1.1, 0.4),
                  start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2)),
    "detector_inside": dict(sdd_mm=123.0, start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2)),
    "source_inside": dict(sid_mm=8.0, sdd_mm=40.0, start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2)),
    "one_slice": dict(volume=(24, 1, 1), rows=5, row_mm=0.3, channels=67, start_angle_rad=0.1,
                      offset_unv_mm=(0.3, 0.0, 0.07)),
    "tilted": dict(tilt_rad=(0.02, 0.01, -0.03), start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2)),
}


@pytest.mark.parametrize("name", list(GEOMS))
def test_forward_matches_oracle(ctx, oracle, name):
    g = small_geometry(**GEOMS[name])
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = np.random.default_rng(5).random((g.volume[2], g.volume[1], g.volume[0])).astype(np.float32)
    got = P.forward(torch.from_numpy(x).cuda(), kind="siddon").cpu().numpy()
    ref = oracle.fp_siddon(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), x)
    assert rel_rmse(got, ref) < 1e-5, rel_rmse(got, ref)
    assert max_abs(got, ref) < 1e-4 * np.abs(ref).max()
    # accumulate adds onto the output
    acc = P.forward(torch.from_numpy(x).cuda(), kind="siddon", out=torch.ones(g.total_views, g.nv, g.nu, device="cuda"),
                    accumulate=True).cpu().numpy()
    assert rel_rmse(acc - 1.0, ref) < 2e-5


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.finfo(np.float32).max])
def test_extreme_voxel_reaches_only_its_rays(ctx, oracle, value):
    """One voxel of an extreme value changes the rays that cross it and no other."""
    g = small_geometry(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2), tilt_rad=(0.02, 0.01, -0.03))
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = np.random.default_rng(6).random((g.volume[2], g.volume[1], g.volume[0])).astype(np.float32)
    one = np.zeros_like(x)
    one[9, 11, 13] = 1.0
    crossed = oracle.fp_siddon(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), one) > 1e-5
    plain = oracle.fp_siddon(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), x)
    x[9, 11, 13] = value
    got = P.forward(torch.from_numpy(x).cuda(), kind="siddon").cpu().numpy()
    # (a segment below 1e-5 mm may or may not be taken: left out)
    near = oracle.fp_siddon(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), one) > 0
    assert crossed.any() and not np.isfinite(got[crossed]).all() if not np.isfinite(value) else (np.abs(got[crossed]) > 1e30).all()
    clear = ~near
    assert np.isfinite(got[clear]).all()
    bulk = np.abs(got[clear] - plain[clear]) < 1e-4 * plain.max()
    assert bulk.mean() > 0.9999
