"""The column form of the Joseph projection (untilted views) against the FP64
oracle: detector rows around multiples of 64 and past one block of 384, z
counts around the 16-byte groups and past one load of 256, a column longer than
a quarter of the waves' LDS, calls with few columns (a column's slices split
over waves) and with many, source or detector inside the volume.  rel-RMSE 1e-5
and 1e-4 of the peak, the projectors' FP32 gates, in proportion to nz above 512:
a sample's z index is an FP32 number of up to nz, so on noise of one-voxel
correlation its rounding moves a sample by 2^-24 nz times the noise's step."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import max_abs, oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

GEOMS = {
    "rows1": dict(rows=1), "rows63": dict(rows=63, row_mm=0.5), "rows65": dict(rows=65, row_mm=0.5),
    "rows385": dict(rows=385, row_mm=0.1, total_views=3, views_per_turn=5),
    "rows449_flipped": dict(rows=449, row_mm=0.1, total_views=3, views_per_turn=5, rotation_direction=-1),
    "nz1": dict(volume=(23, 21, 1), rows=9, row_mm=0.3), "nz2": dict(volume=(23, 21, 2)),
    "nz255": dict(volume=(9, 8, 255), rows=130, voxel_mm=(2.0, 2.0, 0.1)),
    "nz261": dict(volume=(9, 8, 261), rows=130, voxel_mm=(2.0, 2.0, 0.1)),
    "nz1030": dict(volume=(6, 7, 1030), rows=70, voxel_mm=(2.0, 2.0, 0.03)),
    "nz4200": dict(volume=(5, 4, 4200), rows=50, voxel_mm=(2.0, 2.0, 0.008), total_views=5, views_per_turn=5),
    "one_view": dict(total_views=1, channels=301, channel_mm=0.15),
    "few_slices": dict(volume=(3, 70, 18), total_views=7, views_per_turn=7),
    "many": dict(total_views=120, views_per_turn=120, channels=41),
    "source_inside": dict(sid_mm=8.0, sdd_mm=40.0, rows=9),
    "detector_inside": dict(sdd_mm=123.0),
}


@pytest.mark.parametrize("name", list(GEOMS))
def test_forward_matches_oracle(ctx, oracle, name):
    g = small_geometry(**{"start_angle_rad": 0.1, "offset_unv_mm": (0.3, 0.0, 0.2), **GEOMS[name]})
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = np.random.default_rng(7).random((g.volume[2], g.volume[1], g.volume[0])).astype(np.float32)
    got = P.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref = oracle.fp_joseph(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), x)
    index = max(1.0, g.volume[2] / 512)
    assert rel_rmse(got, ref) < 1e-5 * index, rel_rmse(got, ref)
    assert max_abs(got, ref) < 1e-4 * index * np.abs(ref).max()
    # accumulate adds onto the output
    acc = P.forward(torch.from_numpy(x).cuda(), out=torch.ones(g.total_views, g.nv, g.nu, device="cuda"),
                    accumulate=True).cpu().numpy()
    assert rel_rmse(acc - 1.0, ref) < 2e-5 * index


@pytest.mark.parametrize("views", [19, 18])
@pytest.mark.parametrize("volume", [(23, 21, 18), (5, 70, 9)])
def test_split_over_four_and_eight_waves(ctx, oracle, views, volume):
    """2052 and 1944 columns: either side of the split of a column's slices over fewer waves."""
    g = small_geometry(total_views=views, views_per_turn=views, channels=108, channel_mm=0.4, volume=volume, start_angle_rad=0.1,
                       offset_unv_mm=(0.3, 0.0, 0.2))
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = np.random.default_rng(8).random((volume[2], volume[1], volume[0])).astype(np.float32)
    got = P.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref = oracle.fp_joseph(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), x)
    assert rel_rmse(got, ref) < 1e-5, rel_rmse(got, ref)
    assert max_abs(got, ref) < 1e-4 * np.abs(ref).max()
