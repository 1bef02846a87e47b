"""Every ray of a projection of a range of views has the bits that it has in a
projection of all of them, whatever share of the views the range is: calls of
few and many detector columns (which split a column's slices differently) and of
few and many rays for the volume (which sample it in place or from copies)."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2), total_views=40, views_per_turn=40)
RANGES = [(0, 1), (7, 3), (5, 13), (11, 20), (2, 33)]
GEOMS = {
    # 5240, 4323, 2620, 1703 ... 131 columns of one block of rows
    "columns": dict(channels=131, channel_mm=0.4, **OFF),
    "columns_300_rows": dict(channels=131, channel_mm=0.4, rows=300, row_mm=0.15, **OFF),
    "columns_tall": dict(channels=131, channel_mm=0.4, volume=(20, 24, 530), voxel_mm=(1.0, 1.0, 0.06), **OFF),
    # 0.05 to 1.9 rays and slabs a voxel
    "few_rays": dict(channels=16, channel_mm=4.0, rows=12, row_mm=4.0, volume=(64, 62, 63), voxel_mm=(0.4, 0.4, 0.4), **OFF),
    "few_rays_tilted": dict(channels=16, channel_mm=4.0, rows=12, row_mm=4.0, volume=(64, 62, 63), voxel_mm=(0.4, 0.4, 0.4),
                            tilt_rad=(0.02, 0.01, -0.03), **OFF),
    "tilted": dict(channels=131, channel_mm=0.4, tilt_rad=(0.02, 0.01, -0.03), **OFF),
}


@pytest.mark.parametrize("name", list(GEOMS))
@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_range_has_the_bits_of_the_whole(ctx, kind, name):
    g = small_geometry(**GEOMS[name])
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = torch.from_numpy(np.random.default_rng(51).random(P.volume_shape, dtype=np.float32)).cuda()
    full = P.forward(x, kind=kind).cpu().numpy()
    for first, count in RANGES:
        part = P.forward(x, kind=kind, first=first, count=count).cpu().numpy()
        np.testing.assert_array_equal(part, full[first:first + count], err_msg=f"views [{first}, {first + count})")
