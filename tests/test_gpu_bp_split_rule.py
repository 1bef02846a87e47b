"""Backprojections of few views about the counts from which a volume of some
millions of voxels is split by views, against the FP64 sum of the single views'
volumes."""
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import rel_rmse, seeded_projection, small_geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", [2, 11, 12, 18])
@pytest.mark.parametrize("volume", [(128, 120, 140), (160, 150, 171), (224, 200, 190)])
def test_split_matches_single_views(ctx, volume, views):
    g = small_geometry(total_views=18, views_per_turn=18, volume=volume, voxel_mm=(0.15, 0.15, 0.12), offset_unv_mm=(1.5, 0.0, 0.5),
                       start_angle_rad=0.1)
    plan = yk.FdkPlan.from_geometry(ctx, g, filter="hann", parker="disabled")
    filtered, _ = plan.filter(torch.from_numpy(seeded_projection(8, 18, g.nv, g.nu)).cuda())
    got = plan.backproject(filtered[:views].contiguous())
    one = sum(plan.backproject(filtered[i:i + 1].contiguous(), first=i).double() for i in range(views))
    assert rel_rmse(got.cpu().numpy(), one.cpu().numpy()) < 5e-6
    plan.close()
