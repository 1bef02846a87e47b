"""The view split of small backprojections: parts of unequal length, fewer views
than parts want, accumulation, streamed batches and the storages, against the
FP64 sum of the single views' volumes (a single view is never split)."""
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import rel_rmse, seeded_projection, small_geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tilt", [(0.0, 0.0, 0.0), (0.02, 0.01, -0.03)])
@pytest.mark.parametrize("views", [1, 4, 7, 9, 67])
@pytest.mark.parametrize("storage,kahan", [("f32", False), ("f32", True), ("f16", True)])
def test_split_matches_single_views(ctx, storage, kahan, views, tilt):
    g = small_geometry(total_views=views, views_per_turn=max(views, 2), tilt_rad=tilt, offset_unv_mm=(1.5, 0.0, 0.5),
                       start_angle_rad=0.1)
    plan = yk.FdkPlan.from_geometry(ctx, g, filter="hann", storage=storage, kahan=kahan, parker="disabled")
    proj = seeded_projection(7, views, g.nv, g.nu)
    filtered, scales = plan.filter(torch.from_numpy(proj).cuda())
    got = plan.backproject(filtered, scales).cpu().numpy()
    one = sum(plan.backproject(filtered[i:i + 1].contiguous(), None if scales is None else scales[i:i + 1].contiguous(),
                               first=i).double() for i in range(views)).cpu().numpy()
    # single views run in one part; half storage rounds its lerps either way
    tol = 5e-6 if storage == "f32" else 2e-3
    assert rel_rmse(got, one) < tol, rel_rmse(got, one)
    acc = plan.backproject(filtered, scales, volume=torch.ones(plan.volume_shape, device="cuda"), accumulate=True)
    assert rel_rmse(acc.cpu().numpy(), got.astype(float) + 1.0) < 1e-6
    plan.close()


@pytest.mark.parametrize("batch", [5, 16, 40])
def test_streamed_batches_match_whole(ctx, batch):
    g = small_geometry(total_views=40, views_per_turn=40)
    proj = torch.from_numpy(seeded_projection(8, 40, g.nv, g.nu)).cuda()
    plan = yk.FdkPlan.from_geometry(ctx, g, filter="hann")
    whole = plan.reconstruct(proj).cpu().numpy()
    vol = torch.empty(plan.volume_shape, device="cuda")
    for at in range(0, 40, batch):
        plan.execute(proj[at:at + batch], vol, view_offset=at, clear_output=at == 0)
    assert rel_rmse(vol.cpu().numpy(), whole) < 1e-6
    plan.close()
