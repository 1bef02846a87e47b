"""The filter's row-pair groups, against the oracle's FP64 rows: every padded
length from the run-time one (below 64) through those sharing a wave (64 to
512) to a whole workgroup, with row counts that leave a pair without its second
row and groups without a pair.  Gates of the filter stage: rel-RMSE 2e-6 in
FP32, 11 significand bits (8 for bfloat16) in 16-bit storage."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import rel_rmse, seeded_projection, small_geometry
from test_gpu_fdk import oracle_filtered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views,rows", [(1, 1), (3, 5), (2, 16), (5, 67)])
@pytest.mark.parametrize("nu", [2, 13, 20, 32, 33, 100, 128, 200, 301, 700])
def test_rows_match_oracle(ctx, oracle, nu, views, rows):
    g = small_geometry(channels=nu, rows=rows, channel_mm=0.2, row_mm=0.2, total_views=views, views_per_turn=24,
                       volume=(6, 6, 6), voxel_mm=(0.1, 0.1, 0.1), offset_unv_mm=(0.25, 0.0, 0.0))
    plan = yk.FdkPlan.from_geometry(ctx, g, filter="hann", parker="disabled")
    proj = seeded_projection(nu + rows, views, rows, nu)
    ref, _ = oracle_filtered(oracle, plan, g, proj, filt="hann")
    d = torch.from_numpy(proj).cuda()
    assert rel_rmse(plan.filter(d, storage="f32")[0].cpu().numpy(), ref) < 2e-6
    for storage, tol in (("f16", 2.0**-11), ("bf16", 2.0**-8)):
        out, scales = plan.filter(d, storage=storage)
        got = out.float().cpu().numpy() * scales.cpu().numpy()[:, :, None]
        assert rel_rmse(got, ref) < tol
    plan.close()
