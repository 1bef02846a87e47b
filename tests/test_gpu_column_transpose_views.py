"""The Joseph transpose of untilted views by detector columns, in calls of the
views and voxels that it serves, on the geometries of the transpose's test:
against the FP64 oracle, accumulated, and with a pixel that is not finite."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry
from test_gpu_column_transpose import GEOMS

pytestmark = pytest.mark.gpu

VIEWS = 17


def setup(ctx, name):
    g = small_geometry(**{**GEOMS[name], "total_views": VIEWS, "views_per_turn": VIEWS})
    assert np.prod(g.volume) * VIEWS >= 8e6  # by columns from here on
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    return g, P, np.random.default_rng(61).standard_normal((VIEWS, g.nv, g.nu)).astype(np.float32)


def reference(oracle, g, P, y):
    return oracle.bp_joseph_adjoint(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), y.astype(np.float64))


@pytest.mark.parametrize("name", list(GEOMS))
def test_matches_oracle_transpose(ctx, oracle, name):
    g, P, y = setup(ctx, name)
    ref = reference(oracle, g, P, y)
    got = P.adjoint(torch.from_numpy(y).cuda(), kind="joseph").cpu().numpy()
    assert rel_rmse(got, ref) < 2e-5, rel_rmse(got, ref)
    acc = P.adjoint(torch.from_numpy(y).cuda(), kind="joseph", out=torch.ones(P.volume_shape, device="cuda"),
                    accumulate=True).cpu().numpy()
    assert rel_rmse(acc, ref + 1.0) < 2e-5


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
