"""Operator-form backprojections of views with one pixel that is not finite (a
dead pixel's -log 0): it reaches the voxels whose sample takes it and no other,
also where voxels project past the edge of the detector that it lies on."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, small_geometry

pytestmark = pytest.mark.gpu

NU, NV = 13, 7
PIXELS = [(0, 0), (0, 5), (3, 0), (3, 5), (NV - 1, 4), (2, NU - 1), (NV - 1, NU - 1)]


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("kind", ["fdk", "fdk_pseudo_matched", "joseph_voxel"])
@pytest.mark.parametrize("v,u", PIXELS)
def test_extreme_pixel_reaches_only_its_voxels(ctx, oracle, kind, v, u, value):
    # a detector smaller than the volume's projection, 24 views: the paired copy serves the call
    g = small_geometry(channels=NU, rows=NV, start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2))
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    y = np.random.default_rng(31).standard_normal((g.total_views, NV, NU)).astype(np.float32)
    plain = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    one = np.zeros(y.shape)
    one[9, v, u] = 1.0
    met = oracle.bp_fdk_operator(oracle.views_from_float(P.views), one, oracle_volume(oracle, g),
                                 matched={"fdk": 0, "fdk_pseudo_matched": 1, "joseph_voxel": 2}[kind])
    y[9, v, u] = value
    got = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    # (a sample within 1e-4 pixels of the next one may or may not take it)
    sure, clear = met > 1e-4 * met.max(), met == 0.0
    assert sure.any() and clear.any()
    assert not np.isfinite(got[sure]).any()
    assert np.isfinite(got[clear]).all()
    np.testing.assert_array_equal(got[clear], plain[clear])
