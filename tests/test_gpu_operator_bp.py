"""The operator-form backprojections from the paired copy of the views and from
the views themselves, against the FP64 oracle: few and many views, remainders
of the z runs, samples on and past every detector edge, rays steepest along Z,
and volumes that reach behind the source (no sample there).  On white noise a
sample errs by its position's error: three FP32 roundings of a coordinate as
large as the detector; a depth that cancels near the source has five times
that."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2))
GEOMS = {
    "remainders": dict(volume=(17, 33, 9), **OFF),
    "truncated": dict(channels=13, rows=7, tilt_rad=(0.02, 0.01, -0.03), **OFF),
    "large_detector": dict(volume=(9, 8, 3), channels=90, rows=77, **OFF),
    "one_pixel": dict(channels=1, rows=1, channel_mm=9.0, row_mm=9.0, **OFF),
    "steep": dict(sid_mm=40.0, sdd_mm=60.0, rows=150, row_mm=1.1, volume=(16, 15, 60), voxel_mm=(1.0, 1.1, 0.7), **OFF),
    "behind_source": dict(sid_mm=9.0, sdd_mm=40.0, **OFF),
}


def tolerance(name, g):
    return 3.0 * 2.0**-24 * max(g.nu, g.nv, 56) * (5.0 if name == "behind_source" else 1.0)


@pytest.mark.parametrize("views", [1, 2, 3, 24])
@pytest.mark.parametrize("kind", ["fdk", "fdk_pseudo_matched", "joseph_voxel"])
@pytest.mark.parametrize("name", list(GEOMS))
def test_matches_oracle(ctx, oracle, name, kind, views):
    g = small_geometry(**GEOMS[name])
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    y = np.random.default_rng(14).standard_normal((g.total_views, g.nv, g.nu)).astype(np.float32)
    first = 0 if views == g.total_views else 2
    # the pseudo-matched scale and the FDK angle step are those of the plan's
    # views, so the oracle runs over all of them with the others zeroed
    y[:first], y[first + views:] = 0.0, 0.0
    ref = oracle.bp_fdk_operator(oracle.views_from_float(P.views), y.astype(np.float64), oracle_volume(oracle, g),
                                 matched={"fdk": 0, "fdk_pseudo_matched": 1, "joseph_voxel": 2}[kind])
    part = torch.from_numpy(y[first:first + views]).cuda()
    got = P.adjoint(part, kind=kind, first=first).cpu().numpy()
    assert rel_rmse(got, ref) < tolerance(name, g), rel_rmse(got, ref)
    base = np.full_like(got, np.abs(ref).max())
    acc = P.adjoint(part, kind=kind, first=first, out=torch.from_numpy(base).cuda(), accumulate=True).cpu().numpy()
    assert rel_rmse(acc, ref + base) < tolerance(name, g)


@pytest.mark.parametrize("views", [1, 4])
@pytest.mark.parametrize("kind", ["fdk", "fdk_pseudo_matched", "joseph_voxel"])
def test_long_runs(ctx, oracle, kind, views):
    """A volume of enough workgroups for the runs of eight slices, the last one of a single slice."""
    g = small_geometry(volume=(250, 243, 33), voxel_mm=(0.11, 0.1, 0.5), total_views=4, views_per_turn=4, **OFF)
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    y = np.random.default_rng(15).standard_normal((4, g.nv, g.nu)).astype(np.float32)
    y[views:] = 0.0
    ref = oracle.bp_fdk_operator(oracle.views_from_float(P.views), y.astype(np.float64), oracle_volume(oracle, g),
                                 matched={"fdk": 0, "fdk_pseudo_matched": 1, "joseph_voxel": 2}[kind])
    got = P.adjoint(torch.from_numpy(y[:views]).cuda(), kind=kind).cpu().numpy()
    assert rel_rmse(got, ref) < tolerance("long_runs", g), rel_rmse(got, ref)
