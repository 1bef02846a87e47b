"""Transposes of view sets in which some views need another form than the rest:
tilted views and views from above among untilted ones, in every order, and
untilted scans in which the volume reaches the detector or nearly the source in
some views.  Against the FP64 oracle's transposes; on zero-mean input the relative
error is that of a summand, 3 roundings of the source-detector distance over the
smallest voxel or the least depth of a voxel before the source."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2))
TILT = dict(tilt_rad=(0.02, 0.01, -0.03))


def from_above(n):
    """Views from 63 degrees above the orbit (main axis Z) with the tests' detector."""
    out = np.zeros((n, 5, 4), dtype=np.float32)
    for i in range(n):
        a, e = 0.4 * i + 0.1, 1.1
        src = 120.0 * np.array([np.cos(e) * np.cos(a), np.cos(e) * np.sin(a), np.sin(e)])
        u = np.array([-np.sin(a), np.cos(a), 0.0])
        v = np.array([-np.sin(e) * np.cos(a), -np.sin(e) * np.sin(a), np.cos(e)])
        out[i, 0, :3], out[i, 2, :3], out[i, 3, :3] = src, u, v
        out[i, 1, :3] = -src - 21.2 * u - 17.3 * v
        out[i, 4, 0] = a
    return out.reshape(n, 20)


def mixed(pattern):
    """u: untilted, t: tilted, a: from above."""
    plain = small_geometry(**OFF)
    sets = {"u": plain.views(), "t": small_geometry(**OFF, **TILT).views(), "a": from_above(24)}
    return plain, np.stack([sets[c][i] for i, c in enumerate(pattern)]), 2e-5


def scan(depth=1.0, **kw):
    g = small_geometry(**{**OFF, **kw})
    return g, g.views(), max(2e-5, 3.0 * 2.0**-24 * g.sdd_mm / min(min(g.voxel_mm), depth))


SETS = {
    "one_tilted": lambda: mixed("uuuuuuuuuutuuuuuuuuu"),
    "one_above": lambda: mixed("uuuuauuu"),
    "alternating": lambda: mixed("utuatuauttaa"),
    "long_and_short": lambda: mixed("uuuuuuuuutttuuuuttta"),
    "detector_touches": lambda: scan(sdd_mm=133.0),
    "detector_touches_tilted": lambda: scan(sdd_mm=133.0, **TILT),
    # the volume's corners come within 0.4 mm of the source plane
    "source_near": lambda: scan(depth=0.35, sid_mm=16.7, sdd_mm=60.0, channels=160, rows=120),
    "source_near_tilted": lambda: scan(depth=0.1, sid_mm=16.7, sdd_mm=60.0, channels=160, rows=120, tilt_rad=(0.002, 0.0, 0.0)),
}


@pytest.mark.parametrize("name", list(SETS))
@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_matches_oracle_transpose(ctx, oracle, kind, name):
    g, views, tol = SETS[name]()
    n = len(views)
    P = yk.Projector(ctx, views, g.nu, g.nv, g.grid())
    fn = oracle.bp_joseph_adjoint if kind == "joseph" else oracle.bp_siddon_adjoint
    y = np.random.default_rng(71).standard_normal((n, g.nv, g.nu)).astype(np.float32)
    ov, vol = oracle.views_from_float(P.views), oracle_volume(oracle, g)
    ref = fn(ov, g.nu, g.nv, vol, y.astype(np.float64))
    got = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    assert rel_rmse(got, ref) < tol, rel_rmse(got, ref)
    # a range, accumulated
    first, count = 3, n - 5
    ref = fn(ov[first:first + count], g.nu, g.nv, vol, y[first:first + count].astype(np.float64))
    acc = P.adjoint(torch.from_numpy(y[first:first + count]).cuda(), kind=kind, first=first,
                    out=torch.ones(P.volume_shape, device="cuda"), accumulate=True).cpu().numpy()
    assert rel_rmse(acc, ref + 1.0) < tol


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_extreme_pixel_reaches_only_its_voxels(ctx, oracle, kind, value):
    g, views, _ = SETS["source_near"]()
    P = yk.Projector(ctx, views, g.nu, g.nv, g.grid())
    y = np.random.default_rng(72).standard_normal((len(views), g.nv, g.nu)).astype(np.float32)
    plain = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    one = np.zeros(y.shape)
    one[3, 57, 84] = 1.0
    fn = oracle.bp_joseph_adjoint if kind == "joseph" else oracle.bp_siddon_adjoint
    met = fn(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), one)
    y[3, 57, 84] = value
    got = P.adjoint(torch.from_numpy(y).cuda(), kind=kind).cpu().numpy()
    sure, clear = met > 1e-3 * met.max(), met == 0.0
    assert sure.any() and not np.isfinite(got[sure]).any()
    # (a ray within rounding of a support's edge may or may not meet it)
    assert np.isfinite(got[clear]).mean() > 0.999
    assert (np.abs(got[clear] - plain[clear]) <= 1e-5 * np.abs(plain).max()).mean() > 0.999
