"""Algebraic reconstructions on one projector in turn (schedules, subset counts
with and without single-view subsets, weight models) against the same calls on
projectors of their own, bit for bit, and against the FP64 oracle (rel-RMSE
1e-4: FP32 through the iteration)."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

GEOM = dict(total_views=8, views_per_turn=8, sid_mm=80.0, sdd_mm=160.0, channels=32, rows=24, channel_mm=1.0, row_mm=1.0,
            volume=(16, 17, 12), voxel_mm=(1.0, 1.0, 1.0))
CALLS = [
    dict(method="ossart", subsets=3), dict(method="sart"), dict(method="ossart", subsets=4, forward="siddon", back="siddon"),
    dict(method="ossart", subsets=5, back="fdk"), dict(method="sirt", weights="tigre"),
    dict(method="ossart", subsets=3, back="fdk_pseudo_matched", iterations=2), dict(method="ossart", subsets=8, order="sequential"),
    dict(method="sart", weights="detailed", back="joseph"), dict(method="ossart", subsets=3, max_value=0.01),
]


def problem(ctx):
    g = small_geometry(**GEOM)
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = torch.from_numpy(np.random.default_rng(5).random(P.volume_shape).astype(np.float32)).cuda()
    return g, P, P.forward(x, kind="joseph")


def test_calls_in_turn(ctx, oracle):
    g, P, b = problem(ctx)
    for kw in CALLS:
        kw = {**dict(iterations=1, relaxation=0.3, min_value=0.0), **kw}
        got = P.algebraic(b, **kw)
        own = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid()).algebraic(b, **kw)
        assert torch.equal(got, own), kw
        if kw.get("back") == "fdk":  # (not among the oracle's pairs)
            continue
        ref = oracle.algebraic(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), b.cpu().numpy(), **kw)
        assert rel_rmse(got.cpu().numpy(), ref) < 1e-4, (kw, rel_rmse(got.cpu().numpy(), ref))


EDGES = {
    "one_slice": dict(volume=(16, 17, 1), voxel_mm=(1.0, 1.0, 6.0)),
    "one_row": dict(volume=(1, 19, 12), voxel_mm=(5.0, 1.0, 1.0), offset_unv_mm=(0.3, 0.0, 0.2)),
    "overflowing": dict(volume=(40, 41, 30), start_angle_rad=0.1),
    "tilted": dict(tilt_rad=(0.02, 0.01, -0.03), start_angle_rad=0.1),
    "wide_fan": dict(sid_mm=40.0, sdd_mm=60.0, channels=100, channel_mm=0.9, rows=70, start_angle_rad=0.3),
}


@pytest.mark.parametrize("kind", ["joseph", "siddon"])
@pytest.mark.parametrize("weights", ["detailed", "tigre"])
@pytest.mark.parametrize("name", list(EDGES))
def test_row_weights(ctx, oracle, name, weights, kind):
    """One step from zero, x = lambda C^-1 B R^-1 b: the row weights of rays along, through and past every face."""
    g = small_geometry(**{**GEOM, **EDGES[name]})
    P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
    x = torch.from_numpy(np.random.default_rng(6).random(P.volume_shape).astype(np.float32)).cuda()
    b = P.forward(x, kind=kind)
    kw = dict(method="sirt", weights=weights, iterations=1, relaxation=0.7, forward=kind)
    got = P.algebraic(b, **kw).cpu().numpy()
    ref = oracle.algebraic(oracle.views_from_float(P.views), g.nu, g.nv, oracle_volume(oracle, g), b.cpu().numpy(), **kw)
    assert rel_rmse(got, ref) < 1e-4, rel_rmse(got, ref)
