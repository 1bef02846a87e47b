"""Siddon projection and transpose of rays that lie in a plane between two cells:
a centred source, an even number of cells and an odd number of pixels, as
centred scans have them.  Such a ray belongs to the upper cell, for the
projection and for its transpose, whatever the direction it runs in; one in the
upper face of the volume to none.  The views hold multiples of 1/1024 mm, so that
the rays' zeros are exact in FP32 and FP64 alike."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import oracle_volume, rel_rmse, small_geometry

pytestmark = pytest.mark.gpu

NU, NV = 43, 35
# (the last two have middle planes that FP32 origins miss; those whose planes the
# oracle's own FP64 sums miss are left out)
VOXELS = [(1.0, 1.0, 1.0), (0.3, 0.3, 0.3), (0.8, 1.7, 1.3)]
TILTS = {"untilted": (0.0, 0.0, 0.0), "tilted": (0.02, 0.0, 0.0)}


def centred(voxel, tilt, **kw):
    g = small_geometry(channels=NU, rows=NV, total_views=8, views_per_turn=8, voxel_mm=voxel, channel_mm=voxel[0],
                       row_mm=voxel[2], tilt_rad=tilt, **kw)
    views = g.views().reshape(-1, 5, 4)

    def round_off(a):
        return np.round(a.astype(np.float64) * 1024.0) / 1024.0

    middle = round_off(views[:, 1, :3] + (NU // 2) * views[:, 2, :3] + (NV // 2) * views[:, 3, :3])
    for k in (0, 2, 3):
        views[:, k, :3] = round_off(views[:, k, :3])
    views[:, 1, :3] = middle - (NU // 2) * views[:, 2, :3].astype(np.float64) - (NV // 2) * views[:, 3, :3].astype(np.float64)
    return g, views.reshape(-1, 20)


@pytest.mark.parametrize("voxel", VOXELS, ids=["1", "0.3", "mixed"])
@pytest.mark.parametrize("tilt", list(TILTS))
def test_upper_cell(ctx, oracle, tilt, voxel):
    g, views = centred(voxel, TILTS[tilt])
    P = yk.Projector(ctx, views, g.nu, g.nv, g.grid())
    ov, vol = oracle.views_from_float(P.views), oracle_volume(oracle, g)
    rng = np.random.default_rng(41)
    x = rng.random(P.volume_shape, dtype=np.float32)
    ray = ov[:, 3:6] + (NV // 2) * ov[:, 9:12] - ov[:, 0:3]
    assert (ray[:, 2] == 0.0).all()
    ax = P.forward(torch.from_numpy(x).cuda(), kind="siddon").cpu().numpy()
    assert rel_rmse(ax, oracle.fp_siddon(ov, g.nu, g.nv, vol, x)) < 1e-5
    y = rng.standard_normal((8, NV, NU)).astype(np.float32)
    aty = P.adjoint(torch.from_numpy(y).cuda(), kind="siddon").cpu().numpy()
    assert rel_rmse(aty, oracle.bp_siddon_adjoint(ov, g.nu, g.nv, vol, y.astype(np.float64))) < 5e-5
    # view by view, the rays in the plane alone: y of one sign, so the sums do not cancel
    for i in range(8):
        row = np.zeros((1, NV, NU), dtype=np.float32)
        row[0, NV // 2] = 1.0
        row[0, :, NU // 2] = 1.0
        at = P.adjoint(torch.from_numpy(row).cuda(), kind="siddon", first=i).cpu().numpy().astype(np.float64)
        a = P.forward(torch.from_numpy(x).cuda(), kind="siddon", first=i, count=1).cpu().numpy().astype(np.float64)
        assert abs((at * x).sum() / (a * row).sum() - 1.0) < 1e-5, i


@pytest.mark.parametrize("tilt", list(TILTS))
def test_upper_face(ctx, oracle, tilt):
    """The middle row lies in the volume's upper face: projection, transpose and the solvers' row weights leave it out."""
    g, views = centred((1.0, 1.0, 1.0), TILTS[tilt], center_mm=(0.0, 0.0, -9.0))
    P = yk.Projector(ctx, views, g.nu, g.nv, g.grid())
    ov = oracle.views_from_float(P.views)
    vol = oracle.volume(*g.volume, *g.voxel_mm, center=g.center_mm)
    x = np.random.default_rng(42).random(P.volume_shape, dtype=np.float32)
    ax = P.forward(torch.from_numpy(x).cuda(), kind="siddon").cpu().numpy()
    assert rel_rmse(ax, oracle.fp_siddon(ov, g.nu, g.nv, vol, x)) < 1e-5
    assert (ax[:, NV // 2] == 0.0).all()
    row = np.zeros((8, NV, NU), dtype=np.float32)
    row[:, NV // 2] = 1.0
    assert float(P.adjoint(torch.from_numpy(row).cuda(), kind="siddon").abs().max()) == 0.0
    b = ax.copy()
    b[:, NV // 2] = 5.0
    kw = dict(method="sirt", iterations=2, forward="siddon", back="joseph_voxel", relaxation=0.7)
    got = P.algebraic(torch.from_numpy(b).cuda(), **kw).cpu().numpy()
    assert rel_rmse(got, oracle.algebraic(ov, g.nu, g.nv, vol, b, **kw)) < 1e-4
