"""Projector calls captured into a graph, replayed after calls that need larger
scratch arrays than the captured one: the replays go on using theirs.  Each is
replayed three times between eager work, on new inputs, and compared with the
eager call."""
import numpy as np
import pytest
import torch

import fdk_cuda_impl_amd as yk
from helpers import small_geometry

pytestmark = pytest.mark.gpu

OFF = dict(start_angle_rad=0.1, offset_unv_mm=(0.3, 0.0, 0.2))
COUNT = 3  # views of the captured call; the eager ones take all 24


@pytest.mark.parametrize("tilt", [(0.0, 0.0, 0.0), (0.02, 0.01, -0.03)], ids=["untilted", "tilted"])
@pytest.mark.parametrize("kind", ["joseph_voxel", "fdk", "joseph", "siddon"])
def test_backprojection_replays(kind, tilt):
    g = small_geometry(tilt_rad=tilt, **OFF)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = yk.Context(0, synchronous=False)
        P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
        rng = np.random.default_rng(81)
        y = torch.from_numpy(rng.standard_normal((COUNT, g.nv, g.nu)).astype(np.float32)).cuda()
        whole = torch.from_numpy(rng.standard_normal((24, g.nv, g.nu)).astype(np.float32)).cuda()
        out = torch.empty(P.volume_shape, device="cuda")
        P.adjoint(y, kind=kind, out=out)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            P.adjoint(y, kind=kind, out=out)
        for other in ("joseph_voxel", "joseph", "siddon"):
            P.adjoint(whole, kind=other)
        for k in range(3):
            y.copy_(torch.from_numpy(rng.standard_normal((COUNT, g.nv, g.nu)).astype(np.float32)))
            filler = torch.full((1 << 20,), float("nan"), device="cuda")  # reuses what was freed, if anything was
            graph.replay()
            replayed = out.clone()
            eager = P.adjoint(y, kind=kind)
            s.synchronize()
            torch.testing.assert_close(replayed, eager, rtol=0.0, atol=0.0)
            del filler
        P.adjoint(whole, kind=kind)
        s.synchronize()
        P.close()
        ctx.close()


@pytest.mark.parametrize("kind", ["joseph", "siddon"])
def test_projection_replays(kind):
    """The untilted Joseph projection's copies are smaller than those of the Siddon one in the same arrays."""
    g = small_geometry(**OFF)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = yk.Context(0, synchronous=False)
        P = yk.Projector(ctx, g.views(), g.nu, g.nv, g.grid())
        x = torch.rand(P.volume_shape, device="cuda")
        out = torch.empty((24, g.nv, g.nu), device="cuda")
        P.forward(x, kind=kind, out=out)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            P.forward(x, kind=kind, out=out)
        for other in ("siddon", "joseph"):
            P.forward(x, kind=other)
        for k in range(3):
            x.copy_(torch.rand(P.volume_shape, device="cuda"))
            graph.replay()
            replayed = out.clone()
            eager = P.forward(x, kind=kind)
            s.synchronize()
            torch.testing.assert_close(replayed, eager, rtol=0.0, atol=0.0)
        P.close()
        ctx.close()
