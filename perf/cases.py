"""Performance cases of the reconstruction path.

Each case is one call, or one short run, that a program using this package
makes: FDK reconstructions from the smallest to the largest configuration,
streamed from host memory, calibrated (tilted) and short scans; the Joseph
operators and their gradients; and the iterative solvers on top of them.

A case is a dict of plain values.  ``prepare`` makes its scan, inputs and plan
from a seed, ``run`` is one pass through the public entry points, ``work`` the
bytes and operations that pass cannot do without, and ``exact`` the same
outputs in 64 bits by plain torch, without the package's code.

Scans: a circular orbit of radius 500 mm, detector at 1000 mm, a volume 128 mm
across (the scale of the package's 128^3, 256^3 and 512^3 configurations) and
a detector about 1.2 times the magnified volume wide.  The detector sits a
fraction of a pixel off centre and the orbit starts at 0.1 rad, as mounted
detectors do; ``tilt`` adds the detector tilts of a calibrated scanner.
"""
import math

import numpy as np
import torch

import fdk_cuda_impl_amd as yk
from fdk_cuda_impl_amd import autograd

SOD, SDD, WIDTH, START = 500.0, 1000.0, 128.0, 0.1
TILT = (0.002, -0.001, 0.003)  # rad, about the detector's U, V and normal axes


def _scan(op, nx, ny, nz, views, nu, nv, **more):
    c = {"op": op, "nx": nx, "ny": ny, "nz": nz, "views": views, "nu": nu, "nv": nv, "dz": 1.0, "tilt": False}
    c.update(more)
    return c


def _fdk(nx, ny, nz, views, nu, nv, **more):
    return _scan("fdk", nx, ny, nz, views, nu, nv, **{**dict(filter="hann", storage="f32", kahan=False, short=False), **more})


def listed():
    return [
        # the smallest reconstruction (a preview, the smoke run's grid): launches and host work count
        {"name": "fdk_smallest", **_fdk(32, 32, 24, 48, 64, 48)},
        # the plain FP32 configuration: 128^3 from 180 views of 256 x 256
        {"name": "fdk_plain", **_fdk(128, 128, 128, 180, 256, 256, filter="ramlak")},
        # a calibrated scanner's short scan: tilted detector, Parker weights, odd sizes, half storage
        {"name": "fdk_calibrated_short", **_fdk(201, 187, 150, 401, 301, 239, tilt=True, short=True, storage="f16", kahan=True)},
        # the headline configuration: 512^3 from 720 views of 1024 x 768, half storage with compensated sums
        {"name": "fdk_large", **_fdk(512, 512, 512, 720, 1024, 768, storage="f16", kahan=True)},
        # projections arriving in host memory in batches, volume back to the host
        {"name": "fdk_stream_host", **_scan("stream", 256, 256, 200, 360, 512, 384, filter="hann", storage="f32", kahan=False,
                                            short=False, batch=60)},
        # Joseph projection at the iterative configuration (simulation, residuals)
        {"name": "joseph_project", **_scan("project", 256, 256, 256, 360, 512, 384, kind="joseph")},
        # its exact transpose there
        {"name": "joseph_transpose", **_scan("adjoint", 256, 256, 256, 360, 512, 384, kind="joseph")},
        # one gradient of a smoothed-TV least-squares objective on a calibrated scan: forward and backward
        {"name": "joseph_gradient", **_scan("gradient", 161, 150, 121, 180, 320, 241, kind="joseph", tilt=True)},
        # the same with the Siddon model, larger
        {"name": "siddon_gradient", **_scan("gradient", 240, 231, 190, 240, 480, 360, kind="siddon", tilt=True)},
        # CGLS with the default operators
        {"name": "cgls", **_scan("cgls", 128, 128, 128, 120, 256, 192, kind="siddon", iterations=4)},
        # ordered subsets with the default operators and TV steps
        {"name": "ossart_tv", **_scan("algebraic", 128, 128, 100, 120, 256, 192, method="ossart", iterations=1, subsets=10, tv=3)},
        # view-by-view SART on a small grid: many small launches
        {"name": "sart_small", **_scan("algebraic", 64, 60, 48, 40, 128, 96, method="sart", iterations=1, subsets=1, tv=0)},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# relative cost of a voxel and view of each operation
_COST = {"fdk": 1.0, "stream": 4.0, "project": 20.0, "adjoint": 80.0, "gradient": 100.0, "cgls": 40.0, "algebraic": 60.0}


def _cost(c):
    k = {"cgls": c.get("iterations", 1), "algebraic": c.get("iterations", 1)}.get(c["op"], 1)
    return _COST[c["op"]] * k * c["nx"] * c["ny"] * c["nz"] * c["views"]


def draw(rng):
    """A case of the same ranges: grids of 24 to 512 (FDK) or 24 to 256 voxels a
    side, 24 to 720 views, tilted or not, odd sizes among them."""
    most = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["fdk", "fdk", "stream", "project", "adjoint", "adjoint", "gradient", "cgls", "algebraic"])
        n = _log(rng, 24, {"fdk": 512, "stream": 256, "cgls": 144, "algebraic": 144}.get(op, 256))
        nx, ny, nz = (max(16, int(n * rng.uniform(0.75, 1.0))) for _ in range(3))
        views = _log(rng, 24, {"fdk": 720, "stream": 360, "cgls": 120, "algebraic": 120}.get(op, 360))
        nu = max(32, int(n * rng.uniform(1.5, 2.2)))
        nv = max(24, int(nu * rng.uniform(0.6, 0.9)))
        c = _scan(op, nx, ny, nz, views, nu, nv, tilt=rng.random() < 0.4, dz=rng.choice([1.0, 1.0, 1.25]))
        if op in ("fdk", "stream"):
            c["filter"] = rng.choice(["ramlak", "hann", "shepplogan"])
            c["short"] = rng.random() < 0.25
            c["storage"] = rng.choice(["f32", "f32", "f16", "bf16"])
            c["kahan"] = rng.random() < 0.5
            if op == "stream":
                c["batch"] = rng.randrange(max(1, views // 8), views + 1)
        elif op == "adjoint":
            c["kind"] = rng.choice(["joseph", "siddon", "joseph_voxel", "fdk", "fdk_pseudo_matched"])
        elif op == "algebraic":
            c["method"] = rng.choice(["sart", "sirt", "ossart"])
            c["iterations"], c["tv"] = 1, rng.choice([0, 3])
            c["subsets"] = rng.randrange(2, 13) if c["method"] == "ossart" else 1
        else:
            c["kind"] = rng.choice(["joseph", "siddon"])
            if op == "cgls":
                c["iterations"] = rng.randrange(2, 6)
        if _cost(c) <= most:
            return c


# ---------------------------------------------------------------------------
# scans and inputs
# ---------------------------------------------------------------------------
def _voxel(c):
    v = WIDTH / max(c["nx"], c["ny"])
    return v, v, v * c["dz"]


def _pixel(c):
    return 1.2 * WIDTH * (SDD / SOD) / c["nu"]


def _range(c):
    """Scan range and number of views of a full turn."""
    if not c.get("short"):
        return 2.0 * math.pi, c["views"]
    per_turn = int(c["views"] / 0.7)  # 252 degrees: half a turn and the fan with room to spare
    return 2.0 * math.pi * c["views"] / per_turn, per_turn


def _rotate(v, axis, a):
    axis = axis / np.linalg.norm(axis)
    return v * math.cos(a) + np.cross(axis, v) * math.sin(a) + axis * (axis @ v) * (1.0 - math.cos(a))


def _views(c):
    """(views, 20) float32: source, pixel (0, 0), pixel steps along U and V, angle, four floats each."""
    _, per_turn = _range(c)
    px = _pixel(c)
    cu, cv = 0.5 * (c["nu"] - 1) - 0.31, 0.5 * (c["nv"] - 1) - 0.17
    out = np.zeros((c["views"], 20), dtype=np.float32)
    for i in range(c["views"]):
        a = START + 2.0 * math.pi * i / per_turn
        co, si = math.cos(a), math.sin(a)
        u, v, n = np.array([co, si, 0.0]), np.array([0.0, 0.0, 1.0]), np.array([si, -co, 0.0])
        if c["tilt"]:
            v, n = _rotate(v, u, TILT[0]), _rotate(n, u, TILT[0])
            u, n = _rotate(u, v, TILT[1]), _rotate(n, v, TILT[1])
            u, v = _rotate(u, n, TILT[2]), _rotate(v, n, TILT[2])
        centre = np.array([-si, co, 0.0]) * (SDD - SOD)
        out[i, 0:3] = si * SOD, -co * SOD, 0.0
        out[i, 4:7] = centre - (u * cu + v * cv) * px
        out[i, 8:11] = u * px
        out[i, 12:15] = v * px
        out[i, 16] = a
    return out


def _bodies(c, seed):
    """Ellipsoids of a scanned object: centre, semi-axes, rotation about z, attenuation (/ mm)."""
    r = np.random.RandomState(seed)
    half_z = 0.5 * c["nz"] * _voxel(c)[2]
    bodies = [((0.0, 0.0, 0.0), (0.42 * WIDTH, 0.36 * WIDTH, 0.85 * half_z), 0.3, 0.02)]
    for _ in range(7):
        p = r.uniform(-0.25, 0.25, 2) * WIDTH
        bodies.append(((p[0], p[1], r.uniform(-0.5, 0.5) * half_z), tuple(r.uniform(0.03, 0.12, 3) * WIDTH),
                       r.uniform(0.0, math.pi), r.uniform(-0.01, 0.03)))
    return bodies


def _body_maps(c, seed):
    for centre, axes, turn, mu in _bodies(c, seed):
        co, si = math.cos(turn), math.sin(turn)
        yield np.array(centre), np.array([[co, si, 0.0], [-si, co, 0.0], [0.0, 0.0, 1.0]]) / np.array(axes)[:, None], mu


def _projections(c, seed):
    """Line integrals of the object through every pixel, with detector noise."""
    views = _views(c).astype(np.float64)
    out = torch.zeros((c["views"], c["nv"], c["nu"]), device="cuda")
    u = torch.arange(c["nu"], device="cuda", dtype=torch.float32)
    v = torch.arange(c["nv"], device="cuda", dtype=torch.float32)[:, None]
    step = max(1, (1 << 25) // (c["nu"] * c["nv"]))

    def lin(m):  # columns of m at 1, u, v -> values over the detector, per view
        t = torch.tensor(m, device="cuda", dtype=torch.float32)[:, :, None, None]
        return t[:, 0] + u * t[:, 1] + v * t[:, 2]

    for at in range(0, c["views"], step):
        w = views[at:at + step]
        s, d0, du, dv = w[:, 0:3], w[:, 4:7] - w[:, 0:3], w[:, 8:11], w[:, 12:15]
        length = sum(lin(np.stack([d0[:, k], du[:, k], dv[:, k]], 1)) ** 2 for k in range(3)).sqrt_()
        for centre, m, mu in _body_maps(c, seed):
            q = (s - centre) @ m.T
            rays = [lin(np.stack([(x @ m.T)[:, k] for x in (d0, du, dv)], 1)) for k in range(3)]
            a = rays[0] ** 2 + rays[1] ** 2 + rays[2] ** 2
            qs = torch.tensor(q, device="cuda", dtype=torch.float32)[:, :, None, None]
            b = rays[0] * qs[:, 0] + rays[1] * qs[:, 1] + rays[2] * qs[:, 2]
            e = torch.tensor((q * q).sum(1) - 1.0, device="cuda", dtype=torch.float32)[:, None, None]
            out[at:at + step] += (b * b - a * e).clamp_(min=0.0).sqrt_() / a * length * (2.0 * mu)
    g = torch.Generator(device="cuda").manual_seed(seed)
    return out.add_(torch.randn(out.shape, device="cuda", generator=g), alpha=0.01)


def _object(c, seed):
    """The object on the voxel grid."""
    x, y, z = (torch.arange(n, device="cuda", dtype=torch.float32) - 0.5 * (n - 1) for n in (c["nx"], c["ny"], c["nz"]))
    vx, vy, vz = _voxel(c)
    out = torch.zeros((c["nz"], c["ny"], c["nx"]), device="cuda")
    for centre, m, mu in _body_maps(c, seed):
        p = [x * vx - centre[0], (y * vy - centre[1])[:, None], (z * vz - centre[2])[:, None, None]]
        q = sum((p[0] * m[k, 0] + p[1] * m[k, 1] + p[2] * m[k, 2]) ** 2 for k in range(3))
        out += (q <= 1.0) * mu
    g = torch.Generator(device="cuda").manual_seed(seed)
    return out.add_(torch.rand(out.shape, device="cuda", generator=g), alpha=0.002)


def prepare(case, seed):
    c, views = case, _views(case)
    ctx = yk.Context(0)
    grid = yk.grid_of((c["nx"], c["ny"], c["nz"]), _voxel(c))
    s = {"case": c, "ctx": ctx, "grid": grid}
    if c["op"] in ("fdk", "stream"):
        rng, _ = _range(c)
        s["plan"] = yk.FdkPlan(ctx, views, c["nu"], c["nv"], grid, yk.FdkOptions(
            filter=c["filter"], storage=c["storage"], kahan=c["kahan"], scan_range_rad=rng if c["short"] else 0.0,
            start_angle_rad=START))
        p = _projections(c, seed)
        if c["op"] == "stream":
            s["proj"], s["volume"] = p.cpu().numpy(), np.zeros((c["nz"], c["ny"], c["nx"]), dtype=np.float32)
        else:
            s["proj"] = p
        return s
    s["P"] = yk.Projector(ctx, views, c["nu"], c["nv"], grid)
    if c["op"] in ("project", "gradient"):
        s["x"] = _object(c, seed)
    if c["op"] != "project":
        s["b"] = _projections(c, seed)
    return s


LAM, EPS, TV_STEP = 1e-3, 1e-3, 1e-5


def run(state):
    s, c = state, state["case"]
    op = c["op"]
    if op == "fdk":
        return s["plan"].reconstruct(s["proj"])
    if op == "stream":
        s["plan"].reset()
        for at in range(0, c["views"], c["batch"]):
            s["plan"].execute(s["proj"][at:at + c["batch"]], s["volume"], view_offset=at, clear_output=at == 0)
        return s["volume"]
    if op == "project":
        return s["P"].forward(s["x"], kind=c["kind"])
    if op == "adjoint":
        return s["P"].adjoint(s["b"], kind=c["kind"])
    if op == "gradient":  # the objective of autograd.least_squares_tv and its gradient
        x = s["x"].detach().requires_grad_(True)
        r = autograd.project(x, s["P"], c["kind"]) - s["b"]
        f = 0.5 * torch.sum(r.double() * r.double()) + LAM * autograd.smoothed_tv(x, s["ctx"], s["grid"], EPS)
        (g,) = torch.autograd.grad(f, x)
        return f.detach().float(), g
    if op == "cgls":
        x, res = s["P"].cgls(s["b"], iterations=c["iterations"], forward=c["kind"], back=c["kind"])
        return x, res.astype(np.float32)
    return s["P"].algebraic(s["b"], method=c["method"], iterations=c["iterations"], subsets=c["subsets"], min_value=0.0,
                            tv_iterations=c["tv"], tv_strength=TV_STEP if c["tv"] else 0.0, tv_epsilon=EPS)


def work(case):
    c = case
    vox, det = c["nx"] * c["ny"] * c["nz"], c["views"] * c["nu"] * c["nv"]
    n = 2 ** math.ceil(math.log2(2 * c["nu"]))
    # samples of a projection: a ray takes one bilinear sample (12 FLOP) a slice,
    # or crosses about 1.5 voxels of it (2 FLOP each)
    slices = det * max(c["nx"], c["ny"])
    ray = slices * (3 if c.get("kind") == "siddon" else 12)
    back = 25 * vox * c["views"]  # a voxel-driven update
    op = c["op"]
    if op in ("fdk", "stream"):
        flops = back + c["views"] * c["nv"] * 10 * n * math.log2(n) / 2
    elif op == "project":
        flops = ray
    elif op == "adjoint":
        flops = ray if c["kind"] in ("joseph", "siddon") else back
    elif op == "gradient":
        flops = 2 * ray + 30 * vox
    elif op == "cgls":
        return {"bytes": (c["iterations"] + 1) * 4.0 * 2 * (vox + det), "flops": (2 * c["iterations"] + 1) * ray}
    else:
        u = {"sirt": 1, "sart": c["views"]}.get(c["method"], c["subsets"])
        # the row and column weights and one sweep of updates; a volume read and written per update
        return {"bytes": c["iterations"] * 4.0 * (2 * u * vox + 2 * det), "flops": (1 + c["iterations"]) * (ray + back)}
    return {"bytes": 4.0 * (vox + det), "flops": float(flops)}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
class _Exact:
    """The operators of one scan, over a voxel grid (its own by default), in float64."""

    def __init__(self, c, n=None, voxel=None):
        self.c = c
        self.n = n or (c["nx"], c["ny"], c["nz"])
        self.voxel = voxel or _voxel(c)
        self.views = torch.tensor(_views(c), device="cuda", dtype=torch.float64)
        self.voxel32 = [float(np.float32(v)) for v in self.voxel]
        self.shape = self.n[::-1]
        w = self.views.cpu().numpy()
        centre = w[:, 4:7] + 0.5 * (c["nu"] - 1) * w[:, 8:11] + 0.5 * (c["nv"] - 1) * w[:, 12:15] - w[:, 0:3]
        self.axis = np.abs(centre).argmax(1)

    def _rays(self, idx):
        """Source and pixel positions of views idx: (k, 1, 1), (k, nv, nu) per axis, in mm."""
        w = self.views[idx][:, :, None, None]
        u = torch.arange(self.c["nu"], device="cuda", dtype=torch.float64)
        v = torch.arange(self.c["nv"], device="cuda", dtype=torch.float64)[:, None]
        return [w[:, k] for k in range(3)], [w[:, 4 + k] + u * w[:, 8 + k] + v * w[:, 12 + k] for k in range(3)]

    def _groups(self, idx):
        step = max(1, (1 << 23) // (self.c["nu"] * self.c["nv"]))
        for axis in range(3):
            some = [k for k, i in enumerate(idx) if self.axis[i] == axis]
            for at in range(0, len(some), step):
                yield axis, some[at:at + step]

    def _strides(self, axes):
        s = (1, self.n[0], self.n[0] * self.n[1])
        return [s[a] for a in axes]

    def joseph(self, idx, x=None, y=None):
        """A x, or A^T y, of views idx."""
        back = x is None
        out = torch.zeros(self.n[0] * self.n[1] * self.n[2] if back else (len(idx), self.c["nv"], self.c["nu"]), device="cuda", dtype=torch.float64)
        x = None if back else x.reshape(-1)
        for axis, some in self._groups(idx):
            axes = [axis] + [a for a in range(3) if a != axis]
            src, det = self._rays([idx[k] for k in some])
            s, d = ([t[a] / self.voxel32[a] for a in axes] for t in (src, det))
            n, st = [self.n[a] for a in axes], self._strides(axes)
            den = s[0] - d[0]
            a1, a2 = (s[1] - d[1]) / den, (s[2] - d[2]) / den
            b1, b2 = s[1] - a1 * s[0] + 0.5 * (n[1] - 1), s[2] - a2 * s[0] + 0.5 * (n[2] - 1)
            length = (self.voxel32[axes[0]] ** 2 + (a1 * self.voxel32[axes[1]]) ** 2 + (a2 * self.voxel32[axes[2]]) ** 2).sqrt()
            w = y[some] * length if back else torch.zeros_like(a1)
            for k in range(n[0]):
                f1, f2 = a1 * (k - 0.5 * (n[0] - 1)) + b1, a2 * (k - 0.5 * (n[0] - 1)) + b2
                g1, g2 = f1.floor(), f2.floor()
                for e1 in (0, 1):
                    for e2 in (0, 1):
                        j1, j2 = g1 + e1, g2 + e2
                        t = (1 - (f1 - j1).abs()) * (1 - (f2 - j2).abs()) * ((j1 >= 0) & (j1 < n[1]) & (j2 >= 0) & (j2 < n[2]))
                        at = k * st[0] + j1.clamp(0, n[1] - 1).long() * st[1] + j2.clamp(0, n[2] - 1).long() * st[2]
                        if back:
                            out.index_add_(0, at.reshape(-1), (t * w).reshape(-1))
                        else:
                            w += t * x[at]
            if not back:
                out[some] = w * length
        return out.reshape(self.shape) if back else out

    def siddon(self, idx, x=None, y=None):
        """The same for the exact intersection lengths between source and pixel."""
        back = x is None
        out = torch.zeros(self.n[0] * self.n[1] * self.n[2] if back else (len(idx), self.c["nv"] * self.c["nu"]), device="cuda", dtype=torch.float64)
        x = None if back else x.reshape(-1)
        for _, some in self._groups(idx):
            src, det = self._rays([idx[k] for k in some])
            s = [t.expand(len(some), self.c["nv"], self.c["nu"]).reshape(-1) / v + 0.5 * n for t, v, n in zip(src, self.voxel32, self.n)]
            r = [(d.reshape(-1) / v + 0.5 * n) - a for d, v, n, a in zip(det, self.voxel32, self.n, s)]
            length = sum((a * v) ** 2 for a, v in zip(r, self.voxel32)).sqrt()
            main = torch.stack([a.abs() for a in r]).argmax(0)
            total = torch.zeros_like(length)
            w = None if not back else y[some].reshape(-1) * length
            for axis in range(3):
                at = (main == axis).nonzero()[:, 0]
                if not len(at):
                    continue
                axes = [axis] + [a for a in range(3) if a != axis]
                n, st = [self.n[a] for a in axes], self._strides(axes)
                p, q = [s[a][at] for a in axes], [r[a][at] for a in axes]
                acc = torch.zeros_like(p[0])
                for k in range(n[0]):
                    ta, tb = (k - p[0]) / q[0], (k + 1 - p[0]) / q[0]
                    ta, tb = torch.minimum(ta, tb).clamp(0, 1), torch.maximum(ta, tb).clamp(0, 1)
                    cells, cross = [], []
                    for m in (1, 2):  # at most one plane of either minor axis inside a slab
                        j0, j1 = (p[m] + ta * q[m]).floor(), (p[m] + tb * q[m]).floor()
                        t = (torch.maximum(j0, j1) - p[m]) / q[m]
                        cross.append(torch.where(j0 != j1, torch.minimum(torch.maximum(t, ta), tb), tb))
                        cells.append((j0, j1))
                    first, last = torch.minimum(*cross), torch.maximum(*cross)
                    one = cross[0] < cross[1]
                    for seg, j1, j2 in ((first - ta, cells[0][0], cells[1][0]),
                                        (last - first, torch.where(one, cells[0][1], cells[0][0]), torch.where(one, cells[1][0], cells[1][1])),
                                        (tb - last, cells[0][1], cells[1][1])):
                        seg = seg * ((j1 >= 0) & (j1 < n[1]) & (j2 >= 0) & (j2 < n[2]))
                        i = k * st[0] + j1.clamp(0, n[1] - 1).long() * st[1] + j2.clamp(0, n[2] - 1).long() * st[2]
                        if back:
                            out.index_add_(0, i, seg * w[at])
                        else:
                            acc += seg * x[i]
                if not back:
                    total[at] = acc
            if not back:
                out[some] = (total * length).reshape(len(some), -1)
        return out.reshape(self.shape) if back else out.reshape(len(idx), self.c["nv"], self.c["nu"])

    def _derived(self, scan_range=2.0 * math.pi):
        """Per view: source distance, detector distances, angle step, projective map rows of u, v and depth."""
        w = self.views.cpu().numpy()
        angle = np.unwrap(w[:, 16])
        step = np.abs(np.gradient(angle)) if len(angle) > 1 else np.array([1e-8])
        out = []
        for i, g in enumerate(w):
            s, d0, U, V = g[0:3], g[4:7] - g[0:3], g[8:11], g[12:15]
            n = np.cross(V, U)
            n = n / np.linalg.norm(n)
            n = -n if n @ d0 < 0 else n
            plane = d0 @ n
            sod = math.hypot(s[0], s[1])
            radial = np.array([-s[0] / sod, -s[1] / sod, 0.0])
            m = np.linalg.inv(np.array([[U @ U, U @ V], [U @ V, V @ V]])) @ np.stack([plane * U - (d0 @ U) * n, plane * V - (d0 @ V) * n])
            out.append({"src": s, "U": U, "V": V, "d0": d0, "sod": sod, "radial": radial, "plane": plane, "sdd": plane / (radial @ n),
                        "step": step[i], "map": m, "n": n, "fscale": 2.0 * math.pi / scan_range})
        return out

    def _centres(self):
        return [((torch.arange(k, device="cuda", dtype=torch.float64) - 0.5 * (k - 1)) * v).reshape([-1 if a == b else 1 for b in (2, 1, 0)])
                for a, (k, v) in enumerate(zip(self.n, self.voxel32))]

    def voxel_driven(self, idx, y, weight):
        """Sum over views of the bilinear sample at the projected voxel centre times weight."""
        out = torch.zeros(self.shape, device="cuda", dtype=torch.float64)
        der, (nu, nv) = self._derived(_range(self.c)[0]), (self.c["nu"], self.c["nv"])
        dz = max(1, (1 << 24) // (self.n[0] * self.n[1]))
        for z in range(0, self.n[2], dz):
            X, Y, Z = self._centres()
            Z = Z[z:z + dz]
            for k, i in enumerate(idx):
                d = der[i]
                p = [a - float(b) for a, b in zip((X, Y, Z), d["src"])]
                depth = p[0] * float(d["n"][0]) + p[1] * float(d["n"][1]) + p[2] * float(d["n"][2])
                u, v = ((p[0] * float(m[0]) + p[1] * float(m[1]) + p[2] * float(m[2])) / depth for m in d["map"])
                iu, iv = u.floor(), v.floor()
                fu, fv = u - iu, v - iv
                flat, val = y[k].reshape(-1), 0.0
                for e in (0, 1):
                    for f in (0, 1):
                        a, b = iu + e, iv + f
                        ok = (a >= 0) & (a < nu) & (b >= 0) & (b < nv)
                        at = b.clamp(0, nv - 1).long() * nu + a.clamp(0, nu - 1).long()
                        val = val + flat[at] * ((fu if e else 1 - fu) * (fv if f else 1 - fv) * ok)
                out[z:z + dz] += val * weight(d, p, u, v)
        return out

    def back(self, idx, y, kind):
        if kind == "joseph":
            return self.joseph(idx, y=y)
        if kind == "siddon":
            return self.siddon(idx, y=y)
        vx, vy, vz = self.voxel32
        first = self._derived()[idx[0]] if kind == "fdk_pseudo_matched" else None

        def fdk(d, p, u, v):  # the depth along the line from source to axis, over all three components
            s = d["src"]
            cc = -(p[0] * float(s[0]) + p[1] * float(s[1]) + p[2] * float(s[2])) / d["sod"] + (d["sod"] - float(s @ s) / d["sod"])
            return d["sod"] ** 2 * d["step"] * d["fscale"] / cc ** 2

        def matched(d, p, u, v):
            q2 = sum((float(d["d0"][k]) + u * float(d["U"][k]) + v * float(d["V"][k])) ** 2 for k in range(3))
            return q2 ** 1.5 / (p[0] ** 2 + p[1] ** 2 + p[2] ** 2) / d["plane"] * (
                vx * vy * vz / math.sqrt(first["U"] @ first["U"]) / math.sqrt(first["V"] @ first["V"]))

        def length(d, p, u, v):
            a = torch.stack(torch.broadcast_tensors(p[0].abs() / vx, p[1].abs() / vy, p[2].abs() / vz)).amax(0)
            return (p[0] ** 2 + p[1] ** 2 + p[2] ** 2).sqrt() / a

        return self.voxel_driven(idx, y, {"fdk": fdk, "fdk_pseudo_matched": matched, "joseph_voxel": length}[kind])

    def fdk(self, proj):
        c = self.c
        scan_range, _ = _range(c)
        der = self._derived(scan_range)
        n = 2 ** math.ceil(math.log2(2 * c["nu"]))
        f = torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64) / n
        h = math.pi * f  # half the angle pi f / cutoff at cutoff 0.5
        window = {"ramlak": torch.ones_like(f), "hann": 0.5 * (1 + torch.cos(2 * h)), "shepplogan": torch.sinc(f)}[c["filter"]]
        ramp = f * window / math.sqrt(der[0]["U"] @ der[0]["U"])
        u = torch.arange(c["nu"], device="cuda", dtype=torch.float64)
        v = torch.arange(c["nv"], device="cuda", dtype=torch.float64)[:, None]
        rows = []
        for i, d in enumerate(der):
            q2 = sum((float(d["d0"][k]) + u * float(d["U"][k]) + v * float(d["V"][k])) ** 2 for k in range(3))
            p = proj[i].double() * (d["sdd"] / q2.sqrt() * (d["sdd"] / d["sod"] / 2.0))
            if c["short"]:
                p = p * self._parker(d, float(self.views[i, 16]), scan_range)
            rows.append(torch.fft.irfft(torch.fft.rfft(p, n=n, dim=1) * ramp, n=n, dim=1)[:, :c["nu"]])

        def weight(d, p, u, v):
            r = p[0] * float(d["radial"][0]) + p[1] * float(d["radial"][1])
            return d["sod"] ** 2 * d["step"] * d["fscale"] / r ** 2

        return self.voxel_driven(range(c["views"]), rows, weight)

    def _parker(self, d, angle, scan_range):
        """Parker's short-scan weights of one view's columns (on the detector's middle row), times range / pi."""
        c = self.c
        q = d["d0"] + np.arange(c["nu"])[:, None] * d["U"] + 0.5 * (c["nv"] - 1) * d["V"]
        gamma = np.arctan2(q[:, 0] * d["radial"][1] - q[:, 1] * d["radial"][0], q[:, 0] * d["radial"][0] + q[:, 1] * d["radial"][1])
        most = max(abs(gamma[0]), abs(gamma[-1]))
        beta = (angle - float(np.float32(START))) % (2.0 * math.pi)
        rise = np.sin(0.25 * math.pi * beta / np.maximum(most + gamma, 1e-6)) ** 2
        fall = np.sin(0.25 * math.pi * (math.pi + 2 * most - beta) / np.maximum(most - gamma, 1e-6)) ** 2
        w = np.where(beta < 2 * (most + gamma), rise, np.where(beta <= math.pi + 2 * gamma, 1.0, np.where(beta < math.pi + 2 * most, fall, 0.0)))
        return torch.tensor(w * (beta > 0) * (scan_range / math.pi), device="cuda")

    def tv(self, x, eps):
        """Smoothed total variation and its gradient."""
        p, den = [], eps * eps
        for dim, v in ((2, self.voxel32[0]), (1, self.voxel32[1]), (0, self.voxel32[2])):
            g = torch.zeros_like(x)
            g.narrow(dim, 0, x.shape[dim] - 1).copy_(torch.diff(x, dim=dim) / v)
            p.append(g)
            den = den + g * g
        den, grad = den.sqrt(), torch.zeros_like(x)
        for dim, v, g in zip((2, 1, 0), self.voxel32, p):
            q = g / den / v
            grad -= q
            grad.narrow(dim, 1, x.shape[dim] - 1).add_(q.narrow(dim, 0, x.shape[dim] - 1))
        return den.sum(), grad


def _exact_algebraic(c, E, b):
    n, tigre = c["views"], c["method"] == "sart"
    sets = {"sirt": 1, "sart": n}.get(c["method"], c["subsets"])
    if tigre:  # row weights from the chord through a support box
        units = [[i] for i in range(n)]
        px = float(np.linalg.norm(E.views[0, 12:15].cpu().numpy()))
        box = [E.n[0] * E.voxel32[0] * 1.1 / 2, E.n[1] * E.voxel32[1] * 1.1 / 2, max(c["nv"] * px, E.n[2] * E.voxel32[2]) / 2]
        S = _Exact(c, (2, 2, 2), box)
    else:
        units = [list(range(k, n, sets)) for k in range(sets)]
    order = list(range(sets))
    if c["method"] == "ossart" and sets > 1:  # golden-ratio visiting order
        step = max(1, round(sets / 1.6180339887498949))
        while math.gcd(step, sets) != 1:
            step = step + 1 if step + 1 < sets else 1
        order = [k * step % sets for k in range(sets)]
    eps = float(np.float32(1e-6))
    x = torch.zeros(E.shape, device="cuda", dtype=torch.float64)
    for _ in range(c["iterations"]):
        for k in order:
            idx = units[k]
            r = b[idx].double() - E.joseph(idx, x)
            if tigre:
                w = S.joseph(idx, torch.ones((2, 2, 2), device="cuda", dtype=torch.float64))
                r = torch.where(w <= 0.5 * min(E.voxel32), r * 1e-30, r / w)
            else:
                w = E.joseph(idx, torch.ones_like(x))
                r = torch.where(w > eps, r / w.clamp(min=eps), 0.0)
            col = E.back(idx, torch.ones_like(r), "joseph_voxel")
            if tigre or sets == 1:
                col = torch.where(col <= 0, 1e30, col)
            x = (x + E.back(idx, r, "joseph_voxel") / (col + eps)).clamp_(min=0.0)
        for _ in range(c["tv"]):
            x = x - float(np.float32(TV_STEP)) * E.tv(x, float(np.float32(EPS)))[1]
        x = x.clamp_(min=0.0)
    return x


def exact(case, seed):
    c, op = case, case["op"]
    # about what 20 seconds allow
    samples = c["views"] * c["nu"] * c["nv"] * max(c["nx"], c["ny"])
    cost = {"project": 1, "adjoint": 3, "gradient": 4, "cgls": 4 * (c.get("iterations", 1) + 1), "algebraic": 4}.get(op, 0) * samples
    if cost > 6e10 or (op in ("fdk", "stream") and c["nx"] * c["ny"] * c["nz"] * c["views"] > 5e10):
        return None
    E = _Exact(c)
    every = list(range(c["views"]))
    if op in ("fdk", "stream"):
        return E.fdk(_projections(c, seed))
    if op == "project":
        x = _object(c, seed).double()
        return E.joseph(every, x) if c["kind"] == "joseph" else E.siddon(every, x)
    b = _projections(c, seed)
    if op == "adjoint":
        return E.back(every, b.double(), c["kind"])
    A = E.joseph if c.get("kind") == "joseph" else E.siddon
    if op == "gradient":
        x = _object(c, seed).double()
        r = A(every, x) - b
        value, grad = E.tv(x, float(np.float32(EPS)))
        return 0.5 * float((r * r).sum()) + LAM * float(value), A(every, y=r) + LAM * grad
    if op == "cgls":
        x = torch.zeros(E.shape, device="cuda", dtype=torch.float64)
        r = b.double()
        s = A(every, y=r)
        p, gamma, norms = s.clone(), float((s * s).sum()), [float(r.norm())]
        for _ in range(c["iterations"]):
            q = A(every, p)
            alpha = gamma / float((q * q).sum())
            x += alpha * p
            r -= alpha * q
            s = A(every, y=r)
            gamma, last = float((s * s).sum()), gamma
            p = s + (gamma / last) * p
            norms.append(float(r.norm()))
        return x, np.array(norms)
    return _exact_algebraic(c, E, b)
