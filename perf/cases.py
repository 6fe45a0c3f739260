"""The work whose time counts: projections, reconstructions and a training step
through the public entry points, over the sizes that this repository's
configurations, tests and benchmark use, from single small slices to the
32 x 2048^2 stack.

``listed()`` gives the standing cases, ``draw(rng)`` one more of the same
ranges, ``prepare(case, seed)`` the state a caller holds before the call,
``run(state)`` one pass, ``work(case)`` its compulsory bytes and operations and
``exact(case, seed)`` the same outputs in float64 by plain torch.

Kinds of a case:

* ``fwd`` / ``back``: one projection of an image (stack) or one backprojection
  of a sinogram (stack);
* ``grad``: a training step's share, the differentiable forward projection, a
  least-squares loss and its gradient with respect to the image;
* ``tv``: iterations of the total-variation reconstruction of one slice;
* ``batch``: Landweber iterations on slices of different geometry at once.

Inputs are random-ellipse phantoms and their analytic line integrals with
noise, as measured data are.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import gratopy_amd as gratopy
from gratopy_amd.autograd import project
from gratopy_amd.batch import batch_landweber

DEVICE = "cuda:0"
ELLIPSES = 10

# pixel-angle pairs of the benchmark stack (32 x 2048^2, 1440 angles): no drawn
# case is larger
MAX_WORK = 32 * 2048 * 2048 * 1440


def _projection(kind, geom, nx, ny, ns, na, nz=1, dtype="float32", order="F", **more):
    return dict(kind=kind, geom=geom, nx=nx, ny=ny, ns=ns, na=na, nz=nz, dtype=dtype, order=order, **more)


def listed():
    return [
        # the smallest calls: a preview or a unit test, one slice, a few angles;
        # the call's own cost decides
        dict(_projection("fwd", "radon", 64, 64, 91, 30), name="radon-fwd-64"),
        # a small ragged slice in C order, as numpy arrays arrive
        dict(_projection("back", "fan", 100, 75, 130, 45, order="C"), name="fan-back-100x75"),
        # one slice of the small parallel-beam configuration, 256^2 and 180 angles
        dict(_projection("back", "radon", 256, 256, 256, 180), name="radon-back-256"),
        # one slice of the ordinary fanbeam configuration, 512^2 and 360 angles
        dict(_projection("fwd", "fan", 512, 512, 768, 360), name="fan-fwd-512"),
        # a reconstruction of that slice: both directions and the streaming
        # updates between them, iterated
        dict(_projection("tv", "fan", 512, 512, 768, 360, iterations=20), name="fan-tv-512"),
        # one slice at the benchmark's full resolution, each direction
        dict(_projection("fwd", "radon", 2048, 2048, 2560, 1440), name="radon-fwd-2048"),
        dict(_projection("back", "fan", 2048, 2048, 2560, 1440), name="fan-back-2048"),
        # the benchmark's stack, each direction
        dict(_projection("fwd", "fan", 2048, 2048, 2560, 1440, nz=32), name="fan-fwd-2048x32"),
        dict(_projection("back", "fan", 2048, 2048, 2560, 1440, nz=32), name="fan-back-2048x32"),
        # a short odd-sized stack in C order (slice index fastest)
        dict(_projection("fwd", "radon", 301, 257, 403, 179, nz=7, order="C"), name="radon-fwd-301x257x7"),
        # the differentiation configuration: 16 slices, double precision
        dict(_projection("grad", "fan", 512, 512, 768, 360, nz=16, dtype="float64"), name="fan-grad-512x16-f64"),
        # slices of different geometry reconstructed together
        dict(kind="batch", count=16, iterations=5, dtype="float32", mix=3, name="batch-landweber-16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fwd", "fwd", "back", "back", "grad", "tv", "batch"])
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(4, 24), iterations=rng.randint(3, 8),
                    dtype=rng.choice(["float32", "float32", "float64"]), mix=rng.randrange(1 << 20))
    iterations = rng.randint(4, 20) if kind == "tv" else 0
    dtype = rng.choice(["float32", "float32", "float32", "float64"])
    order = rng.choice(["F", "F", "C"])
    geom = rng.choice(["radon", "fan"])
    nz = 1 if kind == "tv" else rng.choice([1, 1, _log_int(rng, 2, 32)])
    # a double-precision pixel-angle and each solver iteration cost a multiple
    # of a single-precision projection
    cap = MAX_WORK / (8 if dtype == "float64" else 4) / (2 if kind == "grad" else 1) / max(1, 2 * iterations)
    while True:
        nx = _log_int(rng, 48, 2048)
        ny = nx if rng.random() < 0.6 else max(32, int(nx * rng.uniform(0.7, 1.3)))
        na = max(16, min(1440, int(nx * rng.uniform(0.4, 1.0))))
        ns = max(48, int(max(nx, ny) * rng.uniform(1.0, 1.5)))
        if nx * ny * na * nz <= cap:
            break
    more = {"iterations": iterations} if kind == "tv" else {}
    return _projection(kind, geom, nx, ny, ns, na, nz=nz, dtype=dtype, order=order, **more)


# ---------------------------------------------------------------------------
# geometry
# ---------------------------------------------------------------------------
def _geometry(case):
    """Physical lengths in pixel units (one pixel is one unit wide): the image
    is max(nx, ny) wide; the parallel detector spans the image diagonal, the
    fan has its source one image width from the centre and twice that from a
    detector two image widths long."""
    n = float(max(case["nx"], case["ny"]))
    if case["geom"] == "radon":
        return dict(n=n, width=math.sqrt(2.0) * n)
    return dict(n=n, width=2.0 * n, R=2.0 * n, RE=1.0 * n)


def _settings(case):
    g = _geometry(case)
    kw = dict(n_detectors=case["ns"], detector_width=g["width"], image_width=g["n"])
    if case["geom"] == "fan":
        return gratopy.ProjectionSettings(DEVICE, gratopy.FANBEAM, (case["nx"], case["ny"]), case["na"],
                                          R=g["R"], RE=g["RE"], **kw)
    return gratopy.ProjectionSettings(DEVICE, gratopy.RADON, (case["nx"], case["ny"]), case["na"], **kw)


def _angles(case):
    period = math.pi if case["geom"] == "radon" else 2 * math.pi
    return torch.arange(case["na"], dtype=torch.float64, device=DEVICE) * (period / case["na"])


def _norm_bound(case):
    """An upper bound of the operator norm, as a caller keeps it for repeated
    reconstructions: the longest path through the image times the largest
    weight a pixel collects over the angles."""
    g = _geometry(case)
    path = math.hypot(case["nx"], case["ny"])
    if case["geom"] == "radon":
        return math.sqrt(path * math.pi)
    return math.sqrt(path * 2 * math.pi * g["R"] / (g["RE"] - 0.5 * path) * 1.2)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _ellipses(case, seed, nz):
    """Centre, half axes, orientation and density of every slice's ellipses
    (nz, ELLIPSES, 6), inside the image's inscribed circle, on the GPU."""
    rng = np.random.default_rng([seed, case["nx"], case["ny"], case["na"], nz])
    r = 0.5 * min(case["nx"], case["ny"])
    dist, ang = 0.6 * r * np.sqrt(rng.random((nz, ELLIPSES))), 2 * np.pi * rng.random((nz, ELLIPSES))
    axes = r * (0.05 + 0.3 * rng.random((2, nz, ELLIPSES)))
    e = np.stack([dist * np.cos(ang), dist * np.sin(ang), axes[0], axes[1],
                  np.pi * rng.random((nz, ELLIPSES)), 0.1 + 0.9 * rng.random((nz, ELLIPSES))], axis=-1)
    return torch.from_numpy(e).to(DEVICE)


def _order(t, order):
    """(n0, n1, nz) values of a (nz, n1, n0) tensor as a 2-D or 3-D array of the given memory order."""
    t = t.permute(2, 1, 0)
    if t.shape[2] == 1:
        t = t[:, :, 0]
    if order == "C":
        return t.contiguous()
    return t.permute(*reversed(range(t.dim()))).contiguous().permute(*reversed(range(t.dim())))


def _phantom(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dtype = getattr(torch, case["dtype"])
    e = _ellipses(case, seed, nz).to(dtype)
    x = (torch.arange(nx, device=DEVICE, dtype=dtype) - 0.5 * (nx - 1))[None, :]
    y = (torch.arange(ny, device=DEVICE, dtype=dtype) - 0.5 * (ny - 1))[:, None]
    img = torch.zeros((nz, ny, nx), dtype=dtype, device=DEVICE)
    for z in range(nz):
        for cx, cy, a, b, phi, rho in e[z]:
            c, s = torch.cos(phi), torch.sin(phi)
            u, v = ((x - cx) * c + (y - cy) * s) / a, ((y - cy) * c - (x - cx) * s) / b
            img[z] += rho * ((u * u + v * v) <= 1)
    return _order(img, case["order"])


def _rays(case):
    """Unit direction (Na, 1 or Ns) and signed distance from the centre of every ray."""
    g = _geometry(case)
    th = _angles(case)[:, None]
    s = (torch.arange(case["ns"], dtype=torch.float64, device=DEVICE) - 0.5 * (case["ns"] - 1))
    s = (s * (g["width"] / case["ns"]))[None, :]
    if case["geom"] == "radon":
        # pixels with x sin - y cos = s
        return torch.sin(th), -torch.cos(th), s.expand(case["na"], -1)
    px, py = -g["RE"] * torch.cos(th), -g["RE"] * torch.sin(th)
    dx, dy = g["R"] * torch.cos(th) + s * torch.sin(th), g["R"] * torch.sin(th) - s * torch.cos(th)
    length = torch.sqrt(dx * dx + dy * dy)
    nx, ny = dy / length, -dx / length
    return nx, ny, px * nx + py * ny


def _sinogram(case, seed, noise=0.005):
    """Line integrals of the ellipses, with noise of the given share of their mean square."""
    nz, dtype = case["nz"], getattr(torch, case["dtype"])
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed + 1)
    nx, ny, d = (t.to(dtype) for t in _rays(case))
    out = torch.zeros((nz, case["na"], case["ns"]), dtype=dtype, device=DEVICE)
    for z, es in enumerate(_ellipses(case, seed, nz).to(dtype)):
        for cx, cy, a, b, phi, rho in es:
            c, s = torch.cos(phi), torch.sin(phi)
            # the ellipse's half width across the ray and the ray's distance from its centre
            w2 = (a * (nx * c + ny * s)) ** 2 + (b * (ny * c - nx * s)) ** 2
            t = d - (nx * cx + ny * cy)
            out[z] += 2 * rho * a * b * torch.sqrt(torch.clamp(w2 - t * t, min=0)) / w2
        scale = noise * torch.sqrt(torch.mean(out[z] ** 2))
        out[z] += scale * torch.randn(out[z].shape, generator=gen, dtype=dtype, device=DEVICE)
    return _order(out, case["order"])


def _batch_cases(case):
    """Slices of the uneven mix: 128..1024 pixels, 60..720 angles, 1.5 detectors per pixel."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for i in range(case["count"]):
        n = int(rng.choice([128, 256, 384, 512, 768, 1024]))
        na = int(rng.choice([60, 120, 360, 720]))
        out.append(_projection("back", "fan" if i % 2 else "radon", n, n, int(math.ceil(1.5 * n)), na,
                               dtype=case["dtype"]))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        cases = _batch_cases(case)
        return dict(kind=kind, iterations=case["iterations"], settings=[_settings(c) for c in cases],
                    sinos=[_sinogram(c, seed + 101 * i) for i, c in enumerate(cases)],
                    norms=[_norm_bound(c) for c in cases])
    state = dict(kind=kind, settings=_settings(case))
    if kind in ("fwd", "grad"):
        state["img"] = _phantom(case, seed)
    if kind in ("back", "grad", "tv"):
        state["sino"] = _sinogram(case, seed)
    if kind == "tv":
        state.update(iterations=case["iterations"], norm=_norm_bound(case))
    return state


def run(state):
    kind = state["kind"]
    if kind == "fwd":
        return gratopy.forwardprojection(state["img"], state["settings"])
    if kind == "back":
        return gratopy.backprojection(state["sino"], state["settings"])
    if kind == "grad":
        img = state["img"].detach().requires_grad_(True)
        sino = project(img, state["settings"])
        loss = 0.5 * ((sino - state["sino"]) ** 2).sum()
        loss.backward()
        return sino.detach(), img.grad
    if kind == "tv":
        return gratopy.total_variation(state["sino"], state["settings"], MU, state["iterations"],
                                       norm_estimate=state["norm"])
    return batch_landweber(state["sinos"], state["settings"], state["iterations"],
                           norm_estimates=state["norms"])


MU = 5e-3


def _pairs(case):
    return case["nx"] * case["ny"] * case["na"] * case["nz"]


def work(case):
    """Inputs read and outputs written once; two multiply-adds per pixel-angle
    pair and direction (each pixel meets two detector bins at each angle)."""
    if case["kind"] == "batch":
        cases = _batch_cases(case)
        e = 8 if case["dtype"] == "float64" else 4
        return {"bytes": sum(e * (c["nx"] * c["ny"] + c["ns"] * c["na"]) for c in cases),
                "flops": sum(8.0 * _pairs(c) for c in cases) * case["iterations"]}
    e = 8 if case["dtype"] == "float64" else 4
    img, sino = case["nx"] * case["ny"] * case["nz"], case["ns"] * case["na"] * case["nz"]
    flops = 4.0 * _pairs(case)
    if case["kind"] == "grad":
        return {"bytes": e * (2 * img + 2 * sino), "flops": 2 * flops + 3.0 * sino}
    if case["kind"] == "tv":
        return {"bytes": e * (img + sino), "flops": case["iterations"] * (2 * flops + 30.0 * img)}
    return {"bytes": e * (img + sino), "flops": flops}


# ---------------------------------------------------------------------------
# float64 values by plain torch
# ---------------------------------------------------------------------------
class _Exact:
    """The projection pair in float64, pixel by pixel: a pixel at detector
    coordinate u gives the hat weights 1 - (u - floor u) and u - floor u to the
    bins floor u and floor u + 1 (fanbeam: over its relative depth t)."""

    def __init__(self, case):
        self.case, self.g = case, _geometry(case)
        self.mid = 0.5 * (case["ns"] - 1)
        self.ds = self.g["width"] / case["ns"]
        self.theta = _angles(case)
        nx, ny = case["nx"], case["ny"]
        self.x = (torch.arange(nx, dtype=torch.float64, device=DEVICE) - 0.5 * (nx - 1))
        self.y = (torch.arange(ny, dtype=torch.float64, device=DEVICE) - 0.5 * (ny - 1))
        if case["geom"] == "radon":
            # the scales are single precision at any type
            self.scale = 1.0 / float(np.float32(self.ds))
            self.row = torch.ones(case["ns"], dtype=torch.float64, device=DEVICE)
            self.weight = math.pi / case["na"]
        else:
            xi = (torch.arange(case["ns"], dtype=torch.float64, device=DEVICE) - self.mid) * self.ds
            self.row = torch.sqrt(xi * xi + self.g["R"] ** 2) / self.g["R"]
            self.scale = 1.0 / self.ds
            self.weight = 2 * math.pi / case["na"]

    def _chunks(self):
        """Per chunk of angles: the angles, the two bins and their weights, pixels as (Ny, Nx)."""
        per = max(1, int(2 ** 26 // (self.case["nx"] * self.case["ny"])))
        ns = self.case["ns"]
        for a0 in range(0, self.case["na"], per):
            th = self.theta[a0 : a0 + per, None, None]
            x, y, c, s = self.x[None, None, :], self.y[None, :, None], torch.cos(th), torch.sin(th)
            u, w = x * s - y * c, None
            if self.case["geom"] == "fan":
                w = self.g["R"] / (x * c + y * s + self.g["RE"])
                u = u * w
            u = u / self.ds + self.mid
            k = torch.floor(u)
            f = u - k
            k = k.long()
            lo, hi = (k >= 0) & (k < ns), (k >= -1) & (k < ns - 1)
            w0, w1 = (1 - f) * lo, f * hi
            if w is not None:
                w0, w1 = w0 * w, w1 * w
            yield a0, th.shape[0], k.clamp(0, ns - 1), (k + 1).clamp(0, ns - 1), w0, w1

    def fwd(self, img):
        """(nz, ny, nx) -> (nz, na, ns)"""
        nz, na, ns = img.shape[0], self.case["na"], self.case["ns"]
        out = torch.zeros((nz, na * ns), dtype=torch.float64, device=DEVICE)
        for a0, n, k0, k1, w0, w1 in self._chunks():
            base = (torch.arange(a0, a0 + n, device=DEVICE) * ns)[:, None, None]
            i0, i1 = (k0 + base).reshape(-1), (k1 + base).reshape(-1)
            for z in range(nz):
                out[z].index_add_(0, i0, (w0 * img[z]).reshape(-1))
                out[z].index_add_(0, i1, (w1 * img[z]).reshape(-1))
        return out.reshape(nz, na, ns) * (self.row * self.scale)

    def back(self, sino, weight=None):
        """(nz, na, ns) -> (nz, ny, nx)"""
        nz = sino.shape[0]
        s = sino * self.row * (self.weight if weight is None else weight)
        out = torch.zeros((nz, self.case["ny"], self.case["nx"]), dtype=torch.float64, device=DEVICE)
        for a0, n, k0, k1, w0, w1 in self._chunks():
            for z in range(nz):
                rows = s[z, a0 : a0 + n]
                v = torch.gather(rows, 1, k0.reshape(n, -1)) * w0.reshape(n, -1)
                v += torch.gather(rows, 1, k1.reshape(n, -1)) * w1.reshape(n, -1)
                out[z] += v.sum(0).reshape(out.shape[1:])
        return out


def _zyx(t):
    """A 2-D or 3-D array as (nz, n1, n0) float64."""
    t = t.double()
    if t.dim() == 2:
        t = t[:, :, None]
    return t.permute(2, 1, 0).contiguous()


def _like(t, case):
    """(nz, n1, n0) back to the layout ``run`` returns."""
    return _order(t, case["order"])


def _tv(case, op, f, norm):
    """Chambolle-Pock iterations as the reconstruction defines them, one slice."""
    sigma, tau = 10.0 / math.sqrt(13), 0.1 / math.sqrt(13)
    m = MU * norm ** 2
    m = m / (sigma + m)
    u = torch.zeros((1, case["ny"], case["nx"]), dtype=torch.float64, device=DEVICE)
    bar, lam = u.clone(), torch.zeros_like(f)
    vx, vy = torch.zeros_like(u), torch.zeros_like(u)
    for _ in range(case["iterations"]):
        vx[..., :-1] += sigma * (bar[..., 1:] - bar[..., :-1])
        vy[:, :-1] += sigma * (bar[:, 1:] - bar[:, :-1])
        length = torch.clamp(torch.sqrt(vx * vx + vy * vy), min=1.0)
        vx, vy = vx / length, vy / length
        lam = (lam + sigma / norm * (op.fwd(bar) - f)) * m
        # the last difference along each axis is zero in the divergence
        px, py = vx.clone(), vy.clone()
        px[..., -1] = 0
        py[:, -1] = 0
        div = px + py
        div[..., 1:] -= vx[..., :-1]
        div[:, 1:] -= vy[:, :-1]
        new = torch.clamp(u + tau * (div - op.back(lam) / norm), min=0)
        u, bar = new, 2 * new - u
    return u


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        cases = _batch_cases(case)
        if sum(_pairs(c) for c in cases) * case["iterations"] > 2e10:
            return None
        out = []
        for i, c in enumerate(cases):
            op, f, w = _Exact(c), _zyx(_sinogram(c, seed + 101 * i)), 1.0 / _norm_bound(c) ** 2
            u = torch.zeros((1, c["ny"], c["nx"]), dtype=torch.float64, device=DEVICE)
            for _ in range(case["iterations"]):
                u = u - w * op.back(op.fwd(u) - f)
            out.append(_like(u, c))
        return out
    if _pairs(case) * max(1, 2 * case.get("iterations", 1)) > 1.5e10:
        return None
    op = _Exact(case)
    if kind == "fwd":
        return _like(op.fwd(_zyx(_phantom(case, seed))), case)
    if kind == "back":
        return _like(op.back(_zyx(_sinogram(case, seed))), case)
    f = _zyx(_sinogram(case, seed))
    if kind == "tv":
        return _like(_tv(case, op, f, _norm_bound(case)), case)
    sino = op.fwd(_zyx(_phantom(case, seed)))
    # the transpose of the forward projection: its scale, without angle weights
    return _like(sino, case), _like(op.back((sino - f) * op.scale, weight=1.0), case)
