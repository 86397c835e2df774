"""Workloads of the projection operators, for timing one version of the package against another.

Each case is one pass of a user's program through the public entry points: a projection and a
backprojection, one training step through an autograd function, one filtered reconstruction, or
one call of the reconstruction server. `listed()` holds the sizes that this repository's own
workloads and tests name (64^2, 1024^2, 16 x 512^2 and 256^3 are its benchmark's, 2048^2 and
384^3 the largest jobs of its serving mix) and ragged ones between them; `draw()` gives more of
the same ranges. Images and volumes are random ellipses and ellipsoids; measured projections are
their analytic line integrals with noise.

`exact()` evaluates the same operators in 64 bits with plain torch: the ray march and the
backprojection's interpolation are torch's grid_sample, and their transposes its gradient.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

import curadon_amd as cm
from curadon_amd.serving import FBPJob, FBPServer

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


# ---------------------------------------------------------------- the cases ---------------

def _fan(op, ny, nx, cells, angles, batch=1, dtype="f32", exact_geometry=False):
    return {"op": op, "ny": ny, "nx": nx, "cells": cells, "angles": angles, "batch": batch,
            "dtype": dtype, "exact_geometry": exact_geometry}


def _cone(op, nz, ny, nx, v, u, angles, dtype="f32", views=False):
    return {"op": op, "nz": nz, "ny": ny, "nx": nx, "v": v, "u": u, "angles": angles,
            "dtype": dtype, "views": views}


def listed():
    return [
        # The smallest projection and backprojection: a test image, an inner step of a small
        # iterative solver. Latency and launches.
        {"name": "fan64_project", **_fan("fan_project", 64, 64, 91, 360)},
        # The headline workload: one projection and one backprojection of a 1024^2 slice.
        {"name": "fan1024_project", **_fan("fan_project", 1024, 1024, 1449, 720)},
        # A scanner whose detector is shifted and whose centre of rotation is off (geometry
        # honoured exactly), a rectangular slice with odd sides, 16-bit storage.
        {"name": "fan_offset_bf16",
         **_fan("fan_project", 383, 451, 701, 501, dtype="bf16", exact_geometry=True)},
        # A training step of a learned reconstruction: 16 slices through the differentiable
        # forward, squared residual, gradient through the matched adjoint.
        {"name": "fan512x16_train", **_fan("fan_train", 512, 512, 724, 512, batch=16)},
        # A reconstruction layer inside a network: the differentiable backprojection of a small
        # batch and its gradient.
        {"name": "fan256x4_layer", **_fan("fan_layer", 256, 256, 363, 400, batch=4)},
        # Filtered backprojection of one ragged slice (odd sides, odd number of angles), FP32.
        {"name": "fan_ragged_fbp", **_fan("fan_fbp", 309, 333, 475, 633)},
        # The largest fan-beam job of the serving mix, 16-bit storage.
        {"name": "fan2048_fbp_f16", **_fan("fan_fbp", 2048, 2048, 2897, 4096, dtype="f16")},
        # The cone-beam workload: one projection and one backprojection of a 256^3 volume.
        {"name": "cone256_project", **_cone("cone_project", 256, 256, 256, 384, 384, 360)},
        # A training step on a ragged 3D patch: forward, residual, gradient.
        {"name": "cone_ragged_train", **_cone("cone_train", 97, 120, 133, 150, 171, 90)},
        # A reconstruction layer on a helical scan given by its views, and its gradient.
        {"name": "cone_helix_layer",
         **_cone("cone_layer", 128, 128, 128, 192, 192, 180, views=True)},
        # The largest cone-beam job of the serving mix: FDK with 16-bit storage.
        {"name": "cone384_fdk_f16",
         **_cone("cone_fdk", 384, 384, 384, 576, 576, 768, dtype="f16")},
        # The server with small jobs of mixed size waiting: the low end of its mix, where a job
        # alone does not fill the GPU.
        {"name": "serve_small_f16", "op": "serve", "sizes": "128 256 128 c64 512 200 c128 256",
         "dtype": "f16"},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Sizes over their logarithm from the smallest listed ones to the largest, sides and
    detectors ragged half of the time, every operation, dtype and geometry option."""
    op = rng.choice(["fan_project", "fan_project", "fan_train", "fan_layer", "fan_fbp", "fan_fbp",
                     "cone_project", "cone_project", "cone_train", "cone_layer", "cone_fdk",
                     "serve"])
    dtype = rng.choice(["f32", "f32", "f16", "bf16"])
    ragged = rng.random() < 0.5
    if op == "serve":
        sizes = [str(_spread(rng, 64, 512)) for _ in range(rng.randint(3, 8))]
        sizes += ["c%d" % _spread(rng, 32, 128) for _ in range(rng.randint(0, 2))]
        return {"op": op, "sizes": " ".join(sizes), "dtype": rng.choice(["f32", "f16", "bf16"])}
    if op.startswith("fan"):
        top = {"fan_project": 1448, "fan_train": 724, "fan_layer": 724, "fan_fbp": 2048}[op]
        n = _spread(rng, 64, top)
        ny = max(48, int(n * rng.uniform(0.7, 1.0))) if ragged else n
        nx = n
        cells = math.ceil(math.sqrt(2) * n) + (rng.randint(-9, 40) if ragged else 0)
        angles = max(60, int(n * rng.uniform(0.6, 2.0)))
        if not ragged:
            nx = ny = n + n % 2
            angles -= angles % 4
        batch = 1
        if op in ("fan_train", "fan_layer"):
            batch = max(1, min(16, int(16 * 512 * 512 / (n * n)), _spread(rng, 1, 16)))
        exact = ragged and op in ("fan_project", "fan_train") and rng.random() < 0.4
        return _fan(op, ny, nx, cells, angles, batch, dtype, exact)
    top = {"cone_project": 256, "cone_train": 144, "cone_layer": 144, "cone_fdk": 320}[op]
    n = _spread(rng, 48, top)
    nz, ny, nx = n, n, n
    v = u = int(1.5 * n)
    angles = max(30, int(n * rng.uniform(0.6, 1.4)))
    if ragged:
        nz, ny = (max(32, int(n * rng.uniform(0.6, 1.0))) for _ in range(2))
        v, u = int(v * rng.uniform(0.7, 1.0)), u + rng.randint(-7, 12)
    views = op in ("cone_project", "cone_layer") and rng.random() < 0.4
    return _cone(op, nz, ny, nx, v, u, angles, dtype, views)


# ---------------------------------------------------------------- geometries --------------

def _fan_distances(c):
    n = max(c["ny"], c["nx"])
    return 2.0 * n, 3.0 * n                      # source to isocentre, source to detector


# detector offset (cells), detector rotation (radians) and centre of rotation of the scanners
# whose geometry is not ideal
OFFSET, PITCH, COR = 6.25, 0.01, 1.5


def _fan_angles(c):
    return np.linspace(0, 2 * np.pi, c["angles"], endpoint=False)


def _fan_geometry(c):
    dso, dsd = _fan_distances(c)
    more = {}
    if c["exact_geometry"]:
        more = {"det_offset": OFFSET, "det_rotation": PITCH, "COR": COR, "exact_geometry": True}
    t = DTYPES[c["dtype"]]
    return cm.FanGeometry(DSD=dsd, DSO=dso, angles=_fan_angles(c), vol_shape=(c["ny"], c["nx"]),
                          det_shape=c["cells"], vol_prec=t, sino_prec=t, **more)


def _cone_distances(c):
    n = max(c["nz"], c["ny"], c["nx"])
    return 2.0 * n, 3.0 * n


def _helix(c):
    """Views of a helical scan about the y axis (1.3 turns) with a panel facing the source and
    turned a little about its normal: source, panel centre, u step, v step."""
    dso, dsd = _cone_distances(c)
    A, h = c["angles"], 0.3 * c["ny"]
    t = 2 * np.pi * 1.3 * np.arange(A) / A
    rise = np.linspace(-h, h, A)
    away = np.stack([np.sin(t), 0 * t, np.cos(t)], 1)      # from the source to the axis
    side = np.stack([np.cos(t), 0 * t, -np.sin(t)], 1)
    up = np.tile([0.0, 1.0, 0.0], (A, 1))
    src = -dso * away + rise[:, None] * up
    centre = src + dsd * away
    ct, st = math.cos(0.02), math.sin(0.02)
    return np.concatenate([src, centre, ct * side + st * up, -st * side + ct * up], 1)


def _cone_angles(c):
    return np.linspace(0, 2 * np.pi, c["angles"], endpoint=False)


def _cone_geometry(c):
    dso, dsd = _cone_distances(c)
    shape, panel, t = (c["nz"], c["ny"], c["nx"]), (c["v"], c["u"]), DTYPES[c["dtype"]]
    if c["views"]:
        return cm.ConeGeometry.from_vec(shape, panel, _helix(c), vol_prec=t, sino_prec=t)
    return cm.ConeGeometry(DSD=dsd, DSO=dso, angles=_cone_angles(c), vol_shape=shape,
                           det_shape=panel, vol_prec=t, sino_prec=t)


# The rays as the reference sets them up, in 64 bits and in the order of operations that its
# formulas give (the sample counts round, so the order matters). Texel i of an image is centred
# at i + 0.5, voxel i of a volume at i.

def _fan_frames(c):
    """Per angle, in texel coordinates: source, source to cell 0, cell step. (A, 2) each."""
    dso, dsd = _fan_distances(c)
    D, ext = c["cells"], (float(c["nx"]), float(c["ny"]))
    src, org, step = [], [], []

    def turned(x, y, co, si):
        return x * co + y * si, -x * si + y * co

    for al in _fan_angles(c):
        co, si = math.cos(al), math.sin(al)
        if c["exact_geometry"]:
            s = turned(-COR, dso, co, si)
            m = turned(OFFSET - COR, -(dsd - dso), co, si)
            u = turned(math.cos(PITCH), math.sin(PITCH), co, si)
            r0 = [m[d] - (D - 1.0) / 2.0 * u[d] - s[d] for d in (0, 1)]
            r1 = [r0[d] + u[d] for d in (0, 1)]
        else:
            s = turned(0.0, dso, co, si)
            p0, p1 = turned(-D / 2.0 + 0.5, -(dsd - dso), co, si), \
                turned(-D / 2.0 + 1.5, -(dsd - dso), co, si)
            r0, r1 = [p0[d] - s[d] for d in (0, 1)], [p1[d] - s[d] for d in (0, 1)]
        src.append([s[d] + 0.5 * ext[d] for d in (0, 1)])
        org.append(r0)
        step.append([r1[d] - r0[d] for d in (0, 1)])
    return tuple(torch.tensor(v, dtype=torch.float64) for v in (src, org, step))


def _clip(s, d, hi):
    """Parameters at which the rays s + t d enter and leave the boxes [-1, hi]."""
    tiny, huge = float(np.finfo(np.float32).tiny), float(np.finfo(np.float32).max)
    t0 = torch.full(d.shape[:-1], tiny, dtype=torch.float64, device=d.device)
    t1 = torch.full_like(t0, huge)
    for k, h in enumerate(hi):
        a = (-1.0 - s[..., k]) / d[..., k]
        b = (h - s[..., k]) / d[..., k]
        t0, t1 = (torch.fmin(torch.fmax(a, t0), torch.fmax(b, t0)),
                  torch.fmax(torch.fmin(a, t1), torch.fmin(b, t1)))
    return t0, t1


def _fan_rays(c, frames, angles):
    """Entry point (in index coordinates), step, step length and number of samples of the rays
    of some angles: (R, 2), (R, 2), (R,), (R,)."""
    src, org, step = (v[angles] for v in frames)
    k = torch.arange(c["cells"], dtype=torch.float64, device=src.device)[None, :, None]
    d = (org[:, None] + k * step[:, None]).reshape(-1, 2)
    s = src[:, None].expand(-1, c["cells"], -1).reshape(-1, 2)
    t0, t1 = _clip(s, d, (float(c["nx"]), float(c["ny"])))
    q = d * (t1 - t0)[:, None]
    m = q.abs().amax(1)
    v = q / m[:, None]
    n = torch.where(t0 > t1 - 1e-6, torch.zeros_like(m), torch.round(m))
    return s + t0[:, None] * d - 0.5, v, torch.hypot(v[:, 0], v[:, 1]), n


def _cone_frames(c):
    """Per angle, in voxel coordinates (x, y, z): pixel (0, 0), u step, v step, source."""
    U, V, n = c["u"], c["v"], [float(c[k]) for k in ("nx", "ny", "nz")]
    mid = [k * 1.0 / 2.0 - 1.0 / 2.0 for k in n]
    out = []
    if c["views"]:
        for w in _helix(c).tolist():
            o = [w[3 + d] - (U - 1.0) / 2.0 * w[6 + d] - (V - 1.0) / 2.0 * w[9 + d] + mid[d]
                 for d in range(3)]
            out.append([o, w[6:9], w[9:12], [w[d] + mid[d] for d in range(3)]])
    else:
        dso, dsd = _cone_distances(c)
        x, y, z = -(U / 2.0) + 0.5, -(V / 2.0) + 0.5, dsd - dso
        for al in _cone_angles(c):
            co, si = math.cos(al), math.sin(al)
            p = [[co * a + si * e + mid[0], b + mid[1], -si * a + co * e + mid[2]]
                 for a, b, e in ((x, y, z), (x + 1.0, y, z), (x, y + 1.0, z), (0.0, 0.0, -dso))]
            out.append([p[0], [p[1][d] - p[0][d] for d in range(3)],
                        [p[2][d] - p[0][d] for d in range(3)], p[3]])
    return torch.tensor(out, dtype=torch.float64)


def _cone_rays(c, frames, a):
    """First sample, step and number of samples of the rays of one angle: (V U, 3), ..., (V U,)."""
    org, du, dv, src = frames[a]
    u = torch.arange(c["u"], dtype=torch.float64, device=frames.device)[None, :, None]
    v = torch.arange(c["v"], dtype=torch.float64, device=frames.device)[:, None, None]
    d = (org + u * du + v * dv - src).reshape(-1, 3)
    budget = torch.ceil(torch.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]))
    s = src.expand_as(d)
    t0, t1 = _clip(s, d, [c[k] + 1.0 for k in ("nx", "ny", "nz")])
    steps = torch.ceil((t1 - t0) * budget)
    dt = torch.where(steps > 0, (t1 - t0) / steps, torch.zeros_like(steps))
    n = torch.where(t0 <= t1, steps + 1.0, torch.zeros_like(steps))
    return s + t0[:, None] * d, dt[:, None] * d, n


# ---------------------------------------------------------------- inputs ------------------

def _density(c):
    """Largest density of an ellipse. Unfiltered operators get attenuations, whose line integrals
    are a few units; reconstructions the densities up to 1 that the serving mix has, whose
    filtered projections 16-bit storage holds well."""
    return 1.0 if c["op"] in ("fan_fbp", "cone_fdk") else \
        8.0 / max(c["nx"], c["ny"], c.get("nz", 0))


def _noise(c):
    return 1.25e-3 * max(c["nx"], c["ny"], c.get("nz", 0)) * _density(c)


def _ellipses(seed, batch, ny, nx, density, count=10):
    """(batch, count, 6): centre, semi-axes, angle, density."""
    r = np.random.RandomState(seed % (1 << 31))
    u = r.rand(batch, count, 6)
    lo, hi = np.array([-.4 * nx, -.4 * ny, nx / 32, ny / 32, 0, 0]), \
        np.array([.4 * nx, .4 * ny, nx / 3.2, ny / 3.2, np.pi, density])
    return torch.tensor(lo + (hi - lo) * u, device=DEV)


def _image(E, ny, nx):
    y = (torch.arange(ny, dtype=torch.float64, device=DEV) - ny / 2 + .5)[:, None]
    x = (torch.arange(nx, dtype=torch.float64, device=DEV) - nx / 2 + .5)[None, :]
    out = torch.zeros(len(E), ny, nx, device=DEV)
    for b, es in enumerate(E.tolist()):
        for cx, cy, p, q, th, rho in es:
            co, si = math.cos(th), math.sin(th)
            inside = (((x - cx) * co + (y - cy) * si) / p) ** 2 + \
                (((y - cy) * co - (x - cx) * si) / q) ** 2 <= 1
            out[b] += rho * inside
    return out


def _noisy(p, seed, level):
    g = torch.Generator(device=DEV).manual_seed(seed + 17)
    return p + level * torch.randn(p.shape, generator=g, device=DEV)


def _chord(A, B, C):
    return torch.where(A > 0, (B * B - A * C).clamp_min(0).sqrt() / A, torch.zeros_like(A)) * 2


def _fan_sinogram(c, E, seed):
    """Line integrals of the ellipses, with the noise of a scan: (batch, A, D)."""
    src, org, step = (v.to(DEV) for v in _fan_frames(c))
    k = torch.arange(c["cells"], dtype=torch.float64, device=DEV)[None, :, None]
    d = org[:, None] + k * step[:, None]
    d = d / d.norm(dim=-1, keepdim=True)
    s = src[:, None] - torch.tensor([c["nx"] / 2, c["ny"] / 2], device=DEV)
    out = torch.zeros(len(E), c["angles"], c["cells"], device=DEV)
    for b, es in enumerate(E.tolist()):
        for cx, cy, p, q, th, rho in es:
            R = torch.tensor([[math.cos(th) / p, -math.sin(th) / q],
                              [math.sin(th) / p, math.cos(th) / q]], dtype=torch.float64,
                             device=DEV)
            e, f = (s - torch.tensor([cx, cy], device=DEV)) @ R, d @ R
            out[b] += rho * _chord((f * f).sum(-1), (e * f).sum(-1), (e * e).sum(-1) - 1)
    return _noisy(out, seed, _noise(c))


def _ellipsoids(seed, nz, ny, nx, density, count=20):
    """(count, 7): centre (x, y, z), semi-axes, density."""
    r = np.random.RandomState(seed % (1 << 31))
    n = np.array([nx, ny, nz], float)
    u = r.rand(count, 7)
    lo = np.concatenate([-.4 * n, n / 32, [0]])
    hi = np.concatenate([.4 * n, n / 3.2, [density]])
    return (lo + (hi - lo) * u).tolist()


def _volume(E, nz, ny, nx):
    ax = [torch.arange(n, dtype=torch.float32, device=DEV) - n / 2 + .5 for n in (nz, ny, nx)]
    z, y, x = ax[0][:, None, None], ax[1][None, :, None], ax[2][None, None, :]
    out = torch.zeros(nz, ny, nx, device=DEV)
    for cx, cy, cz, p, q, r, rho in E:
        out += rho * (((x - cx) / p) ** 2 + ((y - cy) / q) ** 2 + ((z - cz) / r) ** 2 <= 1)
    return out


def _cone_projections(c, E, seed):
    """Line integrals of the ellipsoids, with the noise of a scan: (A, V, U)."""
    f = _cone_frames(c).to(DEV)
    u = torch.arange(c["u"], dtype=torch.float64, device=DEV)[None, None, :, None]
    v = torch.arange(c["v"], dtype=torch.float64, device=DEV)[None, :, None, None]
    out = torch.zeros(c["angles"], c["v"], c["u"], device=DEV)
    mid = torch.tensor([(c[k] - 1) / 2 for k in ("nx", "ny", "nz")], dtype=torch.float64,
                       device=DEV)
    for a in range(0, c["angles"], 32):
        org, du, dv, src = (f[a:a + 32, i][:, None, None] for i in range(4))
        d = org + u * du + v * dv - src
        d = (d / d.norm(dim=-1, keepdim=True)).float()
        s = (src - mid).float()
        for cx, cy, cz, p, q, r, rho in E:
            R = torch.tensor([1 / p, 1 / q, 1 / r], device=DEV)
            e, g = (s - torch.tensor([cx, cy, cz], device=DEV)) * R, d * R
            out[a:a + 32] += rho * _chord((g * g).sum(-1), (e * g).sum(-1), (e * e).sum(-1) - 1)
    return _noisy(out, seed, _noise(c))


def _serve_cases(c):
    """The jobs of a serving case as reconstruction cases: n is an n^2 slice, cn an n^3 volume."""
    jobs = []
    for s in c["sizes"].split():
        n = int(s.lstrip("c"))
        if s.startswith("c"):
            jobs.append(_cone("cone_fdk", n, n, n, n * 3 // 2, n * 3 // 2, 2 * n, c["dtype"]))
        else:
            jobs.append(_fan("fan_fbp", n, n, math.ceil(math.sqrt(2) * n), 2 * n, 1, c["dtype"]))
    return jobs


def _inputs(c, seed):
    """The arrays a program has before the call."""
    t = DTYPES[c["dtype"]]
    if c["op"] == "serve":
        return {"jobs": [_inputs(j, seed + 101 * i)["p"]
                         for i, j in enumerate(_serve_cases(c))]}
    if c["op"].startswith("fan"):
        E = _ellipses(seed, c["batch"], c["ny"], c["nx"], _density(c))
        if c["op"] == "fan_fbp":
            return {"p": _fan_sinogram(c, E, seed)[0]}         # raw projections stay FP32
        p = _fan_sinogram(c, E, seed).to(t)
        if c["op"] == "fan_layer":                             # and the gradient that comes back
            return {"p": p, "g": _noisy(_image(E, c["ny"], c["nx"]), seed, 0.1).to(t)}
        if c["op"] == "fan_train":                             # a perturbed estimate
            r = np.random.RandomState((seed + 1) % (1 << 31)).rand(*E.shape[:2], 1)
            E = E * torch.tensor(0.95 + 0.1 * r, device=DEV)
        x = _image(E, c["ny"], c["nx"]).to(t)
        return {"x": x if c["batch"] > 1 else x[0], "p": p if c["batch"] > 1 else p[0]}
    E = _ellipsoids(seed, c["nz"], c["ny"], c["nx"], _density(c))
    if c["op"] == "cone_fdk":
        return {"p": _cone_projections(c, E, seed)}
    p = _cone_projections(c, E, seed).to(t)
    x = _volume(E, c["nz"], c["ny"], c["nx"])
    if c["op"] == "cone_layer":
        return {"p": p, "g": _noisy(x, seed, 0.1).to(t)}
    return {"x": (x * 0.97 if c["op"] == "cone_train" else x).to(t), "p": p}


def prepare(case, seed):
    s = {"op": case["op"], **_inputs(case, seed)}
    if case["op"] == "serve":
        jobs = _serve_cases(case)
        s["geoms"] = [_fan_geometry(j) if j["op"] == "fan_fbp" else _cone_geometry(j)
                      for j in jobs]
        s["server"] = FBPServer(storage=DTYPES[case["dtype"]])
        return s
    s["geom"] = _fan_geometry(case) if case["op"].startswith("fan") else _cone_geometry(case)
    s["geom"].plan                                             # built once, kept with the geometry
    if case["op"].endswith("_train"):
        s["x"].requires_grad_(True)
    if case["op"].endswith("_layer"):
        s["p"].requires_grad_(True)
    return s


def run(state):
    op = state["op"]
    if op == "serve":
        jobs = [FBPJob(g, p) for g, p in zip(state["geoms"], state["jobs"])]
        state["server"].run(jobs)
        return [j.volume for j in jobs]
    g = state["geom"]
    if op.endswith("_project"):
        return {"sino": cm.forward(state["x"], g), "back": cm.backward(state["p"], g)}
    if op.endswith("_train"):
        q = cm.TorchForward.apply(state["x"], g)
        loss = ((q - state["p"]).float() ** 2).sum()
        grad, = torch.autograd.grad(loss, state["x"])
        return {"sino": q.detach(), "loss": loss.detach(), "grad": grad}
    if op.endswith("_layer"):
        v = cm.TorchBackprojection.apply(state["p"], g)
        grad, = torch.autograd.grad(v, state["p"], state["g"])
        return {"volume": v.detach(), "grad": grad}
    return cm.fbp(state["p"], g)


# ---------------------------------------------------------------- what a pass needs -------

def _samples(c):
    """Samples of one forward march, from some of the angles."""
    every = max(1, c["angles"] // 12)
    picked = list(range(0, c["angles"], every))
    if c["op"].startswith("fan"):
        n = float(_fan_rays(c, _fan_frames(c), picked)[3].sum())
    else:
        f = _cone_frames(c)
        n = sum(float(_cone_rays(c, f, a)[2].sum()) for a in picked)
    return n * c["angles"] / len(picked)


def work(case):
    """Bytes: every input read and every output written once. Operations: per sample of a march
    and per pixel and angle of a backprojection, the interpolation, its position and the sum."""
    if case["op"] == "serve":
        parts = [work(j) for j in _serve_cases(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    b = torch.tensor([], dtype=DTYPES[case["dtype"]]).element_size()
    if case["op"].startswith("fan"):
        vol = case["ny"] * case["nx"] * case["batch"]
        sino = case["angles"] * case["cells"] * case["batch"]
        width, per_sample, per_voxel, rows = case["cells"], 9, 13, 1
        march = case["batch"]
    else:
        vol = case["nz"] * case["ny"] * case["nx"]
        sino = case["angles"] * case["v"] * case["u"]
        width, per_sample, per_voxel, rows = case["u"], 24, 22, 1
        march = 1
    kind = case["op"].split("_")[1]
    back = vol * case["angles"] * per_voxel * rows
    if kind == "project":
        return {"bytes": 2 * b * (vol + sino), "flops": march * per_sample * _samples(case) + back}
    if kind == "train":
        return {"bytes": 2 * b * (vol + sino),
                "flops": 2 * march * per_sample * _samples(case) + 3 * sino}
    if kind == "layer":
        return {"bytes": 2 * b * (vol + sino), "flops": 2 * back}
    return {"bytes": 4 * sino + b * vol, "flops": back + sino * 10 * math.log2(2 * width)}


# ---------------------------------------------------------------- 64 bits -----------------

_CHUNK = 1 << 24                                               # samples evaluated at a time


def _grid(i, n):
    """grid_sample's coordinate of index i along an axis of n elements."""
    return i * (2.0 / (n - 1)) - 1.0 if n > 1 else i


def _sample(img, at):
    """Multilinear samples of img (1, C, ...) at index coordinates at[..., (x, y, ...)], zero
    outside. One element is added on each side, so that an axis of one element works too."""
    img = F.pad(img, (1, 1) * (img.dim() - 2))
    g = torch.stack([_grid(at[..., k] + 1.0, img.shape[-1 - k]) for k in range(at.shape[-1])], -1)
    return F.grid_sample(img, g, mode="bilinear", padding_mode="zeros", align_corners=True)


def _march(img, start, step, n, scale):
    """Sums of samples of img (C, ...) along rays, (C, R)."""
    out = []
    J = int(n.max()) if n.numel() else 0
    if J == 0:
        return torch.zeros(len(img), len(n), dtype=torch.float64, device=img.device)
    j = torch.arange(J, dtype=torch.float64, device=img.device)
    for r in range(0, len(n), max(1, _CHUNK // J)):
        k = slice(r, r + max(1, _CHUNK // J))
        at = start[k, None] + j[:, None] * step[k, None]
        at = at[None] if img.dim() == 3 else at[None, None]
        s = _sample(img[None], at).reshape(len(img), -1, J)
        out.append((s * (j < n[k, None])).sum(-1) * scale[k])
    return torch.cat(out, 1)


def _transposed(f, like, y):
    """Gradient of <f(v), y> with respect to v at 0, that is the transpose of f on y."""
    v = torch.zeros_like(like, requires_grad=True)
    with torch.enable_grad():
        g, = torch.autograd.grad(f(v), v, y)
    return g


class _Fan64:
    """The fan-beam operators in 64 bits."""

    def __init__(self, c, weighting=1):
        self.c, self.p = c, weighting
        self.frames = tuple(v.to(DEV) for v in _fan_frames(c))

    def _angles(self):
        step = max(1, (_CHUNK // max(self.c["ny"], self.c["nx"])) // self.c["cells"])
        for a in range(0, self.c["angles"], step):
            yield list(range(a, min(a + step, self.c["angles"])))

    def forward(self, x):
        out = []
        for a in self._angles():
            s, v, l, n = _fan_rays(self.c, self.frames, a)
            n = torch.nan_to_num(n)
            out.append(_march(x, s, v, n, l).view(len(x), len(a), -1))
        return torch.cat(out, 1)

    def adjoint(self, y):
        out = torch.zeros(len(y), self.c["ny"], self.c["nx"], dtype=torch.float64, device=DEV)
        for a in self._angles():
            s, v, l, n = _fan_rays(self.c, self.frames, a)
            J = int(n.max())
            for r in range(0, len(n), max(1, _CHUNK // J)):
                k = slice(r, r + max(1, _CHUNK // J))
                out += _transposed(lambda w: _march(w, s[k], v[k], n[k], l[k]), out,
                                   y[:, a].reshape(len(y), -1)[:, k])
        return out

    def _view(self, a):
        """Depth normal, its offset, source to detector, cell axis, its offset, cell offset and
        the reciprocal cell size of angle a, in the reference's pixel frame."""
        c = self.c
        dso, dsd = _fan_distances(c)
        al = float(_fan_angles(c)[a])
        co, si = math.cos(al), math.sin(al)
        if not c["exact_geometry"]:
            return (-si, -co, dso, dsd, co, -si, 0.0, c["cells"] / 2.0)
        t = lambda x, y: (x * co + y * si, -x * si + y * co)  # noqa: E731
        s, m = t(-COR, dso), t(OFFSET - COR, -(dsd - dso))
        e = t(math.cos(PITCH), math.sin(PITCH))
        n, d = (-e[1], e[0]), (m[0] - s[0], m[1] - s[1])
        if n[0] * d[0] + n[1] * d[1] < 0:
            n = (-n[0], -n[1])
        return (n[0], n[1], -(n[0] * s[0] + n[1] * s[1]), n[0] * d[0] + n[1] * d[1], e[0], e[1],
                -(e[0] * s[0] + e[1] * s[1]),
                -(e[0] * d[0] + e[1] * d[1]) + c["cells"] / 2.0)

    def _back_one(self, row, a):
        """Backprojection of the row (B, D) of angle a: (B, ny, nx)."""
        c = self.c
        y = (torch.arange(c["ny"], dtype=torch.float64, device=DEV) - c["ny"] / 2 + .5)[:, None]
        x = (torch.arange(c["nx"], dtype=torch.float64, device=DEV) - c["nx"] / 2 + .5)[None]
        nx, ny, n0, L, ex, ey, e0, c0 = self._view(a)
        w = L / (nx * x + ny * y + n0)
        at = w * (ex * x + ey * y + e0) + c0 - 0.5
        lo = at.floor()
        f, i = at - lo, lo.long()
        row = F.pad(row, (2, 2))
        i = i.clamp(-2, c["cells"]) + 2
        return w ** self.p * (row[:, i] * (1 - f) + row[:, i + 1] * f)

    def back(self, p):
        out = torch.zeros(len(p), self.c["ny"], self.c["nx"], dtype=torch.float64, device=DEV)
        for a in range(self.c["angles"]):
            out += self._back_one(p[:, a], a)
        return out

    def back_transposed(self, v):
        row = torch.zeros(len(v), self.c["cells"], dtype=torch.float64, device=DEV)
        return torch.stack([_transposed(lambda r: self._back_one(r, a), row, v)
                            for a in range(self.c["angles"])], 1)

    def filtered(self, p):
        """Cosine weight, band-limited ramp, scale: (B, A, D)."""
        c = self.c
        dso, dsd = _fan_distances(c)
        u = torch.arange(c["cells"], dtype=torch.float64, device=DEV) - (c["cells"] - 1) / 2
        return _ramp(p * (dsd / torch.sqrt(dsd * dsd + u * u))) * \
            (math.pi / c["angles"] * dso / dsd)


def _ramp(p):
    D = p.shape[-1]
    L = 2 * D
    k = torch.arange(L, dtype=torch.float64, device=p.device)
    k = torch.minimum(k, L - k)
    h = torch.where(k.remainder(2) == 1, -1 / (math.pi * k.clamp_min(1)) ** 2, 0 * k)
    h[0] = 0.25
    return torch.fft.irfft(torch.fft.rfft(p, n=L) * torch.fft.rfft(h), n=L)[..., :D]


class _Cone64:
    """The cone-beam operators in 64 bits; fdk: the geometry of the forward with the FDK weight,
    else the backprojection in the reference's frame (in the views' own for a scan given by
    them)."""

    def __init__(self, c, fdk=False):
        self.c, self.fdk = c, fdk
        self.frames = _cone_frames(c).to(DEV)

    def forward(self, x):
        ones = torch.ones(self.c["v"] * self.c["u"], dtype=torch.float64, device=DEV)
        return torch.stack([
            _march(x[None], *_cone_rays(self.c, self.frames, a), ones)
            .view(self.c["v"], self.c["u"]) for a in range(self.c["angles"])])

    def adjoint(self, y):
        out = torch.zeros(self.c["nz"], self.c["ny"], self.c["nx"], dtype=torch.float64,
                          device=DEV)
        for a in range(self.c["angles"]):
            s, v, n = _cone_rays(self.c, self.frames, a)
            hit = n > 0
            s, v, n = s[hit], v[hit], n[hit]
            out += _transposed(lambda w: _march(w[None], s, v, n, torch.ones_like(n)), out,
                               y[a].reshape(1, -1)[:, hit])
        return out

    def _back_one(self, panel, a, rows):
        """Backprojection of one panel onto some z slices."""
        c = self.c
        z = torch.arange(c["nz"], dtype=torch.float64, device=DEV)[rows][:, None, None]
        y = torch.arange(c["ny"], dtype=torch.float64, device=DEV)[None, :, None]
        x = torch.arange(c["nx"], dtype=torch.float64, device=DEV)[None, None, :]
        dso, dsd = _cone_distances(c)
        if self.fdk or c["views"]:
            org, du, dv, src = self.frames[a]
            I = torch.linalg.inv(torch.stack([org - src, du, dv], 1)).tolist()
            s = src.tolist()
            t, tu, tv = (r[0] * (x - s[0]) + r[1] * (y - s[1]) + r[2] * (z - s[2]) for r in I)
            u, v = tu / t, tv / t
            w = (dso / (t * dsd)) ** 2 if self.fdk else (t > 0).double()
        else:
            # voxels turned by the angle and moved by source to detector, plane at dso - dsd
            al = float(_cone_angles(c)[a])
            co, si = math.cos(al), math.sin(al)
            X, Y, Z = x - (c["nx"] - 1) / 2, y - (c["ny"] - 1) / 2, z - (c["nz"] - 1) / 2
            px, py, pz = co * X + si * Z, Y, -si * X + co * Z
            t = (dso - dsd + dso) / (pz + dso)
            u, v = px * t + c["u"] // 2 - 0.5, py * t + c["v"] // 2 - 0.5
            w = 1.0
        u, v = u.expand(z.shape[0], c["ny"], c["nx"]), v.expand(z.shape[0], c["ny"], c["nx"])
        return _sample(panel[None, None], torch.stack([u, v], -1).reshape(1, 1, -1, 2)) \
            .view(u.shape) * w

    def _slices(self):
        step = max(1, _CHUNK // (self.c["ny"] * self.c["nx"]))
        for z in range(0, self.c["nz"], step):
            yield slice(z, min(z + step, self.c["nz"]))

    def back(self, p):
        out = torch.zeros(self.c["nz"], self.c["ny"], self.c["nx"], dtype=torch.float64,
                          device=DEV)
        for a in range(self.c["angles"]):
            for r in self._slices():
                out[r] += self._back_one(p[a].double(), a, r)
        return out

    def back_transposed(self, v):
        out = torch.zeros(self.c["angles"], self.c["v"], self.c["u"], dtype=torch.float64,
                          device=DEV)
        for a in range(self.c["angles"]):
            for r in self._slices():
                out[a] += _transposed(lambda q: self._back_one(q, a, r), out[a], v[r])
        return out

    def filtered(self, p):
        c = self.c
        dso, dsd = _cone_distances(c)
        u = torch.arange(c["u"], dtype=torch.float64, device=DEV) - (c["u"] - 1) / 2
        v = torch.arange(c["v"], dtype=torch.float64, device=DEV) - (c["v"] - 1) / 2
        w = dsd / torch.sqrt(dsd * dsd + (v * v)[:, None] + u * u)
        return torch.stack([_ramp(q.double() * w) for q in p]) * \
            (math.pi / c["angles"] * dsd / dso)


def exact(case, seed):
    op = case["op"]
    with torch.no_grad():
        s = _inputs(case, seed)
        if op == "serve":
            return [_reconstructed(j, p) for j, p in zip(_serve_cases(case), s["jobs"])]
        if op in ("fan_fbp", "cone_fdk"):
            return _reconstructed(case, s["p"])
        fan = op.startswith("fan")
        A = _Fan64(case) if fan else _Cone64(case)
        many = fan and case["batch"] == 1 and not op.endswith("_layer")
        s = {k: v.double()[None] if many else v.double() for k, v in s.items()}
        if op.endswith("_project"):
            out = {"sino": A.forward(s["x"]), "back": A.back(s["p"])}
        elif op.endswith("_train"):
            q = A.forward(s["x"])
            # the residual and its gradient as a program has them: of the stored projections
            q = q.to(DTYPES[case["dtype"]]).double() if case["dtype"] != "f32" else q
            r = q - s["p"]
            out = {"sino": q, "loss": (r * r).sum()}
            if case["dtype"] == "f32":
                out["grad"] = A.adjoint(2 * r)
            else:
                out = {"sino": q, "loss": None, "grad": None}
        else:
            out = {"volume": A.back(s["p"]), "grad": A.back_transposed(s["g"])}
        if many:
            out = {k: v[0] if v is not None and v.dim() else v for k, v in out.items()}
        return out


def _reconstructed(c, p):
    if c["op"] == "fan_fbp":
        A = _Fan64(c, weighting=2)
        return A.back(A.filtered(p[None].double()))[0]
    A = _Cone64(c, fdk=True)
    return A.back(A.filtered(p))
