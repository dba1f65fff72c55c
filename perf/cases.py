"""The work a program has this library do, as cases that can be timed and
compared: ray batches, rendered frames, batched jobs, a differentiable render
with its gradients, and the denoise and post-processing of a finished frame.

A case is a dict of plain values.  `listed()` names the representative ones,
`draw(rng)` gives more of the same ranges, `prepare(case, seed)` makes what a
program holds before the call (scene, rays, frame buffers), `run(state)` is one
pass through the public entry points, and `exact(case, seed)` states the result
in 64 bits with plain torch where that is feasible.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

import raym0nade_amd as rm
from raym0nade_amd._lib import (RM_BUF_BASE_COLOR, RM_BUF_DD, RM_BUF_DS, RM_BUF_EMISSION, RM_BUF_ID, RM_BUF_IS,
                                RM_BUF_MATERIAL, RM_BUF_PIXELS, RM_BUF_POSITION, RM_BUF_SHAPE_NORMAL,
                                RM_BUF_SURFACE_NORMAL, RM_SHADE_FULL, check, lib)
from raym0nade_amd.diff import DiffRenderer
from raym0nade_amd.workloads import JobSpec, build_job

BLOOM, FXAA, DOF = 256, 512, 1024
RADIANCE = (RM_BUF_DD, RM_BUF_DS, RM_BUF_ID, RM_BUF_IS)
T_MIN = 1e-4


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # picking or a probe: a few hundred rays of one screen tile on a small model; latency and launches count
        dict(name="closest_tile", kind="trace", op="closest", rays="camera", w=33, h=31, scene="spheres", grid=2, freq=20),
        # a light-probe bake or a simulation's ray queries: an odd number of incoherent rays, a mid-sized model
        dict(name="closest_uniform_100k", kind="trace", op="closest", rays="uniform", n=100003, scene="soup", tris=200000),
        # camera rays of a 2828 x 2828 image against a million triangles (the benchmark's coherent batch)
        dict(name="closest_camera_8m", kind="trace", op="closest", rays="camera", w=2828, h=2828, scene="soup", tris=1000000),
        # 8M incoherent rays against a million triangles (the benchmark's incoherent batch)
        dict(name="closest_uniform_8m", kind="trace", op="closest", rays="uniform", n=8000000, scene="soup", tris=1000000),
        # visibility queries with a distance per ray (ambient occlusion, line of sight)
        dict(name="any_uniform_1m", kind="trace", op="any", rays="uniform", n=1000003, scene="soup", tris=1000000),
        # an interactive preview: a small, ragged frame of the box scene at few samples
        dict(name="render_preview", kind="render", scene="cornell", w=161, h=119, spp=4, depth=8, post=RM_SHADE_FULL),
        # the box scene as the reference's plain path tracer renders it: 512 x 512, 64 samples, depth 8
        dict(name="render_cornell_512", kind="render", scene="cornell", w=512, h=512, spp=64, depth=8, post=RM_SHADE_FULL),
        # a 1080p frame of 2M triangles under an HDR sky (diffuse, metal and glass), depth 16, with FXAA
        dict(name="render_spheres_1080p", kind="render", scene="spheres", grid=8, freq=40, w=1920, h=1080, spp=16, depth=16,
             post=RM_SHADE_FULL | FXAA),
        # serving: independent jobs of uneven scene, resolution and sample count in one graph launch
        dict(name="batch_12", kind="batch", jobs=12, mix=3, max_log2=8.5),
        # one inverse-rendering step: forward render, then gradients of texels, roughness and emission
        dict(name="adjoint_512", kind="adjoint", w=512, h=512, spp=32, tex=256),
        # denoising a noisy 1080p frame: firefly clamp, the five a-trous passes, tone curve
        dict(name="denoise_1080p", kind="denoise", w=1920, h=1080, post=RM_SHADE_FULL),
        # the final export of a 1080p frame: depth of field, bloom, tone curve
        dict(name="post_dof_bloom_1080p", kind="post", w=1920, h=1080, post=RM_SHADE_FULL | BLOOM | DOF, coc=8.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest"] * 4 + ["any"] * 2 + ["render"] * 4 + ["batch", "adjoint", "denoise", "post"])
    if kind in ("closest", "any"):
        c = dict(kind="trace", op=kind)
        if rng.random() < 0.5:
            c.update(scene="soup", tris=_log(rng, 2000, 1000000))
        else:
            c.update(scene="spheres", grid=rng.randint(1, 8), freq=rng.randint(5, 40))
        if rng.random() < (0.4 if kind == "closest" else 0.2):
            w = _log(rng, 32, 2828)
            c.update(rays="camera", w=w, h=max(16, int(w * rng.uniform(0.5, 1.0))))
        else:
            c.update(rays="uniform", n=_log(rng, 1000, 8000000))
        return c
    if kind == "render":
        w = _log(rng, 96, 1920)
        h = max(48, int(w * rng.uniform(0.5, 1.0) * (0.5625 if w > 1080 else 1.0)))
        spp = min(_log(rng, 4, 64), max(4, 33177600 // (w * h)))
        c = dict(kind="render", w=w, h=h, spp=spp, depth=rng.randint(4, 16), post=RM_SHADE_FULL | rng.choice([0, FXAA, BLOOM]))
        if rng.random() < 0.4:
            c.update(scene="cornell")
        else:
            c.update(scene="spheres", grid=rng.randint(1, 8), freq=rng.randint(5, 40))
        return c
    if kind == "batch":
        return dict(kind="batch", jobs=rng.randint(2, 14), mix=rng.randint(1, 10 ** 6), max_log2=rng.uniform(7.2, 8.5))
    if kind == "adjoint":
        w = _log(rng, 64, 512)
        return dict(kind="adjoint", w=w, h=max(48, int(w * rng.uniform(0.6, 1.0))), spp=_log(rng, 4, 32), tex=rng.choice([64, 128, 200, 256]))
    w = _log(rng, 96, 1920)
    h = max(64, int(w * rng.uniform(0.4, 0.5625 if w > 1400 else 1.0)))
    if kind == "denoise":
        return dict(kind="denoise", w=w, h=h, post=RM_SHADE_FULL | rng.choice([0, BLOOM]))
    post = rng.choice([BLOOM, FXAA, BLOOM | FXAA, DOF, DOF | BLOOM])
    return dict(kind="post", w=w, h=h, post=RM_SHADE_FULL | post, coc=rng.uniform(1.0, 8.0))


# -------------------------------------------------------------------- scenes
def _n_tris(case):
    if case.get("scene") == "soup":
        return case["tris"]
    if case.get("scene") == "spheres":
        return 20 * case["freq"] ** 2 * case["grid"] ** 2 + 2
    return 36


def _generate(case, seed):
    seed = seed % (1 << 30) + 1
    if case["scene"] == "soup":
        return rm.generate(1, seed, n_tris=case["tris"])
    if case["scene"] == "spheres":
        return rm.generate(2, seed, grid=case["grid"], freq=case["freq"], sky_width=512, sky_height=256)
    return rm.generate(0, seed)


def _args(g, case, seed):
    """The scene's own camera at this case's size, keeping its field of view."""
    a = rm.RmRenderArgs.from_buffer_copy(g.args)
    a.accuracy = float(np.float32(a.accuracy * a.width / case["w"]))
    a.width, a.height = case["w"], case["h"]
    a.seed = seed % (1 << 30) + 1
    return a


def _rays(case, g, seed):
    """[n, 6] float32 rays on the GPU: a pinhole camera's, row by row, or origins uniform in the scene's box with
    directions uniform on the sphere."""
    dev = "cuda"
    r = torch.Generator(device=dev)
    r.manual_seed(seed * 7 + 1)
    if case["rays"] == "camera":
        a = _args(g, case, seed)
        v = [torch.tensor(list(x), device=dev, dtype=torch.float32) for x in (a.position, a.direction, a.right, a.up)]
        # a camera moved a little from seed to seed
        pos = v[0] + 0.02 * torch.randn(3, generator=r, device=dev)
        x = torch.arange(case["w"], device=dev, dtype=torch.float32) - case["w"] / 2
        y = torch.arange(case["h"], device=dev, dtype=torch.float32) - case["h"] / 2
        d = v[1] + a.accuracy * (x[None, :, None] * v[2] + y[:, None, None] * v[3])
        d = (d / d.norm(dim=-1, keepdim=True)).reshape(-1, 3)
        return torch.cat([pos.expand_as(d), d], 1).contiguous()
    n = case["n"]
    u = torch.rand(n, 3, generator=r, device=dev)
    if case["scene"] != "soup":
        lo, hi = g.verts[:-2].min((0, 1)), g.verts[:-2].max((0, 1))  # the spheres; the last two are the ground
        u = torch.tensor(lo, device=dev) + u * torch.tensor(hi - lo, device=dev)
    d = torch.randn(n, 3, generator=r, device=dev)
    return torch.cat([u, d / d.norm(dim=-1, keepdim=True)], 1).contiguous()


def _aims(case, n, seed):
    r = torch.Generator(device="cuda")
    r.manual_seed(seed * 7 + 2)
    far = 0.5 if case["scene"] == "soup" else 4.0
    return torch.rand(n, generator=r, device="cuda") * far + 0.01 * far


# -------------------------------------------------------------------- frames
class _Plane:
    """A frame buffer as an array torch can wrap without a copy."""

    def __init__(self, frame, which):
        p = C.c_void_p()
        check(lib().rm_frame_buffer(frame._h, which, C.byref(p)))
        ch = rm.Frame.CHANNELS[which]
        self.frame = frame
        self.__cuda_array_interface__ = {"shape": (frame.height, frame.width, ch), "typestr": "<f4",
                                         "data": (p.value, False), "version": 2, "strides": None}


def _plane(frame, which):
    return torch.as_tensor(_Plane(frame, which), device="cuda")


def _gbuffer(case, seed):
    """A frame as a renderer leaves it at a few samples per pixel: spheres on a ground plane under a sky, noisy radiance
    with some fireflies, NaN geometry where the camera ray missed."""
    dev, w, h = "cuda", case["w"], case["h"]
    r = torch.Generator(device=dev)
    r.manual_seed(seed * 7 + 3)
    rnd = lambda *s: torch.rand(*s, generator=r, device=dev)  # noqa: E731
    k = 24
    cen = torch.stack([rnd(k) * 8 - 4, rnd(k) * 2 - 0.8, rnd(k) * 9 + 3], 1)
    rad = rnd(k) * 0.5 + 0.2
    x = (torch.arange(w, device=dev) - w / 2) / w
    y = (h / 2 - torch.arange(h, device=dev)) / w
    d = torch.stack([x[None, :].expand(h, w), y[:, None].expand(h, w), torch.full((h, w), 0.8, device=dev)], -1)
    d = d / d.norm(dim=-1, keepdim=True)
    t = torch.where(d[..., 1] < -1e-3, -1.0 / d[..., 1].clamp(max=-1e-3), torch.tensor(math.inf, device=dev))  # ground y = -1
    obj = torch.where(torch.isfinite(t), torch.zeros_like(t), torch.full_like(t, -1)).long()
    for i in range(k):
        b = (d * cen[i]).sum(-1)
        disc = b * b - (cen[i] * cen[i]).sum() + rad[i] ** 2
        ti = b - disc.clamp(min=0).sqrt()
        hit = (disc > 0) & (ti > 0.1) & (ti < t)
        t = torch.where(hit, ti, t)
        obj = torch.where(hit, torch.full_like(obj, i + 1), obj)
    t = torch.where(t > 60, torch.tensor(math.inf, device=dev), t)  # the ground's horizon belongs to the sky
    miss = ~torch.isfinite(t)
    obj = torch.where(miss, torch.full_like(obj, -1), obj)
    o = obj.clamp(min=0)
    pos = d * torch.where(miss, torch.zeros_like(t), t)[..., None]
    cen1 = torch.cat([torch.zeros(1, 3, device=dev), cen])
    n = pos - cen1[o]
    n = torch.where((o == 0)[..., None], torch.tensor([0.0, 1.0, 0.0], device=dev), n)
    n = n / n.norm(dim=-1, keepdim=True).clamp(min=1e-6)
    bump = 0.01 * torch.stack([torch.sin(9 * pos[..., 0]), torch.sin(7 * pos[..., 1]), torch.sin(8 * pos[..., 2])], -1)
    sn = n + bump
    sn = sn / sn.norm(dim=-1, keepdim=True)
    base = (rnd(k + 1, 3) * 0.6 + 0.2)[o]
    mat = torch.stack([(rnd(k + 1) < 0.3).float() * 0.95, rnd(k + 1) * 0.75 + 0.05, (rnd(k + 1) < 0.85).float()], 1)[o]
    emis = torch.where((rnd(k + 1) < 0.1)[o][..., None], torch.tensor([6.0, 5.0, 3.5], device=dev), torch.zeros(3, device=dev))
    nan = torch.tensor(math.nan, device=dev)
    m3 = miss[..., None]
    out = {
        RM_BUF_POSITION: torch.where(m3, nan, pos), RM_BUF_SHAPE_NORMAL: torch.where(m3, nan, n),
        RM_BUF_SURFACE_NORMAL: torch.where(m3, nan, sn), RM_BUF_BASE_COLOR: torch.where(m3, torch.zeros_like(base), base),
        RM_BUF_EMISSION: torch.where(m3, torch.tensor([0.5, 0.7, 1.1], device=dev) * (1 + d[..., 1:2]), emis),
        RM_BUF_MATERIAL: torch.where(m3, torch.tensor([0.0, 0.8, 1.0], device=dev), mat),
    }
    lit = (sn * torch.tensor([0.4, 0.8, -0.45], device=dev)).sum(-1).clamp(min=0.02)
    for which, level, spp in ((RM_BUF_DD, 1.2, 12), (RM_BUF_DS, 0.25, 12), (RM_BUF_ID, 0.35, 5), (RM_BUF_IS, 0.1, 5)):
        mean = level * lit[..., None] * (rnd(3) * 0.4 + 0.8)
        # the mean of `spp` exponential samples
        noise = torch.stack([-torch.log(rnd(h, w).clamp(min=1e-7)) for _ in range(spp)])
        m, var = noise.mean(0), noise.var(0) / spp
        m = m * torch.where(rnd(h, w) < 2e-4, torch.tensor(250.0, device=dev), torch.tensor(1.0, device=dev))
        q = torch.cat([mean * m[..., None], ((mean ** 2).sum(-1) * var)[..., None]], -1)
        out[which] = torch.where(m3, torch.zeros_like(q), q)
    return {b: v.contiguous() for b, v in out.items()}


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "trace":
        g = _generate(case, seed)
        rays = _rays(case, g, seed)
        return dict(kind=kind, op=case["op"], scene=rm.Scene(g), rays=rays,
                    aim=_aims(case, rays.shape[0], seed) if case["op"] == "any" else None)
    if kind == "render":
        g = _generate(case, seed)
        a = _args(g, case, seed)
        a.spp, a.max_depth = case["spp"], case["depth"]
        f = rm.Frame(case["w"], case["h"])
        return dict(kind=kind, scene=rm.Scene(g), args=a, frame=f, post=case["post"],
                    out={b: _plane(f, b) for b in RADIANCE + (RM_BUF_PIXELS,)})
    if kind == "batch":
        jobs, outs = [], []
        for i, s in enumerate(_specs(case)):
            s.scene_seed = (seed * 31 + i) % (1 << 30) + 1
            g, scene, a = build_job(s, sky=(256, 128))
            f = rm.Frame(s.side, s.side)
            jobs.append((scene, a, f, RM_SHADE_FULL | FXAA))
            outs.append([_plane(f, RM_BUF_ID), _plane(f, RM_BUF_PIXELS)])
        return dict(kind=kind, jobs=jobs, out=outs)
    if kind == "adjoint":
        g = rm.generate(4, seed % (1 << 30) + 1, tex_size=case["tex"])
        a = _args(g, case, seed)
        a.spp = case["spp"]
        R = DiffRenderer(g, a)
        params = [p.requires_grad_() for p in R.initial_params()]
        r = torch.Generator(device="cuda")
        r.manual_seed(seed * 7 + 4)
        # d loss / d image of an L2 loss: a residual of either sign
        d_img = torch.randn(case["h"], case["w"], 3, generator=r, device="cuda") * 0.1
        return dict(kind=kind, R=R, params=params, d_img=d_img)
    planes = _gbuffer(case, seed)
    f = rm.Frame(case["w"], case["h"])
    views = {b: _plane(f, b) for b in planes}
    for b, v in planes.items():
        views[b].copy_(v)
    noisy = {b: planes[b] for b in RADIANCE}
    if kind == "post":
        f.set_dof(6.0, case["coc"], (0.0, 0.0, 0.0))
    return dict(kind=kind, frame=f, views=views, noisy=noisy, post=case["post"], image=_plane(f, RM_BUF_PIXELS))


def _specs(case):
    r = random.Random(case["mix"])
    out = []
    for i in range(case["jobs"]):
        side = int(round(2.0 ** r.uniform(7.0, case["max_log2"])))
        spp, depth = r.choice([16, 64]), r.randint(8, 16)
        if i % 2 == 0:
            out.append(JobSpec(0, 0, 0, 0, side, spp, depth))
        else:
            out.append(JobSpec(2, 0, r.randint(1, 4), r.randint(4, 24), side, spp, depth))
    return out


# ----------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    if kind == "trace":
        if state["op"] == "closest":
            t, ids = state["scene"].trace_closest(state["rays"])
            return {"t": t, "id": ids}
        return {"occluded": state["scene"].trace_any(state["rays"], aim_dev=state["aim"])}
    if kind == "render":
        f = state["frame"]
        f.render(state["scene"], state["args"])
        f.postprocess(state["post"], state["args"].exposure)
        return state["out"]
    if kind == "batch":
        rm.render_batch(state["jobs"])
        return state["out"]
    if kind == "adjoint":
        img = state["R"].render(*state["params"])
        grads = torch.autograd.grad(img, state["params"], state["d_img"])
        return {"image": img.detach(), "texels": grads[0], "roughness": grads[1], "emission": grads[2]}
    f = state["frame"]
    if kind == "denoise":
        # the denoiser works in place: a new frame's radiance arrives first
        for b in RADIANCE:
            state["views"][b].copy_(state["noisy"][b])
        f.spatial_clamp()
        f.filter()
        f.postprocess(state["post"])
        return {"image": state["image"], **{str(b): state["views"][b] for b in RADIANCE}}
    f.postprocess(state["post"])
    return {"image": state["image"]}


# ---------------------------------------------------------------------- work
def _walk_flops(tris):
    """One root-to-leaf descent: two box tests a level, one leaf of about eight triangles."""
    return 2 * 24 * max(1, math.ceil(math.log2(max(2, tris / 8)))) + 8 * 46


def _scene_bytes(tris):
    return tris * 48 + tris / 8 * 64


def work(case):
    kind = case["kind"]
    if kind == "trace":
        n = case["n"] if case["rays"] == "uniform" else case["w"] * case["h"]
        out = 8 if case["op"] == "closest" else 1 + 4
        tris = _n_tris(case)
        return dict(bytes=n * (24 + out) + _scene_bytes(tris), flops=n * _walk_flops(tris))
    if kind in ("render", "adjoint"):
        px, tris = case["w"] * case["h"], _n_tris(case)
        # 0.7 spp light samples of one walk each, 0.3 spp paths of about three vertices with light samples
        walks = px * (1 + case["spp"] * (0.7 + 0.3 * 4))
        fl = walks * (_walk_flops(tris) + 200)
        by = px * 148 + _scene_bytes(tris)
        if kind == "adjoint":
            return dict(bytes=by + px * 24 + 2 * 5 * case["tex"] ** 2 * 12, flops=2.5 * fl)
        return dict(bytes=by, flops=fl)
    if kind == "batch":
        by = fl = 0.0
        for s in _specs(case):
            tris = 36 if s.config == 0 else 20 * s.freq ** 2 * s.grid ** 2 + 2
            px = s.side * s.side
            by += px * 148 + _scene_bytes(tris)
            fl += px * (1 + s.spp * 1.9) * (_walk_flops(tris) + 200)
        return dict(bytes=by, flops=fl)
    px = case["w"] * case["h"]
    if kind == "denoise":
        # radiance and G-buffer in, radiance and image out; 24 taps x 5 passes of weights and four sums
        return dict(bytes=px * (64 + 64 + 48 + 24 + 12), flops=px * 5 * 24 * 90.0)
    fl = 60.0
    if case["post"] & BLOOM:
        fl += 5 * 10 * 6
    if case["post"] & DOF:
        fl += 20 * math.pi * case["coc"] ** 2 / 3
    return dict(bytes=px * (64 + 24 + 12 + (12 if case["post"] & DOF else 0)), flops=px * fl)


def tolerance(case):
    kind = case["kind"]
    if kind == "trace":
        return "exact"  # the traversal is pinned: ids, distances and occlusion bits
    if kind in ("render", "batch"):
        # the sample sums in another order (1, 3, 5 or 16 accumulator sets a pixel) differ by 1.2e-7, one pixel by 1.4e-4
        return {"rel": 1e-6, "max": 1e-3}
    if kind == "adjoint":
        # texel gradients are sums of float atomics: two runs differ by 1.1e-6
        return {"rel": 5e-6, "max": 1e-3}
    if kind == "denoise":
        # against 64 bits the planes are 1.3e-6 off; a tap at the weight's cut-off may fall to either side of it
        return {"rel": 5e-6, "max": 2e-3}
    return {"rel": 1e-6, "max": 1e-4}  # 1.4e-7 off 64 bits


# --------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "trace":
        return _exact_trace(case, seed)
    if kind == "denoise":
        return _exact_denoise(case, seed)
    if kind == "post" and not case["post"] & (DOF | FXAA):
        return {"image": _finish64({b: v.double() for b, v in _gbuffer(case, seed).items()}, case["post"])}
    return None  # Monte Carlo renders, their gradients, and the image passes that branch on their own values


def _exact_trace(case, seed):
    """Every ray against every triangle (Moeller-Trumbore as matrix products), with the reference's rejection of
    grazing triangles, |a| < 1e-4 |e1|."""
    n = case["n"] if case["rays"] == "uniform" else case["w"] * case["h"]
    if n * _n_tris(case) > 2.5e10:
        return None
    g = _generate(case, seed)
    rays = _rays(case, g, seed).double()
    v = torch.from_numpy(np.ascontiguousarray(g.verts)).cuda().double()
    v0, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    nrm = torch.cross(e1, e2, dim=1)
    A = nrm.t().contiguous()
    U = torch.cat([e2, -torch.cross(e2, v0, dim=1)], 1).t().contiguous()
    V = torch.cat([-e1, torch.cross(e1, v0, dim=1)], 1).t().contiguous()
    c = (v0 * nrm).sum(1)
    thr = 1e-4 * e1.norm(dim=1)
    aim = _aims(case, n, seed).double() if case["op"] == "any" else None
    ts, ids = [], []
    step = max(1, int(6e7 // v.shape[0]))
    inf = torch.tensor(math.inf, device="cuda", dtype=torch.float64)
    for i in range(0, n, step):
        o, d = rays[i:i + step, :3], rays[i:i + step, 3:]
        m = torch.cat([torch.cross(o, d, dim=1), d], 1)
        a = -(d @ A)
        t = (o @ A - c) / a
        ok = a.abs() >= thr
        p = (m @ U) / a
        ok &= (p >= 0) & (p <= 1)
        q = (m @ V) / a
        ok &= (q >= 0) & (p + q <= 1) & (t > T_MIN)
        tm, im = torch.where(ok, t, inf).min(1)
        ts.append(tm)
        ids.append(torch.where(torch.isfinite(tm), im, torch.full_like(im, -1)))
    t = torch.cat(ts)
    if case["op"] == "any":
        return {"occluded": (t < aim).to(torch.uint8)}
    return {"t": t, "id": torch.cat(ids).int()}


def _shift(x, dy, dx):
    """x at (y + dy, x + dx), zero outside."""
    h, w = x.shape[:2]
    out = torch.zeros_like(x)
    if abs(dy) < h and abs(dx) < w:
        out[max(0, -dy):h - max(0, dy), max(0, -dx):w - max(0, dx)] = \
            x[max(0, dy):h - max(0, -dy), max(0, dx):w - max(0, -dx)]
    return out


def _lum(x):
    return 0.3 * x[..., 0] + 0.6 * x[..., 1] + 0.1 * x[..., 2]


def _finish64(p, post):
    """Shading, bloom and the tone curve."""
    img = p[RM_BUF_BASE_COLOR] * (p[RM_BUF_DD] + p[RM_BUF_ID])[..., :3] + (p[RM_BUF_DS] + p[RM_BUF_IS])[..., :3] \
        + p[RM_BUF_EMISSION]
    h5 = (0.0625, 0.25, 0.375, 0.25, 0.0625)
    if post & BLOOM:
        c = _lum(img)[..., None]
        lvl = torch.where(c < 1, torch.zeros_like(img), (img / c.clamp(min=1e-9) ** 0.65 - 1).clamp(min=0))
        for s in (1, 2, 4, 8, 16):
            rows = sum(h5[k + 2] * _shift(lvl, k * s, 0) for k in range(-2, 3))
            lvl = sum(h5[k + 2] * _shift(rows, 0, k * s) for k in range(-2, 3))
            img = img + lvl / 6
    img = img.clamp(min=0)
    c = _lum(img)[..., None]
    soft = img / c.clamp(min=1e-9) * (torch.tanh(3 * (c - 0.75)) / 3 + 0.75)
    return torch.where(c > 0.75, soft, img).clamp(max=1) ** (1 / 2.2)


def _exact_denoise(case, seed):
    p = {b: v.double() for b, v in _gbuffer(case, seed).items()}
    pos, sn, un, mat = (p[b] for b in (RM_BUF_POSITION, RM_BUF_SHAPE_NORMAL, RM_BUF_SURFACE_NORMAL, RM_BUF_MATERIAL))
    seen = torch.isfinite(pos).any(-1)
    h7 = (0.03125, 0.109375, 0.21875, 0.28125, 0.21875, 0.109375, 0.03125)
    h5 = (0.0625, 0.25, 0.375, 0.25, 0.0625)
    h3 = (0.25, 0.5, 0.25)
    ones = torch.ones_like(seen, dtype=torch.float64)
    for b in RADIANCE:
        q = p[b]
        l = _lum(q)
        rows = sum(h7[k + 3] * _shift(l, 0, k) for k in range(-3, 4))
        blur = sum(h7[k + 3] * _shift(rows, k, 0) for k in range(-3, 4)) - h7[3] ** 2 * l
        s = torch.where(l > 36 * blur, blur / (l + 1e-4) / (1 - h7[3] ** 2), ones)
        q = torch.cat([q[..., :3] * s[..., None], q[..., 3:]], -1)
        m = torch.cat([q[..., :3], q[..., 3:], (q[..., :3] ** 2).sum(-1, keepdim=True)], -1)
        e = sum(h3[i + 1] * h3[j + 1] * _shift(m, i, j) for i in (-1, 0, 1) for j in (-1, 0, 1))
        p[b] = torch.cat([q[..., :3], e[..., 3:4] + e[..., 4:] - (e[..., :3] ** 2).sum(-1, keepdim=True)], -1)
    rough = mat[..., 1].clamp(min=0.04)
    for step in (1, 2, 4, 8, 16):
        acc = {b: torch.zeros_like(p[b]) for b in RADIANCE}
        ws = {b: torch.zeros_like(ones) for b in RADIANCE}
        for dy in range(-2, 3):
            for dx in range(-2, 3):
                sy, sx = dy * step, dx * step
                inside = _shift(ones, sy, sx)
                tap = h5[dy + 2] * h5[dx + 2] * inside
                if dy or dx:
                    ok = _shift(seen.double(), sy, sx) > 0
                    pw = (un * _shift(un, sy, sx)).sum(-1).clamp(min=0) ** 1024
                    dd = _shift(pos, sy, sx) - pos
                    s = (sn * dd / dd.norm(dim=-1, keepdim=True)).sum(-1).abs()
                    tan = s / ((1 - s * s).sqrt() + 1e-4)
                    dm = mat - _shift(mat, sy, sx)
                    md = (dm[..., 0] ** 2 + dm[..., 2] ** 2).sqrt()
                for b in RADIANCE:
                    q = _shift(p[b], sy, sx)
                    wt = tap
                    if dy or dx:
                        rd = (p[b][..., :3] - q[..., :3]).norm(dim=-1) / (p[b][..., 3].sqrt() + 1e-2)
                        k = -tan - rd - md
                        g = pw * torch.exp(k) * (rough if b in (RM_BUF_DS, RM_BUF_IS) else 1.0)
                        g = torch.where(ok & ~(pw < 1e-6) & ~(k < -7.5) & torch.isfinite(g), g, torch.zeros_like(g))
                        wt = tap * g
                    ws[b] += wt
                    acc[b] += torch.cat([q[..., :3] * wt[..., None], (q[..., 3] * wt * wt)[..., None]], -1)
        for b in RADIANCE:
            a = torch.cat([acc[b][..., :3] / ws[b][..., None], (acc[b][..., 3] / ws[b] ** 2)[..., None]], -1)
            p[b] = torch.where(seen[..., None], a, torch.zeros_like(a))
    return {"image": _finish64(p, case["post"]), **{str(b): p[b] for b in RADIANCE}}
