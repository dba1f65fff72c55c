"""Calls for which the default walk has a slow way out: timed against the walk
of the binary tree (trace variant 3, four triangles a step) at the settings
that suit it, which the default has to come near at least."""
import contextlib
import time

import numpy as np
import pytest
import torch

import raym0nade_amd as rm
from cutout_util import make_desc

pytestmark = pytest.mark.gpu

BINARY = {rm.TUNE_TRIS_PER_STEP: 4, rm.TUNE_FETCH_MIN: 48}


@contextlib.contextmanager
def tuned(values):
    old = {k: rm.get_tuning(k) for k in values}
    try:
        for k, v in values.items():
            rm.set_tuning(k, v)
        yield
    finally:
        for k, v in old.items():
            rm.set_tuning(k, v)


def ms(fn, reps=5):
    """The least of a few runs, after one to warm up."""
    fn()
    best = float("inf")
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        fn()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def holds(limit, measure):
    """Whether the first of two times is below limit times the second, in one
    of four measurements: other work on the machine only ever adds time."""
    seen = []
    for _ in range(4):
        seen.append(measure())
        if seen[-1][0] < limit * seen[-1][1]:
            return
    raise AssertionError(f"{limit}: {seen}")


def both(scene, rays, binary=BINARY, **kw):
    t = torch.empty(rays.shape[0], device=rays.device)
    i = torch.empty(rays.shape[0], device=rays.device, dtype=torch.int32)
    run = lambda: scene.trace_closest(rays, t_out=t, id_out=i, **kw)  # noqa: E731
    own = ms(run)
    with tuned(binary):
        return own, ms(run)


def describe(v):
    v = np.ascontiguousarray(v, np.float32)
    m = rm._lib.RmMaterial(roughness=0.8, opacity=1.0, ior=1.0, albedo_tex=-1, normal_tex=-1, emissive_tex=-1, specular_tex=-1)
    k = len(v)
    return make_desc(v, np.zeros((k, 3, 2)), np.zeros(k), np.zeros(k), [m], [])


def make(v):
    desc, keep = describe(v)
    S = rm.Scene(desc)
    S.arrays = keep
    return S


def soup(n, seed, size):
    r = np.random.default_rng(seed)
    return (r.random((n, 1, 3)) + size * (r.random((n, 3, 3)) - 0.5)).astype(np.float32)


def uniform(n, dev, length=1.0):
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    d = torch.randn(n, 3, generator=g, device=dev)
    return torch.cat([torch.rand(n, 3, generator=g, device=dev), d / d.norm(dim=1, keepdim=True) * length], 1).contiguous()


def test_doubled_triangles(dev):
    """Every hit is one of two at the same distance, some in different leaves."""
    v = soup(100000, 1, 0.015)
    S, r = make(np.concatenate([v, v])), uniform(1 << 20, dev)
    holds(1.2, lambda: both(S, r))


def test_scene_outside_the_trees_range(dev):
    """Far from the origin the binary tree is walked, at its own claim threshold."""
    S = make(soup(500, 2, 0.2) + np.float32(2e4))
    r = uniform(1 << 20, dev)
    r[:, :3] += 2e4
    r = r.contiguous()
    holds(1.15, lambda: both(S, r, {rm.TUNE_FETCH_MIN: 48}))


def test_negative_tmin(dev):
    """Rays that start behind their origin are outside what the four-wide walk proves."""
    S, r = make(soup(5000, 3, 0.05)), uniform(1 << 20, dev)
    holds(1.3, lambda: both(S, r, tmin=-1.0))


@pytest.mark.parametrize("length", [20.0, 300.0])
def test_long_directions(dev, length):
    """Where boxes are grown much, and where rays leave for the reference's order."""
    S, r = make(soup(5000, 3, 0.05)), uniform(1 << 17, dev, length)
    holds(1.4, lambda: both(S, r))


@pytest.mark.parametrize("tris", [2, 12])
def test_one_ray(dev, tris):
    """The smallest call: its launches are all that it costs."""
    S = make(soup(tris, 5, 0.3))
    r = uniform(1, dev)
    t, i = torch.empty(1, device=dev), torch.empty(1, device=dev, dtype=torch.int32)

    def many():
        for _ in range(200):
            S.trace_closest(r, t_out=t, id_out=i)

    def measure():
        own = ms(many)
        with tuned(BINARY):
            return own, ms(many)

    holds(0.95, measure)


def test_scene_creation(dev):
    """A small scene with its four-wide tree, against one whose place excludes that."""
    near = soup(1000, 6, 0.1)
    far = (near + np.float32(2e4)).astype(np.float32)

    def seconds(v):
        desc, keep = describe(v)
        best = float("inf")
        for _ in range(50):
            t0 = time.perf_counter()
            rm.Scene(desc)
            best = min(best, time.perf_counter() - t0)
        return best

    seconds(near)
    holds(1.55, lambda: (seconds(near), seconds(far)))


def camera(side, dev):
    x = (torch.arange(side, device=dev) + 0.5) / side - 0.5
    d = torch.stack([x[None, :].expand(side, side), x[:, None].expand(side, side), torch.full((side, side), 0.8, device=dev)], -1)
    d = (d / d.norm(dim=-1, keepdim=True)).reshape(-1, 3)
    return torch.cat([torch.tensor([0.51, 0.52, -0.5], device=dev).expand_as(d), d], 1).contiguous()


@pytest.mark.parametrize("tris, side", [(200000, 1500), (5000, 2500)])
def test_shuffled_camera(dev, tris, side):
    """Rays of one origin whose directions come in no order are put in one:
    nearly as fast as the image's own order, with the same results."""
    S = make(soup(tris, 4, 0.015 if tris > 10000 else 0.05))
    r = camera(side, dev)
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    p = torch.randperm(r.shape[0], generator=g, device=dev)
    q = r[p].contiguous()
    t, i = S.trace_closest(r)
    ts, js = S.trace_closest(q)
    assert torch.equal(js, i[p]) and torch.equal(ts.view(torch.int32), t[p].view(torch.int32))

    def measure(rays):
        own = ms(lambda: S.trace_closest(rays))
        with tuned({rm.TUNE_RAY_SORT: 0}):
            return own, ms(lambda: S.trace_closest(rays))

    holds(0.95, lambda: measure(q))
    holds(1.1, lambda: measure(r))
