"""The four-wide walk and the flat test of small scenes (trace variant 3 with
whole leaves, the default) against the oracle's BVH::rayHit / Model::rayHit_test: ids, t and
occlusion bit-exact.  Scenes around the sizes where the tree changes (one
leaf, 64 / 65 triangles, slivers far from the origin, odd and even numbers of levels, uneven leaves,
duplicated triangles, axis-aligned walls, large triangles among small ones);
rays aimed at vertices and edges (exact ties and certificates that fail), from
surfaces, along axes exactly and nearly, from far outside, of lengths other
than 1, and with non-finite parts."""
import numpy as np
import pytest
import torch

import oracle_py as O
import raym0nade_amd as rm
from cutout_util import make_desc

pytestmark = pytest.mark.gpu


def soup(n, seed, size=0.1):
    r = np.random.default_rng(seed)
    c = r.random((n, 1, 3), dtype=np.float32)
    return (c + size * (r.random((n, 3, 3), dtype=np.float32) - 0.5)).astype(np.float32)


def walls(n):
    """Axis-aligned quads on a grid: boxes without thickness, edges shared by four triangles."""
    out = []
    for i in range(n):
        for j in range(n):
            for k in range(3):
                a = np.zeros((4, 3), np.float32)
                u, v = [x for x in range(3) if x != k]
                a[:, u] = np.array([i, i + 1, i + 1, i]) / n
                a[:, v] = np.array([j, j, j + 1, j + 1]) / n
                a[:, k] = 0.25 * (1 + (i + j + k) % 3)
                out += [a[[0, 1, 2]], a[[0, 2, 3]]]
    return np.ascontiguousarray(np.stack(out), dtype=np.float32)


def needles(n):
    """Triangles whose first edge's square is below the float range."""
    v = soup(n, 18, 0.6)
    v[:, 0] = 0.0
    v[:, 1] = np.float32([1e-20, 1e-21, 0.0])
    return v


SCENES = {
    "one_leaf": lambda: soup(10, 1, 0.5), "two_leaves": lambda: soup(11, 2, 0.5), "soup20": lambda: soup(20, 3, 0.4),
    "soup21": lambda: soup(21, 4, 0.4), "soup48": lambda: soup(48, 5, 0.3), "soup49": lambda: soup(49, 6, 0.3),
    "soup64": lambda: soup(64, 13, 0.3), "soup65": lambda: soup(65, 14, 0.3),
    "slivers": lambda: (soup(60, 15, 0.8) * np.array([1, 1e-4, 1]) + np.array([90, 40, -7])).astype(np.float32),
    "soup80": lambda: soup(80, 7, 0.3), "soup81": lambda: soup(81, 8, 0.3), "soup1301": lambda: soup(1301, 9),
    "soup7001": lambda: soup(7001, 10, 0.05), "walls": lambda: walls(9),
    "needles3": lambda: np.concatenate([soup(900, 16, 0.2), needles(3)]),
    "needles12": lambda: np.concatenate([soup(900, 17, 0.2), needles(12)]),
    # outside the tree's range: far from the origin, and too large
    "far_off": lambda: (soup(700, 19, 0.2) + np.float32(2e4)).astype(np.float32), "large": lambda: soup(900, 20, 0.2) * np.float32(500),
    "doubled": lambda: np.repeat(soup(700, 11, 0.2), 2, axis=0),
    "twice": lambda: np.concatenate([soup(701, 11, 0.2)] * 2), "thrice": lambda: np.concatenate([soup(501, 11, 0.2)] * 3),
    "twice_flat": lambda: np.concatenate([soup(31, 11, 0.4)] * 2), "thrice_flat": lambda: np.concatenate([soup(21, 11, 0.4)] * 3),
    "ground": lambda: np.concatenate([soup(3000, 12, 0.02) * np.float32(0.2),
                                      np.array([[[-40, 0, -40], [40, 0, -40], [40, 0, 40]],
                                                [[-40, 0, -40], [40, 0, 40], [-40, 0, 40]]], np.float32)]),
}


def rays_for(v, kind, n, seed):
    r = np.random.default_rng(seed)
    lo, hi = v.min((0, 1)), v.max((0, 1))
    o = lo + r.random((n, 3)) * (hi - lo)
    d = r.standard_normal((n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    tri = v[r.integers(0, len(v), n)]
    if kind == "vertices":
        d = tri[np.arange(n), r.integers(0, 3, n)] - o
    elif kind == "edges":
        a = r.random((n, 1))
        d = tri[:, 0] * a + tri[:, 1] * (1 - a) - o
    elif kind == "surface":
        b = r.random((n, 2))
        b = np.where(b.sum(1, keepdims=True) > 1, 1 - b, b)
        o = tri[:, 0] + b[:, :1] * (tri[:, 1] - tri[:, 0]) + b[:, 1:] * (tri[:, 2] - tri[:, 0])
    elif kind == "axis":
        d = np.zeros((n, 3))
        d[np.arange(n), r.integers(0, 3, n)] = np.where(r.random(n) < 0.5, -1.0, 1.0)
        d += np.where(r.random((n, 1)) < 0.5, 0.0, 2.5e-4 * (r.random((n, 3)) - 0.5))
    elif kind == "far":
        o = o - d * (hi - lo).max() * r.random((n, 1)) * 30
    elif kind == "length":
        d *= 10 ** (r.random((n, 1)) * 8 - 4)
    x = np.concatenate([o, d], 1).astype(np.float32)
    if kind == "odd":
        bad = np.array([np.nan, np.inf, -np.inf, 0.0, 1e30, 1e-30], np.float32)
        m = r.random((n, 6)) < 0.2
        x = np.where(m, bad[r.integers(0, 6, (n, 6))], x).astype(np.float32)
    return np.ascontiguousarray(x)


@pytest.mark.parametrize("scene", list(SCENES))
def test_bit_exact(dev, scene):
    v = SCENES[scene]()
    m = rm._lib.RmMaterial(roughness=0.8, opacity=1.0, ior=1.0, albedo_tex=-1, normal_tex=-1, emissive_tex=-1, specular_tex=-1)
    k = len(v)
    desc, keep = make_desc(v, np.zeros((k, 3, 2)), np.zeros(k), np.zeros(k), [m], [])
    S, OS = rm.Scene(desc), O.OracleScene(desc)
    assert rm.get_tuning(rm.TUNE_TRACE_VARIANT) == 3 and rm.get_tuning(rm.TUNE_TRIS_PER_STEP) == 0
    n = 6000
    for kind in ("box", "vertices", "edges", "surface", "axis", "far", "length", "odd"):
        r = rays_for(v, kind, n, 17)
        rd = torch.from_numpy(r).to(dev)
        for tmin, tmax in ((1e-4, np.inf), (0.05, 0.7), (-0.5, np.inf)) if kind != "odd" else ((1e-4, np.inf),):
            t, ids = S.trace_closest(rd, tmin=tmin, tmax=tmax)
            to, io = OS.closest(r, tmin=tmin, tmax=tmax)
            assert np.array_equal(ids.cpu().numpy(), io), (scene, kind, tmin)
            assert np.array_equal(t.cpu().numpy().view(np.uint32), to.view(np.uint32)), (scene, kind, tmin)
        # distances around the closest hit, some exactly at it
        to, io = OS.closest(r)
        g = np.random.default_rng(5)
        aim = np.where(np.isfinite(to), to, 1.0) * np.where(g.random(n) < 0.3, 1.0, 0.6 + 0.8 * g.random(n))
        aim = aim.astype(np.float32)
        occ = S.trace_any(rd, aim_dev=torch.from_numpy(aim).to(dev))
        assert np.array_equal(occ.cpu().numpy(), OS.any(r, aims=aim)), (scene, kind)


def mixed(n, n_big, ext, small, big, seed):
    """n triangles over ext units, n_big of them large and tilted."""
    r = np.random.default_rng(seed)
    c = r.random((n, 1, 3)) * ext
    v = c + small * np.exp(r.normal(0, 0.7, (n, 1, 1))) * (r.random((n, 3, 3)) - 0.5)
    i = r.permutation(n)[:n_big]
    v[i] = c[i] + big * (r.random((n_big, 3, 3)) - 0.5)
    return v.astype(np.float32), i


def grazing(v, idx, n, length, dev, seed):
    """Rays nearly in the plane of a large triangle, n.d between 0.8e-4 and
    1.6e-3 |e1| (tests reject below 1e-4 |e1|), aimed at points in it and a
    little outside: computed t, u and v are least accurate there."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rnd = lambda *s: torch.rand(*s, generator=g, device=dev, dtype=torch.float64)  # noqa: E731
    T = torch.tensor(v[idx], device=dev, dtype=torch.float64)[torch.randint(0, len(idx), (n,), generator=g, device=dev)]
    e1, e2 = T[:, 1] - T[:, 0], T[:, 2] - T[:, 0]
    m = torch.cross(e1, e2, dim=1)
    l, l1 = m.norm(dim=1, keepdim=True), e1.norm(dim=1, keepdim=True)
    x, a = e1 / l1, rnd(n, 1) * 6.2832
    k = 0.8e-4 * 20.0 ** rnd(n, 1) * l1 / l
    d = length * (x * torch.cos(a) + torch.cross(m / l, x, dim=1) * torch.sin(a)) + m / l * torch.where(rnd(n, 1) < 0.5, -k, k)
    b = rnd(n, 2)
    b = torch.where(b.sum(1, keepdim=True) > 1, 1 - b, b) * 1.1 - 0.05
    o = T[:, 0] + b[:, :1] * e1 + b[:, 1:] * e2 - d / d.norm(dim=1, keepdim=True) * rnd(n, 1) * float(np.ptp(v))
    return torch.cat([o, d], 1).float().contiguous()


# small and large scenes, some in and some outside the tree's range of sizes,
# and long directions, whose computed distances err as in a larger scene
@pytest.mark.parametrize("n, n_big, ext, small, big", [
    (200, 20, 20, 1, 8), (200, 20, 300, 20, 200), (200, 200, 25, 15, 15), (2000, 50, 25, 0.5, 15), (2000, 50, 100, 2, 70),
    (2000, 50, 1000, 20, 700), (2000, 4, 25, 0.5, 20), (50000, 100, 10, 0.05, 5)])
def test_grazing(dev, n, n_big, ext, small, big):
    """Rays for which a triangle's computed t can lie before its own box."""
    for seed in range(3):
        v, idx = mixed(n, n_big, ext, small, big, seed)
        k = len(v)
        m = rm._lib.RmMaterial(roughness=0.8, opacity=1.0, ior=1.0, albedo_tex=-1, normal_tex=-1, emissive_tex=-1, specular_tex=-1)
        desc, keep = make_desc(v, np.zeros((k, 3, 2)), np.zeros(k), np.zeros(k), [m], [])
        S, OS = rm.Scene(desc), O.OracleScene(desc)
        for length in (1.0, 10.0, 60.0, 400.0):
            r = grazing(v, idx, 1 << 20, length, dev, seed)
            aim = 0.5 * ext / length
            t, ids = S.trace_closest(r)
            occ = S.trace_any(r, aim=aim)
            try:
                rm.set_tuning(rm.TUNE_TRACE_VARIANT, 0)
                t0, i0 = S.trace_closest(r)
                occ0 = S.trace_any(r, aim=aim)
                torch.cuda.synchronize()
            finally:
                rm.set_tuning(rm.TUNE_TRACE_VARIANT, 3)
            bad = (ids != i0) | (t.view(torch.int32) != t0.view(torch.int32)) | (occ != occ0)
            assert not bool(bad.any()), (seed, length, int(bad.sum()))
            # the walk compared with, against the oracle
            few = r[:2000].cpu().numpy()
            to, io = OS.closest(few)
            assert np.array_equal(i0[:2000].cpu().numpy(), io)
            assert np.array_equal(t0[:2000].cpu().numpy().view(np.uint32), to.view(np.uint32))


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_reciprocal(dev, sign):
    """The corrected reciprocal of the triangle test against the division, for
    every significand: a = m for a ray (0.25, 0.25, 1) + t (0, 0, -m) and the
    triangle (0, 0, 0), (1, 0, 0), (0, 1, 0), t = 1 / m."""
    v = np.float32([[[0, 0, 0], [1, 0, 0], [0, 1, 0]]])
    if sign < 0:
        v = v[:, [0, 2, 1]]
    v = np.ascontiguousarray(v)
    m = rm._lib.RmMaterial(roughness=0.8, opacity=1.0, ior=1.0, albedo_tex=-1, normal_tex=-1, emissive_tex=-1, specular_tex=-1)
    desc, keep = make_desc(v, np.zeros((1, 3, 2)), np.zeros(1), np.zeros(1), [m], [])
    S = rm.Scene(desc)
    bits = torch.arange(1 << 23, device=dev, dtype=torch.int32) + 0x3f800000
    x = bits.view(torch.float32)
    r = torch.zeros(1 << 23, 6, device=dev)
    r[:, 0] = r[:, 1] = 0.25
    r[:, 2] = 1.0
    r[:, 5] = -x
    t, ids = S.trace_closest(r)
    want = (1.0 / x.double()).float()  # (of 24 bits, so rounding twice does no harm)
    assert bool((ids == 0).all())
    assert torch.equal(t.view(torch.int32), want.view(torch.int32))
    for scale in (2.0 ** -12, 2.0 ** 20, 2.0 ** 25):
        r[:, 5] = -x * scale
        t, ids = S.trace_closest(r, tmin=1e-9)
        assert bool((ids == 0).all())
        assert torch.equal((t * scale).view(torch.int32), want.view(torch.int32)), scale


@pytest.mark.parametrize("tris", [36, 3001])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 511, 1639, 13107, 131073, 524287, 4194305])
def test_ray_counts(dev, n, tris):
    """Every split of a batch over waves and lanes gives the reference walk's results."""
    S = rm.Scene(rm.generate(1, 5, n_tris=tris))
    r = torch.from_numpy(rm.rays(1, n, seed=n)).to(dev)
    t, ids = S.trace_closest(r)
    occ = S.trace_any(r, aim=0.3)
    try:
        rm.set_tuning(rm.TUNE_TRACE_VARIANT, 0)
        t0, i0 = S.trace_closest(r)
        occ0 = S.trace_any(r, aim=0.3)
        torch.cuda.synchronize()
    finally:
        rm.set_tuning(rm.TUNE_TRACE_VARIANT, 3)
    assert torch.equal(ids, i0) and torch.equal(t.view(torch.int32), t0.view(torch.int32)) and torch.equal(occ, occ0)
