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


SCENES = {
    "one_leaf": lambda: soup(10, 1, 0.5), "two_leaves": lambda: soup(11, 2, 0.5), "soup20": lambda: soup(20, 3, 0.4),
    "soup21": lambda: soup(21, 4, 0.4), "soup48": lambda: soup(48, 5, 0.3), "soup49": lambda: soup(49, 6, 0.3),
    "soup64": lambda: soup(64, 13, 0.3), "soup65": lambda: soup(65, 14, 0.3),
    "slivers": lambda: (soup(60, 15, 0.8) * np.array([1, 1e-4, 1]) + np.array([90, 40, -7])).astype(np.float32),
    "soup80": lambda: soup(80, 7, 0.3), "soup81": lambda: soup(81, 8, 0.3), "soup1301": lambda: soup(1301, 9),
    "soup7001": lambda: soup(7001, 10, 0.05), "walls": lambda: walls(9),
    "doubled": lambda: np.repeat(soup(700, 11, 0.2), 2, axis=0),
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
        for tmin, tmax in ((1e-4, np.inf), (0.05, 0.7)) if kind != "odd" else ((1e-4, np.inf),):
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
