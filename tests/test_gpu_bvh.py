"""The optimised path's hierarchy against the brute force over all triangles:
its boxes must hold every point the triangle test can accept, whatever the
triangles' shapes, sizes and count, and wherever the rays start."""
import numpy as np
import pytest

import oracle
from tests import helpers as H
from vrad_amd import scenes
from vrad_amd.raytracer import Environment

pytestmark = pytest.mark.gpu


def _env(v9, ids):
    env = Environment()
    env.AddTriangles(v9, ids)
    env.SetupAccelerationStructure()
    return env


def _soup(rng, n, extent=500.0, size=60.0):
    c = rng.uniform(-extent, extent, (n, 1, 3))
    return (c + rng.normal(size=(n, 3, 3)) * size).astype(np.float32).reshape(n, 9)


def _slivers(rng, n):
    """Triangles a few hundred long and 1e-3 to 1 wide, some of no area."""
    a = rng.uniform(-400, 400, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    w = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-3, 0, (n, 1))
    w[::17] = 0.0
    b = a + d * rng.uniform(100, 600, (n, 1))
    return np.stack([a, b, a + 0.4 * (b - a) + w], 1).astype(np.float32).reshape(n, 9)


def _grid(rng, n):
    """Coplanar unit quads, the same plane and areas everywhere: every
    clustering choice is a tie."""
    k = int(np.ceil(np.sqrt(n / 2)))
    x, y = np.meshgrid(np.arange(k), np.arange(k))
    x, y, z = x.ravel() * 8.0, y.ravel() * 8.0, np.zeros(k * k)
    p = [np.stack([x + i, y + j, z], 1) for i, j in ((0, 0), (8, 0), (8, 8), (0, 8))]
    t = np.concatenate([np.stack([p[0], p[1], p[2]], 1), np.stack([p[0], p[2], p[3]], 1)])
    return t[:n].astype(np.float32).reshape(-1, 9)


def _rays(rng, v9, n):
    """Rays through random points of random triangles (on edges and corners
    too) from near, within and far outside the scene, and axis-aligned ones."""
    v = v9.reshape(-1, 3, 3).astype(np.float64)
    k = rng.integers(0, len(v), n)
    w = rng.dirichlet((0.7, 0.7, 0.7), n)
    w[::5, 0], w[::5] = 0.0, w[::5] / np.maximum(w[::5].sum(1, keepdims=True), 1e-9)
    p = (v[k] * w[:, :, None]).sum(1)
    d = rng.normal(size=(n, 3))
    d[::7] = np.eye(3)[rng.integers(0, 3, len(d[::7]))] * rng.choice([-1.0, 1.0], (len(d[::7]), 1))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    far = 10.0 ** rng.uniform(-2, 6, (n, 1))
    return (p - d * far).astype(np.float32), d.astype(np.float32)


def _check(v9, rng, n_rays, skip=-1):
    n = len(v9)
    ids = np.where(rng.random(n) < 0.1, H.SKY, H.OPAQUE).astype(np.int32)
    env, tri = _env(v9, ids), oracle.precompute(v9, ids)
    o, d = _rays(rng, v9, n_rays)
    print(f"[gpu] {n} triangles, {n_rays} rays", flush=True)
    hg, tg = env.TraceRays(o, d, 0.0, 1e30, skip_id=skip)
    hb, tb = oracle.trace_brute(tri, o, d, 0.0, 1e30, skip=skip)
    assert np.array_equal(hg, hb)
    assert np.array_equal(tg.view(np.uint32), tb.view(np.uint32))
    e = (o + d * rng.uniform(0, 2000, (n_rays, 1))).astype(np.float32)
    e[:3] = o[:3]  # no length
    vg, sg = env.TestLines(o, e)
    vb, sb = oracle.testline(None, tri, o, e)
    assert np.array_equal(vg, vb) and np.array_equal(sg, sb)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 255, 256, 257, 2047, 2048, 2049, 2600])
def test_soup_sizes(n):
    rng = np.random.default_rng(100 + n)
    _check(_soup(rng, n), rng, 3000)


@pytest.mark.parametrize("n", [64, 3000])
def test_slivers(n):
    rng = np.random.default_rng(n)
    _check(_slivers(rng, n), rng, 4000)


@pytest.mark.parametrize("offset", [2000.0, 30000.0, 1e6])
def test_far_from_the_origin(offset):
    rng = np.random.default_rng(7)
    v9 = _soup(rng, 1500, 300.0, 25.0) + np.float32(offset)
    _check(v9.astype(np.float32), rng, 4000)


def test_equal_triangles_and_grids():
    rng = np.random.default_rng(9)
    one = _soup(rng, 1)
    _check(np.repeat(one, 5000, 0), rng, 200)
    _check(_grid(rng, 6000), rng, 3000)


def test_one_triangle_covers_the_rest():
    rng = np.random.default_rng(10)
    v9 = _soup(rng, 3000, 50.0, 1.0)
    v9[1234] = [-9e4, -9e4, 3, 9e4, -9e4, 3, 0, 1.6e5, 3]
    _check(v9, rng, 3000)


def test_level_with_props_vs_oracle_kd():
    """A level with thousands of boxes standing in and through its walls."""
    rng = np.random.default_rng(11)
    s = scenes.level(seed=4, rooms_x=4, rooms_y=4, chop=64.0, tess=64.0, n_lights=4)
    tris = []
    for lo in rng.uniform([0, 0, 0], [s.grid_x[-1], s.grid_y[-1], 200], (600, 3)):
        tris += H.box(tuple(lo), tuple(lo + rng.uniform(1, 60, 3)), 0x04000000)
    v9, ids = H.to_arrays(tris)
    v9, ids = np.concatenate([s.verts9, v9]), np.concatenate([s.ids, ids])
    env, tri, kd = _env(v9, ids), oracle.precompute(v9, ids), oracle.KdTree(v9)
    k = rng.integers(0, len(s.p_area), 60000)
    o = (s.p_origin[k] + np.float32(0.1) * s.p_normal[k]).astype(np.float32)
    d = rng.normal(size=o.shape)
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    hg, tg = env.TraceRays(o, d, 0.0, H.MTL)
    hk, tk = oracle.trace_kd(kd, tri, o, d, 0.0, H.MTL, threads=8)
    assert np.array_equal(hg, hk) and np.array_equal(tg.view(np.uint32), tk.view(np.uint32))
