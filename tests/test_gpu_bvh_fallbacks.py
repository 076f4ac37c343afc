"""What the visibility kernels fall back on: the balanced hierarchy for clustered
trees deeper than the walk's stack holds, and the kd-tree for scenes with more
nodes than the hierarchy's offsets reach.  Both are forced on small scenes by
their knobs; results are those of the brute force and of the ordinary route."""
import contextlib

import numpy as np
import pytest

from tests import helpers as H
from tests import test_gpu_bvh as B
from vrad_amd import _lib, autotune, lightmap, pvs, scenes
from vrad_amd.patches import MakeTransfers, MakeTransfersBatch
from vrad_amd.raytracer import Environment

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def knob(name, value):
    old = autotune.get_knob(name)
    autotune.set_knob(name, value)
    try:
        yield
    finally:
        autotune.set_knob(name, old)


def _nested(n, step):
    """Triangles one inside the other: every cluster's best neighbour is any of
    the smaller ones, so a round of choices merges next to nothing."""
    s = 1000.0 * step ** np.arange(n)
    v = np.array([[-1, -1, 0.2], [1, -1, -0.1], [0, 1.5, 0.3]])
    return (s[:, None, None] * v).astype(np.float32).reshape(n, 9)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 9, 33, 257, 2049, 2600])
def test_balanced_tree(n):
    rng = np.random.default_rng(300 + n)
    with knob("bvh_levels", 1):
        B._check(B._soup(rng, n), rng, 2000)


def test_balanced_tree_of_slivers_and_grids():
    rng = np.random.default_rng(31)
    with knob("bvh_levels", 1):
        B._check(B._slivers(rng, 3000), rng, 2000)
        B._check(B._grid(rng, 6000), rng, 2000)


# 300: some 220 clusters are left after 64 rounds of the last workgroup, 4000: 3150
# after 60 rounds over all workgroups; then neighbours are paired.  Every round
# put the smallest two together, so the tree is too deep and built balanced.
@pytest.mark.parametrize("n", [300, 4000])
def test_rounds_that_merge_next_to_nothing(n):
    rng = np.random.default_rng(n)
    B._check(_nested(n, 1e-4 ** (1.0 / n)), rng, 2000)


@pytest.fixture(scope="module")
def both():
    """A level built for the hierarchy, and again past a limit of 0 nodes."""
    s = scenes.level(seed=3, rooms_x=3, rooms_y=2, chop=48.0, tess=96.0, n_lights=3, sun=True)
    ids = s.ids.copy()
    ids[::11] = H.SKY
    envs = []
    for most in (1 << 25, 0):
        with knob("bvh_max_nodes", most):
            env = Environment()
            env.AddTriangles(s.verts9, ids)
            env.SetupAccelerationStructure()
            envs.append(env)
    return s, envs


@pytest.mark.parametrize("rays_per_lane", [1, 4])
def test_kd_fallback_rays_and_segments(both, rays_per_lane):
    s, envs = both
    rng = np.random.default_rng(1)
    k = rng.integers(0, len(s.p_area), 20001)
    o = (s.p_origin[k] + np.float32(0.1) * s.p_normal[k]).astype(np.float32)
    d = rng.normal(size=o.shape).astype(np.float32)
    e = s.p_origin[rng.permutation(k)]
    with knob("trace_rays_per_lane", rays_per_lane):
        want, got = [(*env.TraceRays(o, d, 0.0, H.MTL), *env.TestLines(o, e)) for env in envs]
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("grouped", [False, True])
def test_kd_fallback_transfers(both, grouped):
    s, envs = both
    o, nr, ar = s.p_origin[:1537], s.p_normal[:1537], s.p_area[:1537]
    kw = {}
    if grouped:
        bsp, vis = scenes.grid_bsp(s.grid_x, s.grid_y, pvs_hops=1)
        kw = dict(cluster=pvs.ClusterFromPoint(bsp, o).astype(np.int32),
                  pvs_rows=pvs.DecompressVis(vis)[0])

    def csr(xf):
        out = xf.download()
        xf.close()
        return out
    print(f"[gpu] fallback transfers grouped={grouped}", flush=True)
    want = csr(MakeTransfers(envs[0], o, nr, ar, **kw))
    got = [csr(MakeTransfers(envs[1], o, nr, ar, **kw)),
           csr(MakeTransfers(envs[1], o, nr, ar, batch_pairs=60000, **kw))]
    if not grouped:  # one scene of each kind together
        got += [csr(x) for x in MakeTransfersBatch([(env, o, nr, ar) for env in envs])]
    for g in got:
        for a, b in zip(want, g):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_kd_fallback_light_and_sky(both):
    s, envs = both
    L = np.concatenate([np.asarray(s.lights), H.light(5, inten=(0.2, 0.3, 0.4))])
    p, q = s.p_origin[:3001], s.p_normal[:3001]
    want = lightmap.GatherSampleLight(envs[0], p, q, L)
    assert want.any()
    got = [lightmap.GatherSampleLight(envs[1], p, q, L),
           *lightmap.GatherSampleLightBatch([(env, p, q, L) for env in envs])]
    for g in got:
        assert np.array_equal(want.view(np.uint32), g.view(np.uint32))
    lo = s.p_origin[:500].astype(np.int16)
    hi = lo + 8
    want, got = [lightmap.CanLeafTraceToSky(env, lo, hi) for env in envs]
    assert np.array_equal(want, got)


@pytest.mark.parametrize("n", [1, 5, 3000])
def test_no_triangle_can_be_hit(n):
    """Triangles of no area (all points equal) have no normal: the scene has a
    tree and no hierarchy."""
    v9 = np.repeat(np.float32([[1, 2, 3]]), 3 * n, 0).reshape(n, 9)
    ids = np.where(np.arange(n) % 2, H.SKY, H.OPAQUE).astype(np.int32)
    env = Environment()
    env.AddTriangles(v9, ids)
    env.SetupAccelerationStructure()
    o = np.float32([[0, 0, 0], [1, 2, 3], [1, 2, 0]])
    d = np.float32([[0.267, 0.534, 0.802], [1, 0, 0], [0, 0, 1]])
    hit, _ = env.TraceRays(o, d, 0.0, 1e30)
    vis, sky = env.TestLines(o, o + 10 * d)
    assert (np.asarray(hit) == -1).all() and np.asarray(vis).all() and not np.asarray(sky).any()
