"""GatherSampleLight with 1 to 16 waves per 64 samples: the terms are added in
list order whichever wave traced them."""
import numpy as np
import pytest

import oracle
from tests import helpers as H
from vrad_amd import lightmap, scenes
from vrad_amd.raytracer import Environment

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def level():
    s = scenes.level(seed=5, rooms_x=3, rooms_y=3, chop=32.0, tess=64.0, n_lights=4, sun=True)
    env = Environment()
    env.AddTriangles(s.verts9, s.ids)
    env.SetupAccelerationStructure()
    return s, env, oracle.precompute(s.verts9, s.ids), oracle.KdTree(s.verts9)


def _lights(rng, s, n, ambient):
    """Points, spots, surfaces and the sun, `ambient` sky-ambient ones among them."""
    out = []
    for k in range(n):
        o = s.p_origin[rng.integers(len(s.p_origin))] + np.float32([0, 0, 40])
        inten = rng.uniform(1, 100, 3).astype(np.float32)
        kind = k % 5
        if kind == 0:
            out.append(lightmap.point_light(o, inten, quadratic=1.0))
        elif kind == 1:
            out.append(lightmap.spot_light(o, rng.normal(size=3), inten, 40.0, 70.0,
                                           exponent=float(rng.choice([0.0, 1.0, 2.5])),
                                           quadratic=1.0))
        elif kind == 2:
            out.append(H.light(0, o, (0, 0, -1), inten))
        elif kind == 3:
            out.append(lightmap.point_light(o, inten, fifty_percent_distance=200.0,
                                            zero_percent_distance=600.0, hardfalloff=True))
        else:
            out.append(lightmap.sun_light((0.2, 0.3, -1.0), inten))
    for k in range(ambient):
        at = int(rng.integers(0, len(out) + 1))
        out.insert(at, H.light(5, inten=rng.uniform(0.1, 1, 3)))
    return np.concatenate([np.asarray(a, lightmap.make_lights(0).dtype) for a in out])


# waves per group: 1 (one light), 2, 4, 8, 16; 16 with sky ambient alone, first,
# last or between; more lights than one batch of a workgroup (192); sizes that
# leave a partial group
@pytest.mark.parametrize("n,lights,ambient", [(1, 1, 0), (63, 3, 0), (65, 5, 0), (1000, 9, 0),
                                              (129, 17, 0), (64, 0, 1), (130, 4, 1), (70, 3, 2),
                                              (200, 200, 0), (90, 400, 1), (7000, 2, 0)])
def test_gather_waves_vs_oracle(level, n, lights, ambient):
    s, env, tri, kd = level
    rng = np.random.default_rng([n, lights, ambient])
    k = rng.integers(0, len(s.p_area), n)
    L = _lights(rng, s, lights, ambient)
    print(f"[gpu] {n} samples, {lights} lights, {ambient} sky ambient", flush=True)
    got = lightmap.GatherSampleLight(env, s.p_origin[k], s.p_normal[k], L)
    want = oracle.gather_light(kd, tri, s.p_origin[k], s.p_normal[k], L, threads=8)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_gather_waves_batch_of_scenes(level):
    s, env, tri, kd = level
    rng = np.random.default_rng(3)
    items = []
    for n, lights, ambient in ((70, 2, 1), (500, 12, 0), (0, 3, 0), (64, 0, 0)):
        k = rng.integers(0, len(s.p_area), n)
        L = _lights(rng, s, lights, ambient) if lights + ambient else lightmap.make_lights(0)
        items.append((env, s.p_origin[k], s.p_normal[k], L))
    for (_, p, q, L), got in zip(items, lightmap.GatherSampleLightBatch(items)):
        want = oracle.gather_light(kd, tri, p, q, L, threads=4) if len(p) else got
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
