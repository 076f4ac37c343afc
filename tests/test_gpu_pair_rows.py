"""MakeTransfers' row-by-row trace (queued survivors, one direction of the bits
and their mirror image) against the plain path's pair list: the same CSR, bit
for bit, where tiles and words end, for patches out of order and for scattered
groups."""
import numpy as np
import pytest

from vrad_amd import _lib, pvs, scenes
from vrad_amd.patches import MakeTransfers, MakeTransfersBatch
from vrad_amd.raytracer import Environment

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def level():
    s = scenes.level(seed=3, rooms_x=3, rooms_y=2, chop=48.0, tess=96.0, n_lights=2, sun=True)
    env = Environment()
    env.AddTriangles(s.verts9, s.ids)
    env.SetupAccelerationStructure()
    bsp, vis = scenes.grid_bsp(s.grid_x, s.grid_y, pvs_hops=1)
    rows = pvs.DecompressVis(vis)[0]
    return s, env, bsp, rows


def csr(xf):
    inf = xf.info()
    out = (int(inf.nnz), int(inf.segments_traced), int(inf.pairs_considered), *xf.download())
    xf.close()
    return out


def same(a, b):
    assert a[:3] == b[:3]
    for x, y in zip(a[3:], b[3:]):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


# 32-column words, 512-row mirror tiles (one, an even and an odd number of
# them), 64-segment batches; patches in order, shuffled (a wave's segments
# run everywhere) and with one group scattered over the indices
@pytest.mark.parametrize("order", ["listed", "shuffled"])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("n", [1, 2, 31, 33, 65, 511, 513, 1024, 1537, 3001])
def test_rows_equal_pair_list(level, n, order, grouped):
    s, env, bsp, rows = level
    rng = np.random.default_rng(n)
    k = np.arange(len(s.p_area))
    if order == "shuffled":
        rng.shuffle(k)
    k = k[:n]
    o, nr, ar = (np.ascontiguousarray(a[k]) for a in (s.p_origin, s.p_normal, s.p_area))
    kw = {}
    if grouped:
        cl = pvs.ClusterFromPoint(bsp, o).astype(np.int32)
        cl[rng.random(n) < 0.02] = -1
        kw = dict(cluster=cl, pvs_rows=rows)
    print(f"[gpu] n={n} {order} grouped={grouped}", flush=True)
    try:
        _lib.check(_lib.lib.vr_set_path(_lib.VR_PATH_PLAIN))
        want = csr(MakeTransfers(env, o, nr, ar, **kw))
    finally:
        _lib.check(_lib.lib.vr_set_path(_lib.VR_PATH_OPT))
    same(csr(MakeTransfers(env, o, nr, ar, **kw)), want)
    if not grouped:
        got = MakeTransfersBatch([(env, o, nr, ar), (env, o[: n // 2], nr[: n // 2], ar[: n // 2])])
        same(csr(got[0]), want)
        got[1].close()
