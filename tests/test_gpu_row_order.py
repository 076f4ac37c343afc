"""Rows dealt to the gather's chunks longest first by the device's sort: bounce
sums equal the restatement's, which follows the same order, at sizes around a
wave's 1024 rows and lengths of one to three bytes, many of them equal."""
import numpy as np
import pytest

import oracle
from vrad_amd import lightmap
from vrad_amd.patches import Transfers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,longest", [(1, 0), (63, 3), (65, 60), (1023, 255), (1024, 256),
                                       (1025, 700), (5000, 4999), (70000, 66000)])
def test_order_bitexact(n, longest):
    rng = np.random.default_rng(n)
    cnt = rng.integers(0, min(longest, 40) + 1, n)  # many ties
    cnt[rng.integers(0, n, 3)] = longest
    cnt[-1] = longest // 2
    rp = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    col = np.concatenate([np.sort(rng.choice(n, c, replace=False)) if c else np.zeros(0, np.int64)
                          for c in cnt]).astype(np.int32)
    coef = (rng.random(len(col)) / max(longest, 1)).astype(np.float32)
    print(f"[gpu] n={n} longest={longest} nnz={len(col)}", flush=True)
    xf = Transfers.from_csr(rp, col, coef)
    e0 = rng.random((n, 3)).astype(np.float32)
    refl = rng.uniform(0.2, 0.8, (n, 3)).astype(np.float32)
    area = rng.uniform(1, 4, n).astype(np.float32)
    tot, en, k = lightmap.BounceLight(xf, e0, refl, area, max_bounces=2, stop_frac=0.0)
    otot, oen, ok = oracle.bounce_f32(rp, col, coef, e0, refl, area, max_bounces=2, stop_frac=0.0,
                                      threads=8)
    assert k == ok
    assert np.array_equal(tot.view(np.uint32), otot.view(np.uint32))
    assert np.array_equal(en.view(np.uint64), oen.view(np.uint64))
