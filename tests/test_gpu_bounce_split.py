"""Stream gather with a chunk's waves shared among 1 to 8 workgroups, and the
energy tree with its last-workgroup stage: the restatement's order at the row
counts where the split or the number of energy blocks changes."""
import numpy as np
import pytest

import oracle
from vrad_amd import _lib, lightmap
from vrad_amd.patches import Transfers

pytestmark = pytest.mark.gpu

PRECISIONS = {"f32": _lib.VR_COEF_F32, "f16": _lib.VR_COEF_F16, "bf16": _lib.VR_COEF_BF16}


# 8 workgroups per chunk up to 32 chunks (8192 rows), 4 to 16384, 2 to 32768;
# 1, 2 and more energy blocks of 2048 rows; tile boundaries of 4096 columns
@pytest.mark.parametrize("prec", list(PRECISIONS))
@pytest.mark.parametrize("n", [2, 257, 2048, 2049, 4097, 8192, 8193, 16384, 16385, 32768, 32769])
def test_split_bitexact(n, prec):
    xf = Transfers.synthetic(seed=n, n_rows=n, mean_len=min(60.0, 0.5 * n), sigma=1.0,
                             max_len=min(900, n - 1))
    kind = PRECISIONS[prec]
    raw = scale = None
    if kind == _lib.VR_COEF_F32:
        rp, col, coef = xf.download()
    else:
        xf.set_precision(kind)
        rp, col, _, coef, scale = xf.download(raw16=True)
    rng = np.random.default_rng(n)
    e0 = rng.random((n, 3)).astype(np.float32)
    refl = rng.uniform(0.2, 0.8, (n, 3)).astype(np.float32)
    area = rng.uniform(1, 4, n).astype(np.float32)
    print(f"[gpu] n={n} {prec} nnz={len(col)}", flush=True)
    for k in (1, 5):
        tot, en, kk = lightmap.BounceLight(xf, e0, refl, area, max_bounces=k, stop_frac=0.0)
        otot, oen, ok = oracle.bounce_f32(rp, col, coef, e0, refl, area, max_bounces=k,
                                          stop_frac=0.0, kind=kind, row_scale=scale, threads=8)
        assert kk == ok == k
        assert np.array_equal(tot.view(np.uint32), otot.view(np.uint32))
        assert np.array_equal(en.view(np.uint64), oen.view(np.uint64))
