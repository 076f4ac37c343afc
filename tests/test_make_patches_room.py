"""MakePatches sizes its output before the library has looked at the arguments:
what the library refuses is refused by it, and any room gives the same array."""
import numpy as np
import pytest

from vrad_amd import _lib, patches


def _faces(n):
    f = np.zeros(n, _lib.FACE_DTYPE)
    f["n_points"] = 4
    f["points"][:, :4] = [[0, 0, 0], [256, 0, 0], [256, 192, 0], [0, 192, 0]]
    f["points"][:, :, 2] = 8.0 * np.arange(n)[:, None]
    f["normal"] = [0, 0, 1]
    f["lux_s"], f["lux_t"] = [1 / 16, 0, 0], [0, 1 / 16, 0]
    return f


@pytest.mark.parametrize("chop", [float("nan"), 0.0, -1.0, float("-inf")])
def test_bad_chop_is_the_librarys_error(chop):
    degenerate = _faces(3)
    degenerate["lux_s"][1] = 0.0
    for f in (_faces(0), _faces(2), degenerate):
        with pytest.raises(_lib.VrError) as e:
            patches.MakePatches(f, max_chop=chop)
        assert e.value.code == _lib.VR_E_INVALID


@pytest.mark.gpu
@pytest.mark.parametrize("room", [0, 1, 7, 100000])
def test_any_room_gives_the_same_patches(monkeypatch, room):
    f = _faces(5)
    want = patches.MakePatches(f, max_chop=4.0, min_chop=4.0)
    assert len(want) > 7
    monkeypatch.setattr(patches, "_patch_room", lambda *_: room)
    got = patches.MakePatches(f, max_chop=4.0, min_chop=4.0)
    assert got.tobytes() == want.tobytes()
    assert got.base is None and got.flags.owndata and want.base is None
    assert len(patches.MakePatches(f[:0])) == 0
