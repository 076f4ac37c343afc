"""The pool of device blocks against a recorded stand-in for the HIP calls: what
it hands out, keeps and gives back, without a GPU."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "vrad_amd", "csrc")
MB, GB = 1 << 20, 1 << 30


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("devmem") / "pool.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so,
                    os.path.join(HERE, "devmem_harness.cpp"), os.path.join(CSRC, "devmem.cpp")],
                   check=True)
    return so


@pytest.fixture
def pool(built, tmp_path):
    """A fresh pool (its own copy of the library) on a device of 64 GB."""
    so = tmp_path / "pool.so"
    so.write_bytes(open(built, "rb").read())
    lib = C.CDLL(str(so))
    for name in ("t_alloc",):
        getattr(lib, name).restype = C.c_void_p
    for name in ("t_used", "t_bytes", "t_syncs", "t_release"):
        getattr(lib, name).restype = C.c_int64
    lib.t_alloc.argtypes = lib.t_setup.argtypes = [C.c_int64]
    lib.t_free_idle.argtypes = lib.t_free.argtypes = lib.t_bytes.argtypes = lib.t_block_device.argtypes = [C.c_void_p]
    lib.t_setup(64 * GB)
    return lib


def test_freed_block_waits_for_the_device(pool):
    """A block given back with work in flight is handed out after a
    synchronisation, which one request pays for all."""
    a, b = pool.t_alloc(MB), pool.t_alloc(3 * MB)
    pool.t_free(a)
    pool.t_free(b)
    assert pool.t_syncs(0) == 0
    assert pool.t_alloc(MB) == a and pool.t_syncs(0) == 1
    assert pool.t_alloc(3 * MB) == b and pool.t_syncs(0) == 1


def test_failed_synchronisation_hands_nothing_out(pool):
    """A synchronisation that fails (a stream of the caller is capturing) says
    nothing about the work that uses a freed block."""
    a = pool.t_alloc(MB)
    pool.t_free(a)
    pool.t_sync_error(1)
    b = pool.t_alloc(MB)
    assert b is not None and b != a
    assert pool.t_bytes(a) >= MB  # nor did it go back to the driver
    pool.t_sync_error(0)
    assert pool.t_alloc(MB) == a and pool.t_syncs(0) == 1


def test_kept_memory_is_bounded(pool):
    """256 MB without a live handle, an eighth of the device with one; the rest
    goes back to the driver."""
    blocks = [pool.t_alloc(100 * MB) for _ in range(5)]
    for p in blocks:
        pool.t_free(p)
    assert pool.t_used() <= 256 * MB
    pool.t_holder(1)
    blocks = [pool.t_alloc(2 * GB) for _ in range(8)]
    for p in blocks:
        pool.t_free(p)
    assert 6 * GB < pool.t_used() <= 8 * GB
    big = pool.t_alloc(9 * GB)
    pool.t_free(big)
    assert pool.t_bytes(big) == -1
    pool.t_holder(-1)
    assert pool.t_used() <= 256 * MB


def test_kept_blocks_go_back_when_memory_runs_out(pool):
    pool.t_holder(1)
    a = pool.t_alloc(7 * GB)
    pool.t_free(a)
    assert pool.t_alloc(60 * GB) is not None
    assert pool.t_bytes(a) == -1


def test_devices_do_not_share_blocks(pool):
    """A request gets memory of the device that is current, and a freed block
    waits for its own device, whichever is current then."""
    pool.t_device(1)
    a = pool.t_alloc(MB)
    pool.t_device(0)
    pool.t_free(a)
    b = pool.t_alloc(MB)
    assert b != a and pool.t_block_device(b) == 0
    pool.t_free(b)
    c = pool.t_alloc(MB)
    assert c == b and (pool.t_syncs(0), pool.t_syncs(1)) == (1, 0)
    pool.t_device(1)
    assert pool.t_alloc(MB) == a and (pool.t_syncs(0), pool.t_syncs(1)) == (1, 1)


def test_trim_waits_for_every_device(pool):
    """The last handle gives back what is above 256 MB on each device, after a
    synchronisation of that device, and leaves the current device as it was."""
    pool.t_holder(1)
    for dev in (1, 0):
        pool.t_device(dev)
        pool.t_free(pool.t_alloc(GB))
    pool.t_holder(-1)
    assert pool.t_used() <= 2 * 256 * MB
    assert (pool.t_syncs(0), pool.t_syncs(1)) == (1, 1) and pool.t_current() == 0


def test_requests_that_fit_the_device_are_served(pool):
    """Sizes are rounded up so that similar requests share blocks, but what that
    adds is bounded (1/128 of the device), so it does not take the memory that a
    set near the device's capacity needs."""
    pool.t_holder(1)
    blocks = [pool.t_alloc(6300 * MB) for _ in range(10)]  # 61.5 of 64 GB
    assert all(blocks) and pool.t_used() <= 63000 * MB + 512 * MB
    assert pool.t_alloc(64 * GB - pool.t_used()) is not None  # to the last byte
    assert pool.t_used() == 64 * GB


def test_small_requests_share_blocks_when_nothing_is_spare(pool):
    """The bound is for what counts: up to 64 KiB a block is always rounded."""
    pool.t_holder(1)
    for n in (6300 * MB, 200 * MB + 1, 3 * MB + 1, MB + 1, 300001, 70001, 5000):
        while True:  # until the size is no longer rounded, or often enough
            p = pool.t_alloc(n)
            if pool.t_bytes(p) == n or pool.t_used() > 60 * GB or n <= 70001:
                break
    a = pool.t_alloc(37000)
    assert pool.t_bytes(a) == 40960
    pool.t_free(a)
    assert pool.t_alloc(39000) == a


def test_similar_requests_share_a_block(pool):
    pool.t_holder(1)
    for n in (1001 * MB, 1010 * MB, 990 * MB):
        a = pool.t_alloc(n)
        pool.t_free(a)
    assert pool.t_used() < 1100 * MB


def test_release_gives_everything_back(pool):
    """All kept blocks of every device; those whose work may still run stay."""
    pool.t_holder(1)
    for dev in (1, 0):
        pool.t_device(dev)
        pool.t_free(pool.t_alloc(GB))
    pool.t_sync_error(1)
    assert pool.t_release() == 2 * GB == pool.t_used()
    pool.t_sync_error(0)
    assert pool.t_release() == 0 == pool.t_used()


class Hip:
    """The HIP runtime the library itself is linked with."""

    def __init__(self):
        from vrad_amd import _lib
        self.lib, self.check, self.held = _lib.lib, _lib.check, []
        self.check(self.lib.vr_init(0))

    def call(self, name, *args):
        assert getattr(self.lib, name)(*args) == 0, name

    def free(self):
        f, t = C.c_size_t(), C.c_size_t()
        self.call("hipMemGetInfo", C.byref(f), C.byref(t))
        return f.value

    def array(self, a):
        p = C.c_void_p()
        self.call("hipMalloc", C.byref(p), C.c_size_t(a.nbytes))
        self.call("hipMemcpy", p, C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes), 1)
        self.held.append(p)
        return p

    def host(self, p, a):
        self.call("hipMemcpy", C.c_void_p(a.ctypes.data), p, C.c_size_t(a.nbytes), 2)
        return a

    def close(self):
        for p in self.held:
            self.call("hipFree", p)


@pytest.fixture
def hip():
    h = Hip()
    yield h
    h.close()


@pytest.mark.gpu
def test_released_memory_is_there_for_others(hip):
    """With a scene alive, freed transfers stay with the library until they are
    asked for; then another allocator of the process gets them."""
    import vrad_amd
    from vrad_amd import scenes
    from vrad_amd.patches import Transfers
    from vrad_amd.raytracer import Environment
    s = scenes.room(seed=1, n_pillars=2, chop=128.0, tess=128.0)
    env = Environment()
    env.AddTriangles(s.verts9, s.ids)
    env.SetupAccelerationStructure()
    vrad_amd.release_memory()
    xf = Transfers.synthetic(seed=1, n_rows=1 << 18, mean_len=512.0, sigma=0.0, max_len=600)
    held = xf.info().stored_bytes
    assert held > GB // 2
    before = hip.free()
    xf.close()
    assert hip.free() - before < held // 2
    vrad_amd.release_memory()
    assert hip.free() - before >= held * 9 // 10


def test_idle_blocks_need_no_synchronisation(pool):
    """A block whose work the caller has waited for is available at once; others
    still wait."""
    a, b = pool.t_alloc(MB), pool.t_alloc(3 * MB)
    pool.t_free_idle(a)
    pool.t_free(b)
    assert pool.t_alloc(MB) == a and pool.t_syncs(0) == 0
    assert pool.t_alloc(3 * MB) == b and pool.t_syncs(0) == 1
    pool.t_free_idle(a)
    assert pool.t_release() == 0 and pool.t_bytes(a) == -1


def test_host_scenes_hold_no_memory():
    """A scene that was never built on the device does not raise what is kept."""
    from vrad_amd import _lib
    import numpy as np
    count = getattr(_lib.lib, "_ZN2vr10dev_holderEi")
    before = count(0)
    h, v9, ids = C.c_void_p(), np.zeros((1, 9), np.float32), np.zeros(1, np.int32)
    v9[0, 3] = v9[0, 7] = 1.0
    _lib.check(_lib.lib.vr_scene_create(C.byref(h), _lib.ptr(v9), _lib.ptr(ids), None, 1))
    _lib.check(_lib.lib.vr_scene_build_host(h, 1))
    assert count(0) == before
    _lib.check(_lib.lib.vr_scene_destroy(h))
    assert count(0) == before


@pytest.mark.gpu
def test_scene_closed_while_a_callers_stream_walks_it(hip):
    """A scene is closed and another built over its blocks while launches on the
    caller's stream still walk it: they finish with its results."""
    import numpy as np
    from vrad_amd import _lib, scenes
    from vrad_amd.raytracer import Environment

    def env(seed):
        s = scenes.level(seed=seed, rooms_x=3, rooms_y=3, chop=64.0, tess=64.0, n_lights=1)
        e = Environment()
        e.AddTriangles(s.verts9, s.ids)
        e.SetupAccelerationStructure()
        return s, e
    s, a = env(1)
    n, rows = 1 << 20, 41
    rng = np.random.default_rng(2)
    i, j = rng.integers(0, len(s.p_area), (2, n))
    cols = np.concatenate([s.p_origin[i] + s.p_normal[i] / 8, s.p_origin[j] + s.p_normal[j] / 8], 1)
    segs = _lib.Segs(*(C.cast(hip.array(np.ascontiguousarray(c, np.float32)), _lib.FP)
                       for c in cols.T))
    got = np.zeros((rows, n), np.uint8)
    out, stream = hip.array(got), C.c_void_p()
    hip.call("hipStreamCreate", C.byref(stream))
    for row in range(rows):
        _lib.check(_lib.lib.vr_test_line_dev(a.handle, C.byref(segs), n, -1,
                                             C.c_void_p(out.value + row * n), None, stream))
        if row == 0:
            hip.call("hipStreamSynchronize", stream)
    a.close()
    _, b = env(2)  # of the same size
    hip.call("hipStreamSynchronize", stream)
    hip.host(out, got)
    hip.call("hipStreamDestroy", stream)
    assert got[0].any() and not got[0].all()
    assert (got[1:] == got[0]).all()
    b.close()
