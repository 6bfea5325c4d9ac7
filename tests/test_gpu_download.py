"""Downloads around the chunk size, and around the size from which further
threads help (four chunks): the state comes back in upload order,
bit for bit, after the engine has put the bodies into key order, for single
systems, systems of a batch (offset slots) and skipped arrays."""
import ctypes as C

import numpy as np
import pytest

from next_amd import ic
from next_amd.nbx import MODE_PHYSICS, PREC_MIXED, Engine, lib

pytestmark = pytest.mark.gpu

CHUNK = 65536                           # from four chunks on; below, chunks of SMALL bodies
SMALL = 16384


def bodies(n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return ic.Particles(*(rng.normal(size=n) for _ in range(6)), np.full(n, 1.0 / n), np.zeros(n, np.int32))


def columns(p):
    return np.stack([p.x, p.y, p.z, p.vx, p.vy, p.vz])


@pytest.mark.parametrize("n", [1, 2, 255, SMALL - 1, SMALL, SMALL + 1, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK,
                               3 * CHUNK + 5, 4 * CHUNK - 1, 4 * CHUNK, 4 * CHUNK + 1, 7 * CHUNK + 3])
def test_upload_order(n):
    p = bodies(n, n)
    with Engine(theta=0.9) as e:
        e.upload(p)
        e.accel()                       # reorders the bodies
        assert np.array_equal(e.download(), columns(p))


def test_batch_offsets_and_removal():
    ps = [bodies(n, n) for n in (3, CHUNK + 7, 1, 2 * CHUNK)]
    with Engine(mode=MODE_PHYSICS, precision=PREC_MIXED, theta=0.9, adaptive_dt=False) as e:
        e.upload_batch(ps)
        e.accel()
        for s, p in enumerate(ps):
            assert np.array_equal(e.download_system(s), columns(p)), s
        assert np.array_equal(e.remove_system(1), columns(ps[1]))
        rest = [ps[0], ps[2], ps[3]]
        for s, p in enumerate(rest):
            assert np.array_equal(e.download_system(s), columns(p)), s
        assert np.array_equal(e.download(), np.concatenate([columns(p) for p in rest], axis=1))


def test_skipped_arrays():
    n = CHUNK + 3
    p = bodies(n, 9)
    fn = C.CDLL(lib()._name).nbx_download
    fn.argtypes = [C.c_void_p] * 7
    with Engine(theta=0.9) as e:
        e.upload(p)
        e.accel()
        y, vz = np.full(n, -7.0), np.full(n, -7.0)
        assert fn(e._h, None, y.ctypes.data, None, None, None, vz.ctypes.data) == 0
        assert np.array_equal(y, p.y) and np.array_equal(vz, p.vz)
        assert fn(e._h, None, None, None, None, None, None) == 0


@pytest.mark.parametrize("n", [4 * CHUNK, 4 * CHUNK + 1])
def test_skipped_arrays_with_helping_threads(n):
    """From four chunks on: every output null (the documented way to skip
    them), or one array only; then the system is removed without its state."""
    p = bodies(n, n)
    L = C.CDLL(lib()._name)
    vp = C.c_void_p
    L.nbx_download.argtypes = [vp] * 7
    L.nbx_download_system.argtypes = [vp, C.c_int32] + [vp] * 6
    L.nbx_remove_system.argtypes = [vp, C.c_int32] + [vp] * 6
    with Engine(theta=0.9) as e:
        e.upload(p)
        e.accel()
        assert L.nbx_download(e._h, *[None] * 6) == 0
        assert L.nbx_download_system(e._h, 0, *[None] * 6) == 0
        x, vy = np.full(n, -7.0), np.full(n, -7.0)
        assert L.nbx_download(e._h, x.ctypes.data, *[None] * 5) == 0
        assert L.nbx_download_system(e._h, 0, None, None, None, None, vy.ctypes.data, None) == 0
        assert np.array_equal(x, p.x) and np.array_equal(vy, p.vy)
        assert L.nbx_remove_system(e._h, 0, *[None] * 6) == 0
        assert e.num_systems() == 0


def test_direct_without_outputs():
    n = 4 * CHUNK
    L = C.CDLL(lib()._name)
    L.nbx_direct.argtypes = [C.c_void_p] * 5
    with Engine(eps=0.01) as e:
        e.upload(bodies(n, 5))
        pot = np.full(n, 7.0)
        assert L.nbx_direct(e._h, *[None] * 4) == 0
        assert L.nbx_direct(e._h, None, None, None, pot.ctypes.data) == 0
        assert np.all(pot < 0.0)
