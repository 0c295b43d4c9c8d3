"""Copies between the device and the caller's memory: staged ones (from 3 MB,
in slots of 8 MB, four of them in a ring) give the bytes that plain ones give,
at sizes around the slots, at odd addresses, into pinned memory, and from two
threads at once."""
import ctypes
import threading

import numpy as np
import pytest

import raymond_amd.api as api
import raymond_amd.scenes as scenes
from tests.test_gpu_parity import random_rays
from tests.test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

BLOCK = 5000


@pytest.fixture(scope="module")
def traced(device):
    desc = scenes.sphere_field(96, 54, grid=2, level=3)
    desc.envmap_resolution = 64
    scene = api.Scene(device, desc)
    scene.build_accel()
    rays = random_rays(BLOCK, -2.0, 2.0, 5, tmin=1e-3, tmax=3.0)
    return scene, rays, scene.trace_closest(rays), scene.trace_any(rays)


def tiled(a, n):
    return np.resize(a, (n,) + a.shape[1:])


def equal(got, want, n):
    for g, w in zip(got, want):
        assert np.array_equal(g.view(np.uint32), tiled(w, n).view(np.uint32))


# rays of 32 bytes and hits of 20: one slot of rays at 262144, of hits at
# 419430, the ring of rays at 1048576, of hits at 1677721
@pytest.mark.parametrize("n", [98303, 98305, 157287, 262143, 262145, 419431, 786433, 1048577, 1700001])
def test_staged_batches(traced, n):
    scene, rays, closest, occluded = traced
    r = tiled(rays, n)
    equal(scene.trace_closest(r), closest, n)
    assert np.array_equal(scene.trace_any(r), tiled(occluded, n))


@pytest.mark.parametrize("offset", [4, 12, 4092])
@pytest.mark.parametrize("pinned", [False, True], ids=["pageable", "pinned"])
def test_odd_addresses_and_pinned_memory(traced, offset, pinned):
    scene, rays, closest, _ = traced
    n = 300001
    sizes = [32 * n, 4 * n, 4 * n, 4 * n, 8 * n]
    if pinned:
        hip = Hip().lib
        ptrs = [ctypes.c_void_p() for _ in sizes]
        for p, size in zip(ptrs, sizes):
            assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size + offset), 0) == 0
        bufs = [np.ctypeslib.as_array((ctypes.c_uint8 * (size + offset)).from_address(p.value))
                for p, size in zip(ptrs, sizes)]
    else:
        bufs = [np.zeros(size + offset, np.uint8) for size in sizes]
    a = [b[offset:] for b in bufs]
    a[0][:] = tiled(rays, n).reshape(-1).view(np.uint8)
    api._check(api.LIB.rm_trace_closest(scene.handle, ctypes.c_void_p(a[0].ctypes.data), n,
                                        *[ctypes.c_void_p(x.ctypes.data) for x in a[1:]]))
    types = [np.float32, np.uint32, np.uint32, np.float32]
    got = [np.frombuffer(x.tobytes(), t) for x, t in zip(a[1:], types)]
    got[3] = got[3].reshape(n, 2)
    if pinned:
        for p in ptrs:
            assert hip.hipHostFree(p) == 0
    equal(got, closest, n)


def test_two_threads(traced):
    """The second copy at a time goes the plain way."""
    scene, rays, closest, _ = traced
    failed = []

    def work(n):
        try:
            for _ in range(3):
                equal(scene.trace_closest(tiled(rays, n)), closest, n)
        except BaseException as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in (700001, 500001)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def test_parameters_there_and_back(device):
    cache = api.RadianceCache(device, log2_table_size=16)
    rng = np.random.default_rng(3)
    mlp, table = cache.read_params()
    table = rng.standard_normal(table.size).astype(np.float32)
    cache.write_params(mlp, table)
    got_mlp, got = cache.read_params()
    assert np.array_equal(got_mlp, mlp) and np.array_equal(got, table)
