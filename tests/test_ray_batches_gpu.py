"""Ray batches at the edges of the trace kernels' work distribution: one ray,
the 64 rays of a batch, one batch per persistent wave, and more.  A ray's hit
does not depend on the batch it is in, so every batch is compared bit for bit
with the same rays asked in blocks of 1000; the blocks' rays against the
oracle."""
import time

import numpy as np
import pytest

import raymond_amd.api as api
import raymond_amd.scenes as scenes
from oracle import binding
from tests.parity import ORACLE_THREADS, assert_hits_equal
from tests.test_gpu_parity import random_rays
from tests.test_zz_no_alloc import Hip, noalloc_trace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[False, True], ids=["flat", "two-level"])
def traced(device, request):
    desc = scenes.sphere_field(96, 54, grid=2, level=3)
    desc.envmap_resolution = 64
    scene = api.Scene(device, desc)
    scene.build_accel(two_level=request.param)
    rays = random_rays(400000, -2.0, 2.0, 5, tmin=1e-3, tmax=3.0)
    parts = [scene.trace_closest(rays[i:i + 1000]) for i in range(0, 400000, 1000)]
    closest = tuple(np.concatenate([p[k] for p in parts]) for k in range(4))
    occluded = np.concatenate([scene.trace_any(rays[i:i + 1000]) for i in range(0, 400000, 1000)])
    orc = binding.OracleScene(desc)
    if request.param:
        orc.set_two_level(True)
    assert_hits_equal(tuple(x[:2000] for x in closest), orc.trace_closest(rays[:2000], threads=ORACLE_THREADS))
    assert np.array_equal(occluded[:2000], orc.trace_any(rays[:2000], threads=ORACLE_THREADS))
    return scene, rays, closest, occluded


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4097, 16383, 52428, 52429, 81921, 262143, 327679, 327681, 400000])
def test_batches_agree_at_every_size(traced, n):
    scene, rays, closest, occluded = traced
    got = scene.trace_closest(rays[:n])
    for g, c in zip(got, closest):
        assert np.array_equal(g.view(np.uint32), c[:n].view(np.uint32))
    assert np.array_equal(scene.trace_any(rays[:n]), occluded[:n])
    if n <= 1 << 18:
        hip = Hip()
        try:
            got = noalloc_trace(hip, scene, rays[:n])
        finally:
            hip.free()
        for g, c in zip(got, closest):
            assert np.array_equal(g.view(np.uint32), c[:n].view(np.uint32))


def test_hit_arrays_may_overlap_the_rays(traced):
    """Hits written over the device rays they came from."""
    scene, rays, closest, _ = traced
    n = 5000
    hip = Hip()
    try:
        buf = hip.upload(rays[:n])
        scene.trace_closest_noalloc(buf, n, buf, buf + 4 * n, buf + 8 * n, buf + 16 * n)
        hip.sync()
        got = (hip.download(buf, n, np.float32), hip.download(buf + 4 * n, n, np.uint32),
               hip.download(buf + 8 * n, n, np.uint32), hip.download(buf + 16 * n, (n, 2), np.float32))
    finally:
        hip.free()
    for g, c in zip(got, closest):
        assert np.array_equal(g.view(np.uint32), c[:n].view(np.uint32))


def test_outputs_may_be_left_out(traced):
    """Any of closest hits' arrays may be null, on both sides of the size from
    which they are copied apart (52428 rays)."""
    scene, rays, closest, _ = traced
    for n in (100, 60000):
        r = np.ascontiguousarray(rays[:n])
        for keep in range(16):
            got = [np.full(c[:n].shape, 7, c.dtype) for c in closest]
            out = [g.ctypes.data if keep >> i & 1 else None for i, g in enumerate(got)]
            assert api.LIB.rm_trace_closest(scene.handle, r.ctypes.data, n, *out) == 0
            for i, (g, c) in enumerate(zip(got, closest)):
                assert np.array_equal(g, c[:n]) if keep >> i & 1 else np.all(g == 7)


def test_a_small_batch_costs_one_copy_back(traced):
    """Closest hits have four arrays, any hits one: with one ray, a call of the
    former that copies them apart takes twice as long as one of the latter
    (64 against 31 us), in one copy as long (32)."""
    scene = traced[0]
    away = np.array([[0.0, 0.0, 100.0, 1e-3, 0.0, 0.0, 1.0, 1.0]], np.float32)  # no traversal

    def least(call):
        best = np.inf
        for _ in range(300):
            t = time.perf_counter()
            call(away)
            best = min(best, time.perf_counter() - t)
        return best

    closest, any_hit = least(scene.trace_closest), least(scene.trace_any)
    print("closest %.1f us, any %.1f us" % (closest * 1e6, any_hit * 1e6))
    assert closest < 1.6 * any_hit
