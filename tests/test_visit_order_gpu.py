"""Closest hits where the order of visits and the dropped node groups could
show: two instances of one shape in the same place (every hit is a tie), rays
along the axes, origins on vertices, and ranges that end or begin exactly at a
hit or one unit in the last place beside it.  Hits are those of the oracle,
bit for bit: they do not depend on the tree or on the order of visits."""
import numpy as np
import pytest

import raymond_amd.api as api
import raymond_amd.scenes as scenes
from oracle import binding
from tests.parity import ORACLE_THREADS, assert_hits_equal
from tests.test_gpu_parity import random_rays

pytestmark = pytest.mark.gpu


def stacked_field():
    desc = scenes.instanced_field(96, 54, grid=4, shapes=2, level=3)
    for k in range(3):
        desc.entities.append(desc.entities[k])
    desc.envmap_resolution = 64
    return desc


def order_rays(desc, n=3000):
    rays = random_rays(n, -3.0, 3.0, 12)
    rng = np.random.default_rng(13)
    verts = desc.arrays()[0]
    axis = np.zeros((n, 3), np.float32)
    axis[np.arange(n), rng.integers(0, 3, n)] = rng.choice([-1.0, 1.0], n)
    along = rays.copy()
    along[:, 4:7] = axis
    on_vertex = rays.copy()
    on_vertex[:, 0:3] = verts[rng.integers(0, len(verts), n)]
    return np.concatenate([rays, along, on_vertex])


@pytest.mark.parametrize("two_level", [False, True], ids=["flat", "two-level"])
def test_hits_do_not_depend_on_the_visit_order(device, two_level):
    desc = stacked_field()
    scene = api.Scene(device, desc)
    scene.build_accel(two_level=two_level)
    orc = binding.OracleScene(desc)
    if two_level:
        orc.set_two_level(True)

    def check(rays):
        hits = scene.trace_closest(rays)
        ref = orc.trace_closest(rays, threads=ORACLE_THREADS)
        assert_hits_equal(hits, ref, rays)
        return hits

    rays = order_rays(desc)
    t = check(rays)[0]
    hit = rays[t >= 0]
    t = t[t >= 0]
    assert len(hit) > 500
    for end in (t, np.nextafter(t, np.float32(np.inf)), np.nextafter(t, np.float32(0))):
        cut = hit.copy()
        cut[:, 7] = end
        check(cut)
        assert np.array_equal(scene.trace_any(cut), orc.trace_any(cut, threads=ORACLE_THREADS))
        cut[:, 3] = end
        cut[:, 7] = np.inf
        check(cut)
