"""The bounce loop's launches: closest hits merged with the previous bounce's
shadow rays against separate launches (timing=1), streams that fit the queue
(no regeneration, a known last iteration) and streams that do not, depths
around the loop's chunks of iterations, against the oracle."""
import numpy as np
import pytest

import raymond_amd.api as api
import raymond_amd.scenes as scenes
from oracle import binding
from tests import parity

pytestmark = pytest.mark.gpu

W, H = 40, 24


@pytest.fixture(scope="module")
def cornell(device):
    desc = scenes.cornell_box(W, H)
    desc.envmap_resolution = 64
    orc = binding.OracleScene(desc)
    orc.build_envmap(threads=4)
    return scenes.build_device_scene(device, desc), orc


@pytest.mark.parametrize("depth", [1, 2, 7, 8, 9, 13, 20])
@pytest.mark.parametrize("spl,samples", [(4, 3), (1, 4)], ids=["fits", "regenerates"])
def test_depths_and_launches(cornell, depth, spl, samples):
    scene, orc = cornell
    ref, res = orc.render(W, H, depth, frames=samples, frame_begin=0, rr_depth=64, threads=parity.ORACLE_THREADS)
    for timing in (0, 1):
        for sort in (0, 1):
            r = api.Renderer(scene, W, H, max_depth=depth, samples_per_launch=spl)
            r.set_uniforms(timing=timing, material_sort=sort, rr_depth=64)
            st = r.execute(samples)
            assert st.total_rays == res.total_rays
            assert st.shadow_total == sum(res.shadow_rays[d] for d in range(32))
            parity.assert_radiance_close(r.image(), ref)


def test_job_times_include_the_last_shadow_rays(device):
    """A job is complete when its shadow rays are: its time is not read before
    they are traced.  In a closed room of albedo 2e-6 the weight of a path
    underflows to zero (2e-6^8 = 2.6e-46) in the shading of iteration 7, the
    last of the first chunk that the host checks: every path ends there, a
    third of them with a shadow ray, whose launch takes 0.4 ms.  The launches
    after it are empty."""
    desc = scenes.tessellated_cornell_box(256, 256, 200000)
    desc.envmap_resolution = 64
    desc.surface_materials = [scenes.diffuse_material("dark", (2e-6, 2e-6, 2e-6))] * 4 + [
        scenes.emission_material("light", (1.0, 1.0, 1.0), 1e6)]
    lo, hi = -3.0, 4.0
    c = [(x, y, z) for x in (lo, hi) for y in (lo, hi) for z in (lo, hi)]
    desc.add_entity(desc.add_shape(scenes.merge(
        [scenes.quad(*(c[k] for k in q), 0) for q in ((0, 2, 6, 4), (1, 5, 7, 3), (0, 4, 5, 1), (2, 3, 7, 6),
                                                      (0, 1, 3, 2), (4, 6, 7, 5))])))
    scene = scenes.build_device_scene(device, desc)
    b = api.Batch(device, [(scene, 256, 256, 60, 12, 1)])
    st = b.render(rr_depth=64, timing=1)
    assert st.iterations >= 8 and st.ms_trace_any > 1.0
    launch = st.ms_trace_any / 8
    gaps = []
    for _ in range(5):
        st = b.render(rr_depth=64)
        assert b.job_times()[0] == st.makespan_ms
        gaps.append(st.ms_total - st.makespan_ms)
    print("from the job's time to the end %.3f ms, shadow rays of an iteration %.3f ms" % (min(gaps), launch))
    assert min(gaps) < 0.5 * launch
