"""The bounce loop's launches: closest hits merged with the previous bounce's
shadow rays against separate launches (timing=1), streams that fit the queue
(no regeneration, a known last iteration) and streams that do not, depths
around the loop's chunks of iterations, against the oracle; two-level trees,
lens rays, batches and caches against their separate launches; job times."""
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


@pytest.fixture(scope="module")
def kinds(device, cornell):
    field = scenes.instanced_field(W, H, grid=4, shapes=3, level=2)
    lamps = scenes.lamp_box(W, H)
    for d in (field, lamps):
        d.envmap_resolution = 64
    return {"two-level": scenes.build_device_scene(device, field, two_level=True),
            "lens": scenes.build_device_scene(device, lamps), "cornell": cornell[0]}


@pytest.mark.parametrize("kind", ["two-level", "lens"])
@pytest.mark.parametrize("spl,samples", [(5, 5), (2, 5)], ids=["fits", "regenerates"])
def test_two_level_and_lens_launches(kinds, kind, spl, samples):
    """The merged launch, direct and from a captured graph, against the
    separate ones: the same rays at every depth, the same image up to the
    order of its sums."""
    ref = None
    for timing, graph in ((1, 0), (0, 0), (0, 1)):
        r = api.Renderer(kinds[kind], W, H, max_depth=9, samples_per_launch=spl)
        if kind == "lens":
            r.set_lens(api.lens_desc(scenes.singlet_lens(50.0, 2.8), stop_index=3, relative_stop=0.7,
                                     camera_scale=0.01, spectral=True))
        r.set_uniforms(timing=timing, use_graph=graph, rr_depth=64, material_sort=1)
        st = r.execute(samples)
        got = (list(st.rays), list(st.shadow_rays), st.total_rays), r.image()
        assert st.shadow_total > 0
        ref = ref or got
        assert got[0] == ref[0]
        parity.assert_radiance_close(got[1], ref[1])


@pytest.mark.parametrize("queue,graph", [(0, 0), (2048, 0), (0, 1), (2048, 1)])
def test_batch_launches(device, kinds, queue, graph):
    """Jobs of several depths in a queue that holds them and in one that does not."""
    scene = kinds["cornell"]
    b = api.Batch(device, [(scene, 40, 24, 3, 9, 1), (scene, 24, 32, 7, 1, 2), (scene, 33, 17, 2, 20, 3)])
    st = b.render(queue_paths=queue, rr_depth=3, timing=1)
    ref = [b.image(j) for j in range(3)]
    got = b.render(queue_paths=queue, rr_depth=3, use_graph=graph)
    assert (got.closest_rays, got.shadow_rays) == (st.closest_rays, st.shadow_rays)
    for j in range(3):
        parity.assert_radiance_close(b.image(j), ref[j])
    t = b.job_times()
    assert np.all(t > 0.0) and got.makespan_ms == t.max() <= got.ms_total


@pytest.mark.parametrize("spl", [8, 2], ids=["fits", "regenerates"])
def test_cache_launches(device, kinds, spl):
    """A training cache sees the same vertices; with fixed parameters the
    frames through it are the same."""
    counts, images = [], []
    for timing in (1, 0):
        c = api.RadianceCache(device, log2_table_size=12, seed=3, train_shift=2, batch_size=256)
        r = api.Renderer(kinds["cornell"], W, H, max_depth=9, samples_per_launch=spl)
        r.set_uniforms(timing=timing, rr_depth=64, material_sort=1)
        r.set_cache(c, mode=1)
        r.execute(8)
        s = c.stats()
        counts.append((s.queries, s.train_records, s.samples, s.steps))
        assert np.isfinite(s.last_loss) and min(counts[-1]) > 0
        c = api.RadianceCache(device, log2_table_size=12, seed=3)
        r = api.Renderer(kinds["cornell"], W, H, max_depth=9, samples_per_launch=spl)
        r.set_uniforms(timing=timing, rr_depth=64, material_sort=1)
        r.set_cache(c, mode=2)
        r.execute(8)
        images.append(r.image())
    assert counts[0] == counts[1]
    parity.assert_radiance_close(images[1], images[0])
