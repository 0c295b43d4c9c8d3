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
