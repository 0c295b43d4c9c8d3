"""Raw cache batches at the edges of the kernels' 32-sample tiles: row-major
inputs and outputs, staging buffers kept from a larger batch, and table
gradients that are cleared as they are read."""
import numpy as np
import pytest

import raymond_amd.api as api
from oracle import binding
from tests.test_rcache_cpu import numpy_gradients, random_features, random_params
from tests.test_rcache_gpu import check_gradients, rel_l2

pytestmark = pytest.mark.gpu

LOG2 = 12


@pytest.mark.parametrize("n", [1, 31, 32, 33, 129, 17476, 17477])
def test_rows_at_tile_edges(device, n):
    rng = np.random.default_rng(n)
    mlp, table = random_params(rng, LOG2)
    c = api.RadianceCache(device, log2_table_size=LOG2, seed=1)
    c.write_params(mlp, table)
    big = random_features(rng, 300)
    big_t = rng.uniform(0, 1, (300, 3)).astype(np.float32)
    c.infer(big)  # the buffers keep this batch's size
    f = random_features(rng, n)
    y = binding.rc_forward(LOG2, mlp, table, f)
    # the forward bound of test_rcache_gpu (FP16 encodings and activations)
    assert rel_l2(c.infer(f), y) < 1e-2
    t = (y + rng.normal(size=y.shape) * 0.5).astype(np.float32)
    rm, rt, rloss = binding.rc_gradients(LOG2, mlp, table, f, t)
    half = numpy_gradients(LOG2, mlp, table, f, t, fp16=True)
    # after another batch's gradients, whether or not its table gradients were
    # read: nothing of them is left in the sums of the weights, the table or
    # the loss
    for read_table in (True, False):
        c.gradients(big, big_t, table=read_table)
        gm, gt, loss = c.gradients(f, t)
        assert abs(loss - rloss) < 1e-2 * rloss
        check_gradients(gm, gt, rm, rt, half)
