"""AdaGrad rows that take the lanes of half a wavefront: the double sum over a gradient's squares goes on from one row of sixteen lanes to
the next, in element order.  Lengths of which the last lanes hold less than four elements or none, signs with one record to many, on
both paths."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull

from test_gpu_big_groups import ADAGRAD_HP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("few_launches", [True, False])
@pytest.mark.parametrize("dim", [64, 65, 68, 72, 100, 124, 127, 128])
def test_sums_of_squares(tn, oracle, dim, few_launches):
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, "AdaGrad", dim, ADAGRAD_HP, reserve=20000, zero_init=True)
    tn.core.set_sparse_table_small_batch_path(pair.h, few_launches)
    pool = synth.splitmix64(np.arange(1, 3001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool[:2500].view(np.uint64))
    for step in range(2):
        values = [np.concatenate([pool[s:40], pool[(rng.random(300) ** 2 * len(pool)).astype(np.int64)]]) for s in range(20)]
        counts = check_pull(pair, values)
        # elements of very different size: another order of the sum would show
        grads = [(rng.standard_normal((c, dim)) * 10.0 ** rng.uniform(-4, 0, (c, dim))).astype(np.float32) for c in counts]
        pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values])
        assert pair.assert_rows_match(all_signs(values)) > 0.999
