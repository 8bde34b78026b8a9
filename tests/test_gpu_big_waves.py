"""Signs with many records under Adam and Ftrl on the large-batch path: rows of every power-of-two dim from 4 to 64, whose chunks are 4 to
64 records, signs of 15, 16, 17, 40 and 70 records; a dim that has no kernel of its own."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, kernels_of
from test_gpu_big_groups import batch
from test_gpu_chunk_edges import HP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opt", ["Adam", "Ftrl"])
@pytest.mark.parametrize("dim", [4, 8, 16, 32, 64, 12])
def test_signs_in_most_slots(tn, oracle, opt, dim):
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, opt, dim, HP[opt], reserve=200000, zero_init=True)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    pool = synth.splitmix64(np.arange(1, 26001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool[:20000].view(np.uint64))
    for step in range(2):
        values = batch(rng, pool, step)
        counts = check_pull(pair, values)
        grads = synth.make_grads(counts, dim, 0.05, seed=step)
        labels = [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values]
        assert any(k.startswith("k_apply_all") for k in kernels_of(tn, lambda: pair.push_op(values, grads, labels)))
        assert pair.assert_rows_match(all_signs(values)) > 0.99
