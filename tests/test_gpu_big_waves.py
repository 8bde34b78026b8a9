"""Signs with many records on the large-batch path: under Adam and Ftrl rows of every power-of-two dim to 64, under AdaGrad those of 1 and
2, whose chunks are 4 to 64 records, signs of 15, 16, 17, 40 and 70 records; a dim that has no kernel of its own."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, kernels_of
from test_gpu_big_groups import ADAGRAD_HP, batch
from test_gpu_chunk_edges import HP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opt,dim,cvm", [(opt, dim, False) for opt in ("Adam", "Ftrl") for dim in (1, 2, 4, 8, 16, 32, 64, 12)] +
                         [("AdaGrad", 1, False), ("AdaGrad", 2, False), ("AdaGrad", 1, True), ("AdaGrad", 2, True)])
def test_signs_in_most_slots(tn, oracle, opt, dim, cvm):
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, opt, dim, HP.get(opt, ADAGRAD_HP), use_cvm=cvm, reserve=200000, zero_init=True)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    pool = synth.splitmix64(np.arange(1, 26001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool[:20000].view(np.uint64))
    for step in range(2):
        values = batch(rng, pool, step)
        counts = check_pull(pair, values, loose_col=(dim + 1) if cvm else None)
        grads = synth.make_grads(counts, pair.wf, 0.05, seed=step)
        labels = [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values]
        applied = [k for k in kernels_of(tn, lambda: pair.push_op(values, grads, labels)) if k.startswith("k_apply_all<")]
        # (", 0>": the kernel whose signs with many records go through LDS record by record, whatever the row's length)
        assert [k.endswith(", 0>") for k in applied] == [dim == 12 or opt == "Ftrl" and dim == 64]
        # (with cvm one of the dim + 2 columns is a logarithm, which follows the libm in use)
        assert pair.assert_rows_match(all_signs(values)) > 0.99 * ((dim + 1) / (dim + 2) if cvm else 1)
