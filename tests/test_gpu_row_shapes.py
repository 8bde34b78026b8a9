"""Rows of any length share the update kernels' lanes out four elements each: lengths around every lane count, the last
part whole or not, gradients off a 16-byte boundary (the cvm columns), the longest row that is shared and one beyond."""
import numpy as np
import pytest

from helpers import Pair, all_signs, check_pull

pytestmark = pytest.mark.gpu

HYPER = {"AdaGrad": dict(learning_rate=0.05, initial_g2sum=0.1, epsilon=1e-8), "Adam": dict(learning_rate=1e-3),
         "Ftrl": dict(learning_rate=0.05, beta=1.0, lambda1=0.01, lambda2=1.0)}


@pytest.mark.parametrize("small_path", [True, False])
@pytest.mark.parametrize("opt,dim,cvm", [("AdaGrad", 1, False), ("AdaGrad", 5, False), ("AdaGrad", 10, True),
                                         ("AdaGrad", 8, True), ("AdaGrad", 128, True), ("AdaGrad", 130, False),
                                         ("Adam", 2, False), ("Adam", 7, False), ("Adam", 33, False), ("Adam", 127, False),
                                         ("Ftrl", 3, False), ("Ftrl", 20, False), ("Ftrl", 65, False), ("Ftrl", 129, False)])
def test_row_lengths(tn, oracle, opt, dim, cvm, small_path):
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, opt, dim, HYPER[opt], use_cvm=cvm, reserve=1 << 16)
    tn.core.set_sparse_table_small_batch_path(pair.h, small_path)
    # signs shared by up to 20 slots: one record, a few, many
    vocab = rng.integers(1, 1 << 62, 400, dtype=np.uint64)
    values = [vocab[rng.integers(0, 60 + 17 * s, 170)].view(np.int64) for s in range(20)]
    pair.populate(all_signs(values))
    for _ in range(2):
        counts = check_pull(pair, values, loose_col=dim + 1 if cvm else None)
        grads = [rng.standard_normal((int(u), pair.wf)).astype(np.float32) for u in counts]
        labels = [rng.integers(0, 2, len(v)) for v in values]
        pair.push_op(values, grads, labels)
        same = pair.assert_rows_match(all_signs(values))
        assert same > (0.9 if cvm else 0.95)  # (the log column follows the libm in use)
