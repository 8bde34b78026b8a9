"""Batches of more slots than two words of a slot mask have bits, on the large-batch path, up to and beyond the 255 slots
that are grouped through LDS: signs in every slot, in the slots around the words' edges, in one."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull

pytestmark = pytest.mark.gpu
HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


@pytest.mark.parametrize("slots,opt,dim", [(128, "AdaGrad", 8), (129, "AdaGrad", 8), (193, "AdaGrad", 16), (255, "AdaGrad", 16),
                                           (255, "Adam", 12), (256, "AdaGrad", 8)])
def test_signs_of_all_slots(tn, oracle, slots, opt, dim):
    rng = np.random.default_rng(slots + dim)
    hyper = HP if opt == "AdaGrad" else dict(learning_rate=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8)
    pair = Pair(tn, oracle, opt, dim, hyper, reserve=200000, zero_init=True)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    pool = synth.splitmix64(np.arange(1, 30001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool[:20000].view(np.uint64))
    edges = [s for s in (0, 63, 64, 127, 128, 191, 192, slots - 1) if s < slots]
    for step in range(3):
        values = []
        for s in range(slots):
            v = pool[rng.integers(100, 20000 if step == 0 else 30000, int(rng.integers(90, 200)))]
            v[:12] = np.tile(pool[:4], 3)
            if s in edges:
                v[12:15] = pool[4:7]
            if s == slots // 2:
                v[15] = -1  # the sign that marks a free entry
            values.append(rng.permutation(v))
        counts = check_pull(pair, values)
        grads = synth.make_grads(counts, dim, 0.05, seed=step)
        pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values])
        assert pair.assert_rows_match(all_signs(values)) > 0.99
