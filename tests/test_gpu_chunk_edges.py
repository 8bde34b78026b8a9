"""Signs with as many records as a chunk of the few-launch path's update kernel holds, one less, one more, and two chunks and one:
the rows whose chunks are four rounds (sixteen records of rows of 16, eight of rows of 32)."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, kernels_of

pytestmark = pytest.mark.gpu

HP = {"Adam": dict(learning_rate=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8),
      "Ftrl": dict(learning_rate=0.05, beta=1.0, lambda1=0.001, lambda2=1.0)}


@pytest.mark.parametrize("opt,dim", [("Adam", 16), ("Adam", 32), ("Ftrl", 32)])
@pytest.mark.parametrize("slots", [15, 16, 17, 33])
def test_signs_of_a_chunk(tn, oracle, opt, dim, slots):
    rng = np.random.default_rng(dim * 100 + slots)
    pool = synth.splitmix64(np.arange(1, 601, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, opt, dim, HP[opt], reserve=20000, zero_init=True)
    pair.populate(pool.view(np.uint64))
    # every number of records from the slots' down to one, and signs of one slot
    values = [np.concatenate([pool[s:slots], pool[40 + 10 * s:50 + 10 * s]]) for s in range(slots)]
    for step in range(2):
        counts = []
        assert "k_small_slots" in kernels_of(tn, lambda: counts.append(check_pull(pair, values)))
        grads = synth.make_grads(counts[0], dim, 0.01, seed=step)
        pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values])
        assert pair.assert_rows_match(all_signs(values)) > 0.99
