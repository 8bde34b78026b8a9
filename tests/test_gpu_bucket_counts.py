"""Batches of the few-launch path around the size from which its buckets hold more lookups: as many buckets as before, one lookup
over, a bucket for so many lookups, slots so many that the buckets' LDS asks for smaller ones; spread signs and frequent ones."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots,lookups,dim", [(16, 4096, 8), (17, 3856, 8), (24, 8192, 16), (40, 5000, 40), (100, 2000, 4), (200, 500, 8),
                                               # parts of slots that do not divide the buckets; fewer of them where rows are wide
                                               (20, 6500, 16), (20, 5494, 40), (20, 8192, 64)])
def test_larger_buckets(tn, oracle, slots, lookups, dim):
    rng = np.random.default_rng(slots + lookups)
    pool = synth.splitmix64(np.arange(1, 60001, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", dim, dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8), reserve=200000, zero_init=True)
    pair.populate(pool[:50000].view(np.uint64))
    for step in range(2):
        frac = rng.random((slots, lookups)) ** (1 if step == 0 else 4)  # distinct for the most part; then a third of them frequent
        values = [pool[(f * len(pool)).astype(np.int64)] for f in frac]
        counts = []
        assert any(k.startswith("k_small_slots") for k in kernels_of(tn, lambda: counts.append(check_pull(pair, values))))
        grads = synth.make_grads(counts[0], dim, 0.01, seed=step)
        names = kernels_of(tn, lambda: pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values]))
        assert any(k.startswith("k_small_apply") for k in names) and "k_remap_insert" not in names  # (no bucket overflowed)
        assert pair.assert_rows_match(all_signs(values)) > 0.99


@pytest.mark.parametrize("slots,lookups", [(20, 4700), (20, 5300), (20, 8100)])
def test_buckets_of_distinct_signs(tn, oracle, slots, lookups):
    """Nearly as many signs as records: the buckets' tables are as full as they get."""
    rng = np.random.default_rng(lookups)
    pool = synth.splitmix64(np.arange(1, slots * lookups + 1, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", 4, dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8), reserve=400000, zero_init=True)
    pair.populate(pool.view(np.uint64))
    for _ in range(2):
        values = list(rng.permutation(pool).reshape(slots, lookups))
        values[1][:50] = values[0][:50]
        counts = check_pull(pair, values)
        grads = synth.make_grads(counts, 4, 0.01)
        names = kernels_of(tn, lambda: pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values]))
        assert any(k.startswith("k_small_apply") for k in names) and "k_remap_insert" not in names
        assert pair.assert_rows_match(all_signs(values)) > 0.99
