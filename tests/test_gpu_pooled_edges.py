"""Pooled gradients of batches with a slot of more lookups than the small path takes: examples that end at, before and
behind the 64 lookups a wavefront looks at, that go on over several of them and take a whole slot; signs with few, many and
all lookups of a slot; rows of any length.

The examples have powers of two of lookups and the gradients are small multiples of 2^-8: the sums of the lookups of a sign,
divided or not, are exact in 32 bits in any order (at most 20 bits are in use), so the order in which long sums are added
makes no difference."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, dev
from test_gpu_small_edges import HP

pytestmark = pytest.mark.gpu
NAMES = {C.SUM: "sum", C.MEAN: "mean", C.SQRTN: "sqrtn"}


def by_counts(counts, n):
    """Example ids of n lookups: example i has counts[i % len(counts)] of them."""
    return np.repeat(np.arange(n), np.resize(counts, n))[:n].astype(np.int64)


@pytest.mark.parametrize("dim,slots,n", [(16, 5, 9000), (10, 5, 5001), (1, 3, 4097), (130, 5, 6000), (8, 130, 4160), (4, 3, 150000)])
def test_pooled_push_of_a_large_batch(tn, oracle, dim, slots, n):
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, "AdaGrad", dim, HP, reserve=200000)
    pool = synth.splitmix64(np.arange(1, 3000, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    values, examples = [], []
    for s in range(slots):
        m = n if s < 5 else 70 + s
        kind = s % 5
        if kind == 0:    # every sign a few times, a frequent one; examples of 32, 64, 1, 128, 2, 256 lookups
            m -= m % 484
            v, e = pool[rng.integers(0, 2999, m)], by_counts([32, 64, 1, 128, 2, 256, 1], m)
            v[rng.random(m) < 0.2] = pool[7]
        elif kind == 1:  # one example, one sign
            m = 1 << (m.bit_length() - 1)
            v, e = np.repeat(pool[:1], m), np.full(m, n - 1, np.int64)
        elif kind == 2:  # 64 .. 1023 lookups a sign, one lookup an example
            v, e = pool[np.minimum(rng.geometric(0.02, m), 2999) - 1], np.arange(m, dtype=np.int64)
        elif kind == 3:  # distinct signs
            m = min(m, 2998) & ~1
            v, e = pool[:m][rng.permutation(m)], np.repeat(np.sort(rng.permutation(n)[:m // 2]), 2)
        else:            # no lookups
            v, e = pool[:0], np.zeros(0, np.int64)
        values.append(v)
        examples.append(e)
    for combiner in (C.MEAN, C.SUM):
        gm, gv, cm, cv, counts = pair.pull_op(values)
        pooled = [(rng.integers(-8, 9, (n, dim)) / 256).astype(np.float32) for _ in values]
        labels = [rng.integers(0, 2, len(v)).astype(np.int64) for v in values]
        grads = [C.combine_backward(cm[s], examples[s], pooled[s], n, combiner, int(counts[s])) for s in range(slots)]
        assert pair.o.push_op(values, grads, labels)[0] == 0
        tn.ops.sparse_table_push_pooled([dev(v) for v in values], [dev(e) for e in examples], [dev(p) for p in pooled],
                                        [dev(l) for l in labels], pair.h, NAMES[combiner])
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(all_signs(values))
