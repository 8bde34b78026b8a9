"""The reduction of pooled gradients by parts of a slot (k_lookup_keys, k_reduce_pooled) at the sizes where it changes its
work: one part and two, the first slot whose frequent signs are spread over its parts, a part of one round of lookups and
one more, examples with as many lookups as an item has bits for, slots of very different lengths, rows of one and of several
runs of sixteen elements.  Sums are exact in 32 bits in any order (test_gpu_pooled_edges.py says why)."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, dev
from test_gpu_pooled_edges import NAMES, by_counts
from test_gpu_small_edges import HP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,lens", [
    (16, [1600, 1601, 1]), (12, [6403, 6404, 0, 3]), (4, [2048, 2049, 4097]),  # 1 / 2 parts, 4 / 8, one round and two
    (20, [12801, 70]), (64, [7000, 7000]), (8, [60000] + [5] * 40), (3, [9000, 1, 9000])])
@pytest.mark.parametrize("kind", ["few signs", "one sign", "distinct", "long examples"])
def test_parts_of_slots(tn, oracle, dim, lens, kind):
    rng = np.random.default_rng(dim * 7 + len(kind))
    pair = Pair(tn, oracle, "AdaGrad", dim, HP, reserve=400000)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    pool = synth.splitmix64(np.arange(1, max(lens) + 2, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    batch = max(lens) + 5
    values, examples = [], []
    for n in lens:
        if kind == "distinct":
            v = rng.permutation(pool[:n])
        elif kind == "one sign":
            v = np.repeat(pool[:1], n)
        else:
            v = pool[np.minimum(rng.geometric(0.01, n), len(pool)) - 1]
            v[rng.random(n) < 0.3] = pool[0]
        if kind == "long examples":  # (what is left at the end: one lookup each, so that all divide by powers of two)
            e = by_counts([2048, 1024, 1, 4096, 2], n)
            if n:
                tail = int((e == e[-1]).sum())
                e[n - tail:] = e[-1] + np.arange(tail)
        else:
            e = by_counts([1, 2, 4], n // 7 * 7) if n >= 7 else np.arange(n, dtype=np.int64)
            v = v[:len(e)]
        values.append(v)
        examples.append(e)
    pulled = pair.pull_op(values)
    cm, counts = pulled[2], pulled[4]
    combiner = C.SUM if kind == "one sign" else C.MEAN
    pooled = [(rng.integers(-8, 9, (batch, dim)) / 256).astype(np.float32) for _ in values]
    labels = [rng.integers(0, 2, len(v)).astype(np.int64) for v in values]
    grads = [C.combine_backward(cm[s], examples[s], pooled[s], batch, combiner, int(counts[s])) for s in range(len(lens))]
    assert pair.o.push_op(values, grads, labels)[0] == 0
    tn.ops.sparse_table_push_pooled([dev(v) for v in values], [dev(e) for e in examples], [dev(p) for p in pooled],
                                    [dev(l) for l in labels], pair.h, NAMES[combiner])
    tn.ops.sparse_table_sync(pair.h)
    assert pair.assert_rows_match(all_signs(values)) > 0.99
