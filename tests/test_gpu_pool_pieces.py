"""Pooled gradients of slots whose lookups take the reduction's workgroup one, two, three or four turns, and whose sums are cut into
pieces of four, eight or sixteen places: lengths on, before and behind each of these; a sign's lookups within a piece, over two and
over all of them.  Sums exact in 32 bits in any order (small multiples of 2^-8; examples of 1, 2 or 4 lookups)."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, dev, kernels_of
from test_gpu_small_edges import HP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [3, 16, 36])
@pytest.mark.parametrize("lens", [[1, 2, 5, 15, 16, 17], [63, 64, 65, 127, 128, 129], [511, 512, 513, 600], [1023, 1024, 1000, 900],
                                  [1025, 2047, 2048, 1537], [1535, 1536, 3071, 3073]])
def test_pieces(tn, oracle, dim, lens):
    rng = np.random.default_rng(sum(lens) + dim)
    pair = Pair(tn, oracle, "AdaGrad", dim, HP, reserve=100000)
    pool = synth.splitmix64(np.arange(1, 5001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    batch = max(lens)
    for kind in range(3):
        values, examples = [], []
        for n in lens:
            if kind == 0:    # distinct signs
                v = rng.permutation(pool)[:n]
            elif kind == 1:  # a sign with half of the lookups, some with a few
                v = np.where(rng.random(n) < 0.5, pool[3], pool[rng.integers(0, max(1, n // 3), n)])
            else:            # one sign
                v = np.repeat(pool[:1], n)
            values.append(v)
            examples.append(np.repeat(np.arange(n), np.resize([1, 4, 2, 2, 1], n))[:n].astype(np.int64))
        gm, gv, cm, cv, counts = pair.pull_op(values)
        pooled = [(rng.integers(-8, 9, (batch, dim)) / 256).astype(np.float32) for _ in values]
        labels = [rng.integers(0, 2, n).astype(np.int64) for n in lens]
        grads = [C.combine_backward(cm[s], examples[s], pooled[s], batch, C.SUM, int(counts[s])) for s in range(len(lens))]
        assert pair.o.push_op(values, grads, labels)[0] == 0
        names = kernels_of(tn, lambda: tn.ops.sparse_table_push_pooled(
            [dev(v) for v in values], [dev(e) for e in examples], [dev(p) for p in pooled], [dev(l) for l in labels], pair.h, "sum"))
        assert any(k.startswith("k_small_pool") for k in names)
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(all_signs(values))
