"""Pooled gradients of slots beyond the path of few launches whose examples end at, before and behind the runs of 64 lookups, the 512
of a wavefront and the 64 on either side of them, and go on over several of any: extents are read off all of these."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, dev, kernels_of
from test_gpu_small_edges import HP

pytestmark = pytest.mark.gpu


# lookups of the examples in turn, powers of two: the sums of small multiples of 2^-8 are exact in any order, divided or not
@pytest.mark.parametrize("lens", [[1], [64], [32, 64], [512], [1, 512], [1024, 1, 2], [64, 1, 2, 1], [2048, 256, 1], [8192, 1]])
@pytest.mark.parametrize("n", [8193, 8704, 9216 + 63, 9280 + 1])
def test_extents(tn, oracle, lens, n):
    rng = np.random.default_rng(n + len(lens) + lens[0])
    dim = 4
    pair = Pair(tn, oracle, "AdaGrad", dim, HP, reserve=50000)
    pool = synth.splitmix64(np.arange(1, 4001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    # (what is left of a slot for less than an example of the turn: one lookup an example)
    def examples(m):
        counts = []
        while sum(counts) < m:
            c = lens[len(counts) % len(lens)]
            counts.append(c if sum(counts) + c <= m else 1)
        return np.repeat(np.arange(len(counts)), counts).astype(np.int64)

    ids = [examples(m) for m in (n, n - 1, 700)]
    values = [pool[rng.integers(0, len(pool), len(e))] for e in ids]
    batch = max(int(e[-1]) for e in ids) + 1
    _, _, cm, _, counts = pair.pull_op(values)
    pooled = [(rng.integers(-8, 9, (batch, dim)) / 256).astype(np.float32) for _ in values]
    labels = [rng.integers(0, 2, len(v)).astype(np.int64) for v in values]
    grads = [C.combine_backward(cm[s], ids[s], pooled[s], batch, C.MEAN, int(counts[s])) for s in range(len(ids))]
    assert pair.o.push_op(values, grads, labels)[0] == 0
    names = kernels_of(tn, lambda: tn.ops.sparse_table_push_pooled(
        [dev(v) for v in values], [dev(e) for e in ids], [dev(p) for p in pooled], [dev(l) for l in labels], pair.h, "mean"))
    assert any(k.startswith("k_lookup_keys") for k in names)
    tn.ops.sparse_table_sync(pair.h)
    pair.assert_rows_match(all_signs(values))
