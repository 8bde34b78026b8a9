"""Pooled gradients of slots in which a few signs have most of the lookups: signs with as many lookups as are dealt to several
workgroups and one fewer, as many of them as a slot can have, the only sign there is, frequent signs behind many others and in
one run, more of them than are dealt out; rows of one and of several runs of sixteen elements, on both paths.  Sums are exact in
32 bits in any order (test_gpu_pooled_edges.py says why)."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, dev, kernels_of
from test_gpu_pooled_edges import NAMES, by_counts
from test_gpu_small_edges import HP

pytestmark = pytest.mark.gpu


def step(tn, pair, rng, values, combiner):
    """A pull, a push of pooled gradients and a second one on the same plan, both compared; the launches of the first push, the
    largest number of lookups of a sign in a slot."""
    batch = max(len(v) for v in values) + 5
    examples = [by_counts([1, 2, 4], len(v) // 7 * 7) for v in values]
    values = [v[:len(e)] for v, e in zip(values, examples)]
    pulled = pair.pull_op(values)
    cm, counts = pulled[2], pulled[4]
    names = None
    for again in range(2):
        pooled = [(rng.integers(-8, 9, (batch, pair.wf)) / 256).astype(np.float32) for _ in values]
        labels = [rng.integers(0, 2, len(v)).astype(np.int64) for v in values]
        grads = [C.combine_backward(cm[s], examples[s], pooled[s], batch, combiner, int(counts[s])) for s in range(len(values))]
        assert pair.o.push_op(values, grads, labels)[0] == 0
        args = [[dev(x) for x in xs] for xs in (values, examples, pooled, labels)]
        launched = kernels_of(tn, lambda: tn.ops.sparse_table_push_pooled(*args, pair.h, NAMES[combiner]))
        names = names or launched
        tn.ops.sparse_table_sync(pair.h)
        assert pair.assert_rows_match(all_signs(values)) > 0.99
    return names, max(np.unique(v, return_counts=True)[1].max() for v in values if len(v))


def with_counts(rng, pool, n, counts):
    """n lookups: counts[k] of them sign k in random places, the others signs behind those."""
    v = pool[len(counts) + rng.integers(0, 300, n)]
    v[rng.permutation(n)[:sum(counts)]] = np.repeat(pool[:len(counts)], counts)
    return v


@pytest.mark.parametrize("dim", [1, 16, 20, 64])
@pytest.mark.parametrize("slots,n,counts,spread", [
    (3, 2100, [1023], False), (3, 2100, [1024], True), (2, 2044, [2044], False),  # (one round whatever the signs)
    (3, 4095, [4095], True), (9, 8190, [1024] * 7, True), (9, 8190, [8190], True), (9, 8190, [3000, 1500, 1023], True)])
def test_small_batches(tn, oracle, dim, slots, n, counts, spread):
    rng = np.random.default_rng(n + dim + counts[0])
    pair = Pair(tn, oracle, "AdaGrad", dim, HP, reserve=100000)
    pool = synth.splitmix64(np.arange(1, 402, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    values = [with_counts(rng, pool, n, counts), pool[:7], pool[7:7]]  # (beside a slot of seven lookups, and one of none)
    values += [with_counts(rng, pool, n, counts) for _ in range(slots)]
    names, most = step(tn, pair, rng, values, C.MEAN)
    assert spread == (most >= 1024 and n > 2048)
    assert any(k.startswith("k_small_pool") for k in names)
    assert any(k.startswith("k_small_pool_shares") for k in names) == spread


@pytest.mark.parametrize("dim,lens", [(16, [6405, 1, 30002]), (20, [1603, 1596, 3206]), (64, [6405, 4004]), (4, [200004])])
@pytest.mark.parametrize("kind", ["late", "late, several", "more than are dealt out", "in one run", "one sign", "none"])
def test_large_batches(tn, oracle, dim, lens, kind):
    rng = np.random.default_rng(dim * 7 + len(kind))
    pair = Pair(tn, oracle, "AdaGrad", dim, HP, reserve=400000)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    pool = synth.splitmix64(np.arange(1, 3002, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    values = []
    for n in lens:
        v = pool[200 + rng.integers(0, 2800, n)]
        if kind == "late":
            v[rng.random(n) < 0.8] = pool[0]
            v[:min(n, 100)] = pool[200:][:min(n, 100)]
        elif kind == "late, several":
            m = rng.random(n) < 0.7
            v[m] = pool[rng.integers(0, 5, m.sum())]
            v[:min(n, 100)] = pool[200:][:min(n, 100)]
        elif kind == "more than are dealt out":  # (200 k lookups: 2 k of each)
            v = pool[100 + rng.integers(0, 80, n)]
            v[:min(n, 90)] = pool[200:][:min(n, 90)]
        elif kind == "in one run":
            v[n // 2:] = np.sort(pool[rng.integers(0, 4, n - n // 2)])
        elif kind == "one sign":
            v[:] = pool[0]
        values.append(v)
    names, most = step(tn, pair, rng, values, C.SUM if kind == "one sign" else C.MEAN)
    spread = max(lens) > 6403 or most >= 1024  # (a slot of eight parts, or a heavy sign)
    assert any(k.startswith("k_reduce_pooled_shares") for k in names) == ("k_pool_frequent" in names) == spread
