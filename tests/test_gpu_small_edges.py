"""The path of few launches (tensornet_amd/csrc/small_batch.h) at the sizes where its kernels change their work: shares
of a slot (one workgroup, two, the most), signs that all fall into one share, more slots than the other path's slot
masks have bits, a bucket that overflows, pooled gradients of signs with one piece of lookups, several, a whole slot's."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


def mix64(x):
    with np.errstate(over="ignore"):
        x = np.asarray(x, np.uint64).copy()
        x ^= x >> np.uint64(33)
        x *= np.uint64(0xFF51AFD7ED558CCD)
        x ^= x >> np.uint64(33)
        x *= np.uint64(0xC4CEB9FE1A85EC53)
        x ^= x >> np.uint64(33)
    return x


def low_hashes(n):
    """n signs from the lowest 1/256 of the hash range: one share of a slot, few buckets."""
    out, at = [], 1
    while len(out) < n:
        s = synth.splitmix64(np.arange(at, at + (1 << 18), dtype=np.uint64))
        out.extend(s[mix64(s) >> np.uint64(56) == 0].tolist())
        at += 1 << 18
    return np.array(out[:n], np.uint64)


def step(pair, values, rng):
    counts = check_pull(pair, values)
    grads = synth.make_grads(counts, pair.wf, 0.01, seed=1)
    pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values])
    assert pair.assert_rows_match(all_signs(values)) > 0.99


@pytest.mark.parametrize("lens", [[128], [129], [1, 0, 128, 257], [2048, 5], [4096, 4095, 1], [300] * 129, [40] * 512, [0, 7] * 100])
def test_slot_lengths(tn, oracle, lens):
    rng = np.random.default_rng(sum(lens))
    pool = synth.splitmix64(np.arange(1, 6001, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP, reserve=100000, zero_init=True)
    pair.populate(pool[:3000].view(np.uint64))
    for _ in range(2):
        step(pair, [pool[(rng.random(n) ** 2 * len(pool)).astype(np.int64)] for n in lens], rng)


def test_all_signs_of_a_slot_in_one_share(tn, oracle):
    """4096 distinct signs of one hash range: one workgroup takes them all, the others none; then a slot of one sign."""
    rng = np.random.default_rng(3)
    low = low_hashes(4096).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP, reserve=100000, zero_init=True)
    pair.populate(low[:2000].view(np.uint64))
    step(pair, [low, low[:700], np.repeat(low[:1], 4096), np.full(5, -1, np.int64)], rng)


def test_a_bucket_that_overflows(tn, oracle):
    """300 slots with the same 20 signs of one bucket: more records than it has room for, the push analyses the batch."""
    rng = np.random.default_rng(4)
    low = low_hashes(20).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP, reserve=100000, zero_init=True)
    values = [rng.permutation(low) for _ in range(300)]
    step(pair, values, rng)
    step(pair, values, rng)


@pytest.mark.parametrize("opt,dim,cvm,n", [("AdaGrad", 16, False, 4096), ("AdaGrad", 8, True, 1000), ("Ftrl", 10, False, 33),
                                           ("AdaGrad", 128, False, 700), ("AdaGrad", 1, False, 2049)])
def test_pooled_gradients(tn, oracle, opt, dim, cvm, n):
    """A sign that is all of a slot, signs with 1 .. 100 lookups, examples with one lookup and with all of a slot's."""
    rng = np.random.default_rng(dim)
    hyper = HP if opt == "AdaGrad" else dict(learning_rate=0.05, beta=1.0, lambda1=0.001, lambda2=1.0)
    pair = Pair(tn, oracle, opt, dim, hyper, use_cvm=cvm, reserve=100000)
    pool = synth.splitmix64(np.arange(1, 300, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    batch = n + 3
    values = [np.repeat(pool[:1], n), pool[np.minimum(rng.geometric(0.02, n), 299) - 1], pool[rng.integers(0, 299, n)], pool[:0]]
    examples = [np.sort(rng.integers(0, batch, n)), np.full(n, batch - 1), np.arange(n), np.zeros(0, np.int64)]
    for combiner in (C.MEAN, C.SQRTN, C.SUM):
        gm, gv, cm, cv, counts = pair.pull_op(values)
        pooled = [(rng.standard_normal((batch, pair.wf)) * 0.01).astype(np.float32) for _ in values]
        labels = [rng.integers(0, 2, len(v)).astype(np.int64) for v in values]
        grads = [C.combine_backward(cm[s], examples[s], pooled[s], batch, combiner, int(counts[s])) for s in range(len(values))]
        assert pair.o.push_op(values, grads, labels)[0] == 0
        tn.ops.sparse_table_push_pooled([dev(v) for v in values], [dev(e) for e in examples], [dev(p) for p in pooled],
                                        [dev(l) for l in labels], pair.h, {C.SUM: "sum", C.MEAN: "mean", C.SQRTN: "sqrtn"}[combiner])
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(all_signs(values))
