"""The path of few launches with slots of up to 8192 lookups (more than eight slots), and its signs with many records, which a
wavefront applies chunk by chunk: rows of every power of two up to 64 elements under each optimizer, with as many records
as a chunk, one more, several chunks; counts that are no whole numbers; a slot whose gradient matrix has too few rows."""
import numpy as np
import pytest
import torch

from tensornet_amd import _lib, synth

from helpers import Pair, all_signs, check_pull, dev, kernels_of

pytestmark = pytest.mark.gpu

HP = {"AdaGrad": dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8),
      "Adam": dict(learning_rate=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8),
      "Ftrl": dict(learning_rate=0.05, beta=1.0, lambda1=0.001, lambda2=1.0)}


def push(pair, values, counts, rng, seed):
    grads = synth.make_grads(counts, pair.wf, 0.01, seed=seed)
    pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values])
    assert pair.assert_rows_match(all_signs(values)) > 0.99


@pytest.mark.parametrize("lens", [[4097] * 9, [8192] + [1] * 11, [8192, 8191, 4096, 0] * 4, [8193] + [5] * 10])
def test_long_slots(tn, oracle, lens):
    rng = np.random.default_rng(sum(lens))
    pool = synth.splitmix64(np.arange(1, 12001, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP["AdaGrad"], reserve=100000, zero_init=True)
    pair.populate(pool[:9000].view(np.uint64))
    for kind in range(3):
        values = []
        for n in lens:
            if kind == 0:
                v = rng.permutation(pool)[:n]  # distinct signs
            elif kind == 1:
                v = pool[(rng.random(n) ** 4 * len(pool)).astype(np.int64)]
            else:
                v = np.repeat(pool[:1], n)
            values.append(v)
        names = []
        counts = None

        def pull():
            nonlocal counts
            counts = check_pull(pair, values)
        names = kernels_of(tn, pull)
        assert ("k_small_slots_long" in names) == (max(lens) <= 8192)
        push(pair, values, counts, rng, kind)


@pytest.mark.parametrize("opt", ["AdaGrad", "Adam", "Ftrl"])
@pytest.mark.parametrize("dim", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("slots", [13, 64, 65, 131])
def test_signs_with_many_records(tn, oracle, opt, dim, slots):
    rng = np.random.default_rng(dim * 100 + slots)
    pool = synth.splitmix64(np.arange(1, 2001, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, opt, dim, HP[opt], reserve=20000, zero_init=True)
    pair.populate(pool.view(np.uint64))
    values = []
    for s in range(slots):  # signs in every slot, in all but a few, in every other one, ... and in a few
        v = [p for i, p in enumerate(pool[:40]) if s % (1 + i // 4) == 0 and s < slots - i]
        values.append(rng.permutation(np.concatenate([np.array(v, np.int64), rng.choice(pool[40:], 20)])))
    for seed in range(2):
        counts = check_pull(pair, values)
        push(pair, values, counts, rng, seed)
    push(pair, values, counts, rng, 7)  # again on the plan


def test_a_sign_without_all_its_gradient_rows(tn, oracle):
    """Slot 3's matrix has no rows: its records are left out and reported, those of the sign's other slots applied."""
    dim, slots = 16, 70
    pool = synth.splitmix64(np.arange(1, 11, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", dim, HP["AdaGrad"], reserve=1000, zero_init=True)
    pair.populate(pool.view(np.uint64))
    other = Pair(tn, oracle, "AdaGrad", dim, HP["AdaGrad"], reserve=1000, zero_init=True)
    other.populate(pool.view(np.uint64))
    values = [pool.copy() for _ in range(slots)]
    zeros = [np.zeros(len(v), np.int64) for v in values]
    counts = check_pull(pair, values)
    grads = synth.make_grads(counts, dim, 0.01, seed=1)
    with pytest.raises(_lib.TensorNetError):
        tn.ops.sparse_table_push([dev(v) for v in values], [dev(g if s != 3 else g[:0]) for s, g in enumerate(grads)],
                                 [dev(z) for z in zeros], pair.h)
    tn.ops.sparse_table_sync(pair.h)
    rest = [v for s, v in enumerate(values) if s != 3]
    check_pull(other, rest)
    other.push_op(rest, [g for s, g in enumerate(grads) if s != 3], zeros[1:])
    torch.cuda.synchronize()
    (gw, gs, _), _ = pair.export(pool.view(np.uint64))
    (ow, os_, _), _ = other.export(pool.view(np.uint64))
    assert (gw == ow).all() and (gs == os_).all()
