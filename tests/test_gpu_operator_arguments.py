"""What the operators keep alive of the sequences they are given (tensornet_amd/csrc/bind.cc)."""
import gc
import threading
import time
import weakref

import numpy as np
import pytest
import torch

from oracle import combine as C
from tensornet_amd import synth

from helpers import ATOL, RTOL, Pair, all_signs, dev

pytestmark = pytest.mark.gpu

ADAGRAD_HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)
BATCH, SLOTS, D = 64, 3, 8


def setup(tn, oracle, seed):
    rng = np.random.default_rng(seed)
    pool = synth.splitmix64(np.arange(1, 301, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, "AdaGrad", D, ADAGRAD_HP)
    pair.populate(pool.view(np.uint64))
    values = [pool[rng.integers(0, len(pool), 2 * BATCH)] for _ in range(SLOTS)]
    examples = [np.repeat(np.arange(BATCH, dtype=np.int64), 2)] * SLOTS
    labels = [rng.integers(0, 2, 2 * BATCH).astype(np.int64) for _ in range(SLOTS)]
    return rng, pair, values, examples, labels


def handed_out(refs, arrays):
    """Tensors that nobody holds but whoever iterates."""
    for a in arrays:
        t = dev(a)
        refs.append(weakref.ref(t))
        yield t


def test_bound_operators_hold_what_an_iterator_hands_out(tn, oracle):
    """A generator can be gone over once: what the operators marshalled is what they have to keep."""
    rng, pair, values, examples, labels = setup(tn, oracle, 1)
    refs = []
    variables = [np.full((2 * BATCH + 1, D), -7.0, np.float32)] * SLOTS
    held = [dev(v) for v in variables]
    pull = tn.ops.BoundSparseTablePull((v for v in held), handed_out(refs, values), pair.h)
    combine = tn.ops.BoundEmbeddingLookupSparse(iter(held), iter(pull.mapped), handed_out(refs, examples), BATCH, pair.h)
    rc, cm, counts = pair.o.pull_op(values, [v.copy() for v in variables])
    assert rc == 0
    grads = synth.make_grads(counts, D, 0.01, seed=1)
    push = tn.ops.BoundSparseTablePush(handed_out(refs, values), handed_out(refs, grads), handed_out(refs, labels), pair.h)
    pooled = [rng.standard_normal((BATCH, D)).astype(np.float32) * 0.01 for _ in range(SLOTS)]
    push_pooled = tn.ops.BoundSparseTablePushPooled(handed_out(refs, values), handed_out(refs, examples), handed_out(refs, pooled),
                                                    handed_out(refs, labels), pair.h)
    ops = [pull, combine, push, push_pooled]
    gc.collect()
    assert len(refs) == 9 * SLOTS and all(r() is not None for r in refs)
    mapped = pull()
    assert all((m.cpu().numpy() == c).all() for m, c in zip(mapped, cm))
    out = combine()
    for s in range(SLOTS):
        want = C.combine_forward(cm[s], examples[s], held[s].cpu().numpy(), BATCH, C.MEAN)
        np.testing.assert_allclose(out[s].cpu().numpy(), want, rtol=RTOL, atol=ATOL)
    push()
    pull()
    push_pooled()
    tn.ops.sparse_table_sync(pair.h)
    assert pair.o.push_op(values, grads, labels)[0] == 0
    reduced = [C.combine_backward(cm[s], examples[s], pooled[s], BATCH, C.MEAN, int(counts[s])) for s in range(SLOTS)]
    assert pair.o.push_op(values, reduced, labels)[0] == 0
    pair.assert_rows_match(all_signs(values))
    del ops, pull, combine, push, push_pooled
    gc.collect()
    assert all(r() is None for r in refs)


@pytest.mark.parametrize("op", ["pull", "push", "pooled", "combine"])
def test_an_operator_holds_its_tensors_while_it_runs(tn, oracle, op):
    """A second thread empties the caller's lists while the call waits for the device: the tensors stay until it ends."""
    rng, pair, values, examples, labels = setup(tn, oracle, 2)
    variables = [np.full((2 * BATCH + 1, D), -7.0, np.float32)] * SLOTS
    gm = tn.ops.sparse_table_pull([dev(v) for v in variables], [dev(v) for v in values], pair.h)
    counts = tn.ops.sparse_table_last_unique_counts(pair.h, SLOTS)
    grads = synth.make_grads(counts, D, 0.01, seed=1)
    pooled = [rng.standard_normal((BATCH, D)).astype(np.float32) * 0.01 for _ in range(SLOTS)]
    if op == "pull":
        lists, call = [variables, values], lambda r, v: tn.ops.sparse_table_pull(r, v, pair.h)
    elif op == "push":
        lists, call = [values, grads, labels], lambda v, g, l: tn.ops.sparse_table_push(v, g, l, pair.h)
    elif op == "pooled":
        lists, call = [values, examples, pooled, labels], lambda *a: tn.ops.sparse_table_push_pooled(*a, pair.h)
    else:
        lists = [variables, [m.cpu().numpy() for m in gm], examples]
        call = lambda r, m, e: tn.ops.embedding_lookup_sparse(r, m, e, BATCH, pair.h)
    lists = [[dev(a) for a in arrays] for arrays in lists]
    refs = [weakref.ref(t) for tensors in lists for t in tensors]
    torch.cuda.synchronize()
    entered, ended, seen = threading.Event(), threading.Event(), []

    def empty_the_lists():
        entered.wait()
        time.sleep(0.02)
        if ended.is_set():
            return
        for tensors in lists:
            tensors.clear()
        gone = [r() is None for r in refs]
        if not ended.is_set():  # (all this time the call was on its way)
            seen.append(not any(gone))

    other = threading.Thread(target=empty_the_lists)
    other.start()
    torch.cuda._sleep(200_000_000)  # the device is busy for a tenth of a second or so
    entered.set()
    call(*lists)
    ended.set()
    other.join()
    torch.cuda.synchronize()
    tn.ops.sparse_table_sync(pair.h)
    assert seen == [True]
    assert all(r() is None for r in refs)
