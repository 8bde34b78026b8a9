"""The passes of a pull that share a launch (grouping, probes and flags; ranks and new rows; member lists and mapped ids; the copy of
the rows and the status) at sizes where their workgroups do not divide evenly: odd numbers of tiles, one bucket, slots that do not
fill a workgroup's wavefronts, rows to insert or none.  A push on the plan, whose errors reach the host by themselves."""
import numpy as np
import pytest

from tensornet_amd import _lib, synth

from helpers import Pair, all_signs, check_pull, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


@pytest.mark.parametrize("slots,lookups,vocab,resident", [
    (1, 1024, 1 << 20, 0), (1, 2049, 100, 100), (3, 4095, 5000, 2500), (9, 683, 300, 300), (63, 131, 4000, 0),
    (128, 97, 90, 45), (129, 97, 90, 45), (255, 65, 30000, 15000)])
def test_uneven_workgroups(tn, oracle, slots, lookups, vocab, resident):
    rng = np.random.default_rng(slots * 7 + lookups)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP, zero_init=True)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    ids = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64)).view(np.int64)
    if resident:
        pair.populate(ids[:resident].view(np.uint64))
    values = [ids[rng.integers(0, vocab, lookups)] for _ in range(slots)]
    values[0][0] = -1  # the sign that equals a free entry's key
    for _ in range(2):
        counts = check_pull(pair, values)
        grads = synth.make_grads(counts, 8, 0.01)
        labels = [(rng.random(lookups) < 0.3).astype(np.int64) for _ in range(slots)]
        pair.push_op(values, grads, labels)
        pair.assert_rows_match(all_signs(values))
    assert tn.ops.sparse_table_last_unique_counts(pair.h, slots) == counts.tolist()


@pytest.mark.parametrize("slots", [2, 40])
def test_a_short_gradient_matrix_is_reported(tn, oracle, slots):
    """By the call that waits next, and once; records that have a gradient row are applied."""
    rng = np.random.default_rng(slots)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP)
    tn.core.set_sparse_table_small_batch_path(pair.h, False)
    ids = synth.splitmix64(np.arange(1, 3001, dtype=np.uint64)).view(np.int64)
    pair.populate(ids.view(np.uint64))
    values = [rng.permutation(ids)[:1500] for _ in range(slots)]
    check_pull(pair, values)
    grads = [np.ones((1500 if s else 1400, 8), np.float32) for s in range(slots)]
    labels = [np.zeros(1500, np.int64) for _ in range(slots)]
    tn.ops.sparse_table_push([dev(v) for v in values], [dev(g) for g in grads], [dev(l) for l in labels], pair.h)
    with pytest.raises(_lib.TensorNetError) as e:
        tn.ops.sparse_table_sync(pair.h)
    assert "fewer rows" in str(e.value)
    tn.ops.sparse_table_sync(pair.h)
    rest = set(ids.tolist()) - set(values[0][1400:].tolist())
    assert pair.o.push_op([values[0][:1400]] + values[1:], grads, [labels[0][:1400]] + labels[1:])[0] == 0
    pair.assert_rows_match(np.array(sorted(rest), dtype=np.int64).view(np.uint64))
