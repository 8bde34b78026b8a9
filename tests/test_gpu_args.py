"""The descriptors of up to 52 slots go among a kernel's arguments, those of more through pinned memory: pull, push, pooled push and
combiner on either side of that number, against the oracle."""
import numpy as np
import pytest

from oracle import combine as C
from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


@pytest.mark.parametrize("slots", [1, 8, 51, 52, 53, 54])
@pytest.mark.parametrize("lookups", [7, 5000])
def test_numbers_of_slots(tn, oracle, slots, lookups):
    if slots <= 8 and lookups > 4096:
        lookups = 4096
    rng = np.random.default_rng(slots + lookups)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP, zero_init=True)
    vocab = 9000
    ids = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64)).view(np.int64)
    pair.populate(ids[:8000].view(np.uint64))
    lens = [max(0, lookups - s) for s in range(slots)]
    values = [ids[rng.integers(0, vocab, n)] for n in lens]
    batch = 40
    examples = [np.sort(rng.integers(0, batch, n)) for n in lens]
    labels = [(rng.random(n) < 0.3).astype(np.int64) for n in lens]
    for pooled in (False, True, False):
        counts = check_pull(pair, values)
        gm, gv, cm, cv, _ = pair.pull_op(values)
        out = tn.ops.embedding_lookup_sparse(gv, gm, [dev(e) for e in examples], batch, pair.h, "sum")
        for s in range(slots):
            want = C.combine_forward(cm[s], examples[s], cv[s], batch, C.SUM)
            np.testing.assert_allclose(out[s].cpu().numpy(), want, rtol=1e-5, atol=1e-6)
        if pooled:  # whole numbers: the sums are exact in any order
            dout = [rng.integers(-4, 5, (batch, 8)).astype(np.float32) / 64 for _ in range(slots)]
            grads = [C.combine_backward(cm[s], examples[s], dout[s], batch, C.SUM, int(counts[s])) for s in range(slots)]
            assert pair.o.push_op(values, grads, labels)[0] == 0
            tn.ops.sparse_table_push_pooled([dev(v) for v in values], [dev(e) for e in examples], [dev(g) for g in dout],
                                            [dev(l) for l in labels], pair.h, "sum")
            tn.ops.sparse_table_sync(pair.h)
        else:
            pair.push_op(values, synth.make_grads(counts, 8, 0.05), labels)
        pair.assert_rows_match(all_signs(values))
