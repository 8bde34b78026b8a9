"""Small batches (and one through LDS) that leave work on the default stream, and calls on other streams right after them: what the
last call left is waited for, in either direction and more than once."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


@pytest.mark.parametrize("slots,small", [(12, True), (4, True), (12, False)])
def test_calls_alternate_between_streams(tn, oracle, slots, small):
    rng = np.random.default_rng(slots)
    lookups, vocab = 1200, 4000
    pair = Pair(tn, oracle, "AdaGrad", 8, HP)
    tn.core.set_sparse_table_small_batch_path(pair.h, small)
    ids = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64)).view(np.int64)
    base = pair.populate(ids.view(np.uint64))
    values = [ids[rng.integers(0, vocab, lookups)] for _ in range(slots)]
    grads = [rng.standard_normal((lookups, 8)).astype(np.float32) * np.float32(0.1) for _ in range(slots)]
    labels = [(rng.random(lookups) < 0.3).astype(np.int64) for _ in range(slots)]
    gvalues, ggrads, glabels = [[dev(x) for x in xs] for xs in (values, grads, labels)]
    variables = [torch.zeros((lookups + 1, 8), device="cuda") for _ in range(slots)]
    own = [torch.cuda.Stream() for _ in range(2)]
    default = torch.cuda.default_stream()
    torch.cuda.synchronize()
    for i, (first, second) in enumerate([(default, own[0]), (own[0], default), (default, own[1]), (own[1], own[0]), (own[0], default)]):
        with torch.cuda.stream(first):
            tn.ops.sparse_table_pull(variables, gvalues, pair.h)
            tn.ops.sparse_table_push(gvalues, ggrads, glabels, pair.h)  # its updates are still running
        with torch.cuda.stream(second):
            out = tn.ops.table_pull(pair.h, dev(ids), 8)
            tn.ops.sparse_table_pull(variables, gvalues, pair.h)
        torch.cuda.synchronize()
        assert pair.o.push_op(values, grads, labels)[0] == 0
        np.testing.assert_allclose(out.cpu().numpy(), pair.o.pull(ids.view(np.uint64)), rtol=1e-5, atol=1e-7)
        want = [np.zeros((lookups + 1, 8), np.float32) for _ in range(slots)]
        assert pair.o.pull_op(values, want)[0] == 0
        for s in range(slots):
            np.testing.assert_allclose(variables[s].cpu().numpy(), want[s], rtol=1e-5, atol=1e-7)
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(base)
