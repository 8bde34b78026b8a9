"""A table that is used on the default stream and on others: a call on a stream of its own waits for the table's last call on the default
one, not for what has been queued there since."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)
BUSY = 60_000_000  # cycles, tens of milliseconds


@pytest.mark.parametrize("small", [True, False])
def test_what_the_default_stream_does_meanwhile_is_not_waited_for(tn, oracle, small):
    """Several streams of their own: one that shares a hardware queue with the default stream waits for its kernels anyway."""
    rng = np.random.default_rng(4)
    slots, lookups, vocab = 6, 900, 2000
    pair = Pair(tn, oracle, "AdaGrad", 8, HP)
    tn.core.set_sparse_table_small_batch_path(pair.h, small)
    ids = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64)).view(np.int64)
    base = pair.populate(ids.view(np.uint64))
    values = [ids[rng.integers(0, vocab, lookups)] for _ in range(slots)]
    grads = [rng.standard_normal((lookups, 8)).astype(np.float32) * np.float32(0.1) for _ in range(slots)]
    labels = [(rng.random(lookups) < 0.3).astype(np.int64) for _ in range(slots)]
    gvalues, ggrads, glabels = [[dev(x) for x in xs] for xs in (values, grads, labels)]
    variables, served = [[torch.zeros((lookups + 1, 8), device="cuda") for _ in range(slots)] for _ in range(2)]
    default = torch.cuda.default_stream()
    free = []
    for i in range(7):
        own = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(default):
            tn.ops.sparse_table_pull(variables, gvalues, pair.h)
            if small:  # (behind a push of a large batch the host waits for the stream)
                tn.ops.sparse_table_push(gvalues, ggrads, glabels, pair.h)
                assert pair.o.push_op(values, grads, labels)[0] == 0
            if i > 0:
                torch.cuda._sleep(BUSY)
            busy = torch.cuda.Event()
            busy.record()
        with torch.cuda.stream(own):
            tn.ops.sparse_table_pull(served, gvalues, pair.h)
        own.synchronize()
        if i > 0:  # (the first call on another stream is what makes the table leave events)
            free.append(not busy.query())
        want = [np.zeros((lookups + 1, 8), np.float32) for _ in range(slots)]
        assert pair.o.pull_op(values, want)[0] == 0
        for s in range(slots):
            np.testing.assert_allclose(served[s].cpu().numpy(), want[s], rtol=1e-5, atol=1e-7)
    assert any(free)
    tn.ops.sparse_table_sync(pair.h)
    pair.assert_rows_match(base)
