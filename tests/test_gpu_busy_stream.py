"""Pull and push on a stream that has tens of milliseconds of other work ahead of them: the calls wait for the words their kernels
write to pinned memory, on every path, also where a push finds that its signs are not the last pull's."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, all_signs, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)
BUSY = 60_000_000  # cycles: well beyond what a call polls for before it looks at the stream


@pytest.mark.parametrize("path", ["few launches", "small", "large"])
def test_pull_and_push_behind_other_work(tn, oracle, path):
    rng = np.random.default_rng(3)
    slots, lookups, vocab = (3, 1_100_000, 3000) if path == "large" else (12, 1500, 3000)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP)
    tn.core.set_sparse_table_small_batch_path(pair.h, path == "few launches")
    ids = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64)).view(np.int64)
    batches = [[ids[rng.integers(0, vocab, lookups)] for _ in range(slots)] for _ in range(2)]
    base = pair.populate(ids.view(np.uint64))
    grads = [rng.standard_normal((vocab, 8)).astype(np.float32) * np.float32(0.01) for _ in range(slots)]
    labels = [(rng.random(lookups) < 0.3).astype(np.int64) for _ in range(slots)]
    ggrads, glabels = [dev(g) for g in grads], [dev(l) for l in labels]
    stream = torch.cuda.Stream()
    for pulled, pushed in ((0, 0), (1, 1), (1, 0)):
        values = [dev(v) for v in batches[pulled]]
        others = [dev(v) for v in batches[pushed]]
        variables = [torch.zeros((vocab + 1, 8), device="cuda") for _ in range(slots)]
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            torch.cuda._sleep(BUSY)
            mapped = tn.ops.sparse_table_pull(variables, values, pair.h)
            torch.cuda._sleep(BUSY)
            tn.ops.sparse_table_push(others, ggrads, glabels, pair.h)
        torch.cuda.synchronize()
        want = [np.zeros((vocab + 1, 8), np.float32) for _ in range(slots)]
        rc, want_mapped, _ = pair.o.pull_op(batches[pulled], want)
        assert rc == 0
        for s in range(slots):
            assert (mapped[s].cpu().numpy() == want_mapped[s]).all()
            np.testing.assert_allclose(variables[s].cpu().numpy(), want[s], rtol=1e-5, atol=1e-7)
        assert pair.o.push_op(batches[pushed], grads, labels)[0] == 0
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(base)
