"""Calls on one stream right after calls on another, with nothing in between: a sparse table orders them itself.  Among the
streams is the default one, which streams of the caller's own are not ordered behind."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


@pytest.mark.parametrize("first", ["default", "own"])
@pytest.mark.parametrize("what", ["push", "decay"])
def test_a_call_waits_for_what_another_stream_still_runs(tn, oracle, first, what):
    """The first stream is busy when the call is queued on it, the second is not.  (Several second streams: one that shares
    a hardware queue with the first would be ordered behind it in any case.)"""
    rng = np.random.default_rng(1)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP)
    base = pair.populate(synth.splitmix64(np.arange(1, 2001, dtype=np.uint64)))
    infos = np.zeros(len(base), dtype=oracle.sign_info_dtype)
    infos["sign"], infos["batch_show"], infos["batch_click"] = base, 3, 1
    signs = dev(base.view(np.int64))
    ones = torch.ones(len(base), dtype=torch.int64, device="cuda")
    records = tn.ops.make_sign_infos(signs, 3 * ones, ones)
    one = torch.cuda.default_stream() if first == "default" else torch.cuda.Stream()
    for _ in range(6):
        two = torch.cuda.Stream()
        grads = (rng.standard_normal((len(base), 8)) * 0.1).astype(np.float32)
        ggrads = dev(grads)
        torch.cuda.synchronize()
        with torch.cuda.stream(one):
            torch.cuda._sleep(25_000_000)
            if what == "push":
                tn.ops.table_push(pair.h, records, ggrads)
            else:
                tn.core.show_decay(pair.h, 1)
        with torch.cuda.stream(two):
            if what == "push":
                out = tn.ops.table_pull(pair.h, signs, 8)
            else:
                tn.ops.table_push(pair.h, records, ggrads)
        torch.cuda.synchronize()
        if what == "push":
            assert pair.o.push(infos, grads) == 0
            np.testing.assert_allclose(out.cpu().numpy(), pair.o.pull(base), rtol=1e-5, atol=1e-7)
        else:
            pair.o.show_decay(1)
            assert pair.o.push(infos, grads) == 0
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(base)
