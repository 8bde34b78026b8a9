"""A pull of the table or a load of rows between a batch's pull and its push: the plan the push takes up is the batch's, with its
counts, on the path of few launches and on the general one."""
import ctypes as C

import numpy as np
import pytest
import torch

from tensornet_amd import _lib, synth
from tensornet_amd._lib import TensorNetError

from helpers import Pair, dev

pytestmark = pytest.mark.gpu

HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)


@pytest.mark.parametrize("small", [True, False])
@pytest.mark.parametrize("between", ["static", "table", "load", "nothing"])
def test_a_push_after_a_pull_of_the_table(tn, oracle, between, small):
    rng = np.random.default_rng(7)
    slots, lookups, vocab, dim = 5, 900, 2000, 8
    pair = Pair(tn, oracle, "AdaGrad", dim, HP)
    tn.core.set_sparse_table_small_batch_path(pair.h, small)
    ids = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64)).view(np.int64)
    base = pair.populate(ids.view(np.uint64))
    values = [ids[rng.integers(0, vocab, lookups - 100 * s)] for s in range(slots)]
    some = np.ascontiguousarray(ids[:300])
    gsome, out = dev(some), torch.zeros((300, dim), device="cuda")
    rows = pair.o.pull(some.view(np.uint64))
    for step in range(3):
        _, _, _, _, counts = pair.pull_op(values)
        grads = synth.make_grads(counts, dim, 0.05, seed=step)
        labels = [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values]
        gvalues, ggrads, glabels = [[dev(x) for x in xs] for xs in (values, grads, labels)]
        if between == "static":
            stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
            _lib.check(_lib.load().tn_sparse_table_pull_static(pair.h, C.c_void_p(gsome.data_ptr()), 300, dim,
                                                               C.c_void_p(out.data_ptr()), stream))
        elif between == "table":
            out = tn.ops.table_pull(pair.h, gsome, dim)
        elif between == "load" and step == 0:  # (the rows they have)
            tn.ops.table_load_rows(pair.h, gsome, dev(rows))
        if between in ("static", "table"):
            np.testing.assert_allclose(out.cpu().numpy(), pair.o.pull(some.view(np.uint64)), rtol=1e-5, atol=1e-7)
        assert pair.o.push_op(values, grads, labels)[0] == 0
        tn.ops.sparse_table_push(gvalues, ggrads, glabels, pair.h)
        assert tn.ops.sparse_table_last_unique_counts(pair.h, slots) == list(counts)
        tn.ops.sparse_table_sync(pair.h)
        pair.assert_rows_match(base)


@pytest.mark.parametrize("small", [True, False])
def test_too_few_rows_are_refused_after_a_pull_of_the_table(tn, oracle, small):
    rng = np.random.default_rng(8)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP)
    tn.core.set_sparse_table_small_batch_path(pair.h, small)
    ids = synth.splitmix64(np.arange(1, 501, dtype=np.uint64)).view(np.int64)
    pair.populate(ids.view(np.uint64))
    values = [ids[rng.integers(0, 500, 400)] for _ in range(3)]
    counts = pair.pull_op(values)[4]
    out = torch.zeros((500, 8), device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    gids = dev(ids)
    _lib.check(_lib.load().tn_sparse_table_pull_static(pair.h, C.c_void_p(gids.data_ptr()), 500, 8, C.c_void_p(out.data_ptr()), stream))
    grads = [torch.zeros((int(c) - (1 if s == 1 else 0), 8), device="cuda") for s, c in enumerate(counts)]
    labels = [torch.zeros(400, dtype=torch.int64, device="cuda") for _ in values]
    with pytest.raises(TensorNetError) as e:
        tn.ops.sparse_table_push([dev(v) for v in values], grads, labels, pair.h)
        tn.ops.sparse_table_sync(pair.h)
    assert e.value.code == 1
