"""A pull whose grouping has more work items than a row of workgroups takes (65536): 129 slots of 131072 lookups.  Its ids and rows, and a
push on the plan it leaves."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, kernels_of
from test_gpu_big_groups import ADAGRAD_HP

pytestmark = pytest.mark.gpu


def test_rows_of_workgroups(tn, oracle):
    slots, lookups, vocab, dim = 129, 1 << 17, 20000, 4
    pair = Pair(tn, oracle, "AdaGrad", dim, ADAGRAD_HP, reserve=200000)
    h = pair.h
    base = synth.splitmix64(np.arange(1, vocab + 1, dtype=np.uint64))
    pair.populate(base, seed=3)
    signs = torch.from_numpy(base.view(np.int64)).cuda()
    rows = torch.from_numpy(synth.snapshot_rows(base, dim, seed=3)).cuda()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    ids = torch.randint(0, vocab, (slots, lookups), device="cuda", generator=gen)
    values = list(signs[ids])
    variables = list(torch.zeros((slots, vocab + 1, dim), device="cuda"))
    mapped = tn.ops.sparse_table_pull(variables, values, h)
    counts = tn.ops.sparse_table_last_unique_counts(h, slots)
    for s in range(slots):
        assert counts[s] == int(mapped[s].max()) + 1 == len(torch.unique(ids[s]))
        assert torch.equal(variables[s][mapped[s]], rows[ids[s]])
    for s in (0, 64, slots - 1):
        first = np.unique(ids[s].cpu().numpy(), return_index=True)[1]
        assert torch.equal(mapped[s][torch.from_numpy(np.sort(first)).cuda()].cpu(), torch.arange(len(first)))
    grads = [torch.randn((c, dim), device="cuda", generator=gen) * 0.05 for c in counts]
    labels = list((torch.rand((slots, lookups), device="cuda", generator=gen) < 0.3).long())
    names = kernels_of(tn, lambda: tn.ops.sparse_table_push(values, grads, labels, h))
    assert any(k.startswith("k_verify_values") for k in names) and "k_remap_insert" not in names  # (on the pull's plan)
    tn.ops.sparse_table_sync(h)
    host = [[t.cpu().numpy() for t in side] for side in (values, grads, labels)]
    assert pair.o.push_op(*host)[0] == 0
    assert pair.assert_rows_match(base) > 0.99
    tn.core.clear_sparse_table(h)
