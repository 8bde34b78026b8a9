"""A pull whose grouping has more work items than a row of workgroups takes (65536): 129 slots of 131072 lookups."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

pytestmark = pytest.mark.gpu


def test_rows_of_workgroups(tn):
    slots, lookups, vocab, dim = 129, 1 << 17, 20000, 4
    h = tn.core.create_sparse_table(tn.core.AdaGrad(), "", dim, False, "")
    tn.core.reserve_sparse_table(h, 200000)
    signs = synth.splitmix64_torch(torch.arange(1, vocab + 1, device="cuda"))
    rows = synth.snapshot_rows_torch(signs, dim, seed=3)
    tn.ops.table_load_rows(h, signs, rows)
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
    tn.core.clear_sparse_table(h)
