"""The mapped ids of a large batch are there when the pull returns, for a reader on any stream, which the caller has not ordered behind
the call's: only the copy of the rows may still be running then."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots,lookups", [(3, 1_100_000), (100, 30_001), (200, 9000), (300, 9000)])
def test_read_from_another_stream(tn, slots, lookups):
    vocab, dim = 200_000, 16
    h = tn.core.create_sparse_table(tn.core.AdaGrad(), "", dim, False, "")
    tn.core.reserve_sparse_table(h, vocab)
    signs = synth.splitmix64_torch(torch.arange(1, vocab + 1, device="cuda"))
    tn.ops.table_load_rows(h, signs, synth.snapshot_rows_torch(signs, dim, seed=3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(slots)
    ids = torch.randint(0, vocab, (slots, lookups), device="cuda", generator=gen)
    values = list(signs[ids])
    variables = list(torch.zeros((slots, min(vocab, lookups) + 1, dim), device="cuda"))
    pull = tn.ops.BoundSparseTablePull(variables, values, h)
    flat = torch.as_strided(pull.mapped[0], (slots, lookups), (lookups, 1))  # (one allocation holds them all)
    pull()
    torch.cuda.synchronize()
    want = flat.clone()
    for s in (0, slots - 1):
        _, first, inverse = np.unique(ids[s].cpu().numpy(), return_index=True, return_inverse=True)
        assert (want[s].cpu().numpy() == np.argsort(np.argsort(first))[inverse]).all()
    other = torch.cuda.Stream()
    for _ in range(4):
        flat.fill_(-1)
        torch.cuda.synchronize()
        pull()
        with torch.cuda.stream(other):
            seen = flat.clone()
        torch.cuda.synchronize()
        assert torch.equal(seen, want)
    tn.core.clear_sparse_table(h)
