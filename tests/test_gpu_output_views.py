"""The per-slot tensors that pull and combine return: consecutive parts of one allocation, whether they were made while the call
waited for the device, after a call that does not wait, or after one that failed."""
import numpy as np
import pytest
import torch

from tensornet_amd import _lib, synth
from tensornet_amd._lib import TensorNetError

from helpers import Pair, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1], [0, 5, 0, 300, 1, 0], [7] * 40, [5000] * 9])
@pytest.mark.parametrize("no_wait", [False, True])
def test_views(tn, oracle, lens, no_wait):
    rng = np.random.default_rng(len(lens))
    pair = Pair(tn, oracle, "AdaGrad", 8, dict(learning_rate=0.01), reserve=20000)
    pool = synth.splitmix64(np.arange(1, 4001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    values = [pool[rng.integers(0, len(pool), n)] for n in lens]
    dv = [dev(v) for v in values]
    room = [torch.zeros((n + 1, 8), device="cuda") for n in lens]
    _lib.check(_lib.load().tn_sparse_table_set_async(pair.h, int(no_wait)))
    for fails in (True, False):
        if fails:
            with pytest.raises(TensorNetError):
                tn.ops.sparse_table_pull(room, dv, pair.h + 1000)  # no such table
            continue
        mapped = tn.ops.sparse_table_pull(room, dv, pair.h)
        torch.cuda.synchronize()
        at = 0
        for v, m in zip(values, mapped):
            assert m.shape == (len(v),) and m.is_contiguous() and m.storage_offset() == at
            assert m.untyped_storage().data_ptr() == mapped[0].untyped_storage().data_ptr()
            first = np.unique(v, return_index=True)
            order = first[0][np.argsort(first[1])]  # distinct signs as they come up
            assert (order[m.cpu().numpy()] == v).all()
            at += len(v)
        examples = [dev(np.sort(rng.integers(0, 16, n)).astype(np.int64)) for n in lens]
        pooled = tn.ops.embedding_lookup_sparse(room, mapped, examples, 16, pair.h, "sum")
        for s, p in enumerate(pooled):
            assert p.shape == (16, 8) and p.is_contiguous() and p.storage_offset() == s * 128
            rows = room[s].double()[mapped[s]]
            want = torch.zeros((16, 8), dtype=torch.float64, device="cuda").index_add_(0, examples[s], rows)
            size = torch.zeros_like(want).index_add_(0, examples[s], rows.abs())
            # a float sum of n terms in any order is within n * 2^-24 of the sum of their sizes (n: at most all of them)
            assert bool(((p.double() - want).abs() <= len(values[s]) * 2.0 ** -24 * size).all())
