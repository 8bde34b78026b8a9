"""The rows a pull copies out, in pieces of four, two or one element: every remainder of the row length, variables at every
4-byte boundary (one slot off is enough to change the pieces of all), on the path of few launches with its second half in one launch or two, and on the other."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, dev, kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,cvm", [(1, False), (2, False), (3, False), (4, False), (6, False), (8, True), (12, False), (13, True),
                                     (62, False), (64, False)])
@pytest.mark.parametrize("slots,longest,kernel", [(4, 600, "k_small_group_finish"), (12, 600, "k_small_pull_rest"),
                                                  (12, 8193, "k_gather_vars")])
def test_pieces(tn, oracle, dim, cvm, slots, longest, kernel):
    rng = np.random.default_rng(dim + slots)
    pair = Pair(tn, oracle, "AdaGrad", dim, dict(learning_rate=0.01), use_cvm=cvm, reserve=20000)
    width = dim + 2 * cvm
    pool = synth.splitmix64(np.arange(1, 2001, dtype=np.uint64)).view(np.int64)
    pair.populate(pool.view(np.uint64))
    values = [pool[rng.integers(0, len(pool), n)] for n in [*rng.integers(0, 600, slots - 1), longest]]
    dv = [dev(v) for v in values]
    for off in (0, 1, 2, 3):
        bufs = [torch.full((off * (s == 1) + (len(v) + 1) * width + 4,), 7.0, device="cuda") for s, v in enumerate(values)]
        room = [b[off * (s == 1):][:(len(v) + 1) * width].view(-1, width) for s, (b, v) in enumerate(zip(bufs, values))]
        mapped = []
        names = kernels_of(tn, lambda: mapped.extend(tn.ops.sparse_table_pull(room, dv, pair.h)))
        pieces = (4, 1) if kernel == "k_gather_vars" else (4, 2, 1)
        per = next(k for k in pieces if width % k == 0 and off % k == 0)
        assert "%s<%d>" % (kernel, per) in names
        for s, v in enumerate(values):
            signs, first = np.unique(v, return_index=True)
            order = signs[np.argsort(first)]
            assert (order[mapped[s].cpu().numpy()] == v).all()
            got = bufs[s].cpu().numpy().view(np.int32)
            want = np.full(len(got), 7.0, np.float32).view(np.int32)
            if len(order):
                rows = tn.ops.table_export_rows(pair.h, dev(order))[0].cpu().numpy()
                want[off * (s == 1):][:rows.size] = rows.view(np.int32).ravel()
            assert (got == want).all()  # the rows bit for bit, nothing before or behind them
