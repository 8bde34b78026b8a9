"""The forward combiner takes the examples of a slot some dozens to a workgroup and finds their lookups by search: batches
around a workgroup's share, slots with none, few and very many lookups, examples with all of them, rows of any length,
and ids out of order where the search has passed them by."""
import numpy as np
import pytest
import torch

from oracle import combine as C
from tensornet_amd._lib import TensorNetError

from helpers import ATOL, RTOL, dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def table(tn):
    return tn.core.create_sparse_table(tn.core.AdaGrad(), "", 4, False, "")


@pytest.mark.parametrize("batch,lens,dim", [(1, [0, 1, 9], 16), (63, [64, 1, 0, 300], 8), (64, [255, 256, 257], 4), (65, [65536, 3], 16),
                                            (5000, [70000, 10, 4999], 1), (129, [400] * 300, 10), (70000, [300, 70000] * 3, 16),
                                            (40, [90, 7], 130), (40, [90, 7], 256), (3, [20], 33)])
def test_forward(tn, table, batch, lens, dim):
    rng = np.random.default_rng(batch + dim)
    var, ids, ex = [], [], []
    for i, n in enumerate(lens):
        rows = max(1, n // 2)
        var.append(rng.standard_normal((rows, dim)).astype(np.float32))
        ids.append(rng.integers(0, rows, n))
        e = np.full(n, batch - 1) if i == 1 else np.sort((rng.random(n) ** 2 * batch).astype(np.int64))
        ex.append(e)
    for combiner, name in ((C.MEAN, "mean"), (C.SUM, "sum"), (C.SQRTN, "sqrtn")):
        out = tn.ops.embedding_lookup_sparse([dev(v) for v in var], [dev(i) for i in ids], [dev(e) for e in ex], batch, table, name)
        for s in range(len(lens)):
            want = C.combine_forward(ids[s], ex[s], var[s], batch, combiner)
            np.testing.assert_allclose(out[s].cpu().numpy(), want, rtol=RTOL, atol=1e-6)


@pytest.mark.parametrize("where", [0, 1, 255, 256, 40000, 99998])
@pytest.mark.parametrize("value", [0, 50000, 99999, -1, 100000])
def test_one_id_out_of_order_is_found(tn, table, where, value):
    """100 000 lookups, the i-th of example i, one of them given to another example or to none."""
    n = 100000
    ex = torch.arange(n, device="cuda")
    ex[where] = value
    ids = torch.zeros(n, dtype=torch.int64, device="cuda")
    var = torch.ones((1, 4), device="cuda")
    if max(where - 1, 0) <= value <= where + 1 and value < n:  # still in order
        tn.ops.embedding_lookup_sparse([var], [ids], [ex], n, table)
        return
    with pytest.raises(TensorNetError) as e:
        tn.ops.embedding_lookup_sparse([var], [ids], [ex], n, table)
    assert e.value.code == 1
    ex[where] = where
    tn.ops.embedding_lookup_sparse([var], [ids], [ex], n, table)  # and the error does not stay
