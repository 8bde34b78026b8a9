"""Example ids out of order by whole runs of lookups, in a workgroup of the forward combiner that is not its slot's first: the call is
refused, an example whose run lost its start sums nothing, and the others what is theirs.  On both sides of the 2048 lookups
whose rows a workgroup keeps in LDS."""
import numpy as np
import pytest
import torch

from oracle import combine as C
from tensornet_amd._lib import TensorNetError

from helpers import RTOL, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 60])  # (descriptors among the kernel's arguments, and in memory)
@pytest.mark.parametrize("run", [2, 3, 40])
def test_a_run_behind_its_neighbour(tn, run, slots):
    batch, dim, rows, moved = 256, 8, 500, 70
    table = tn.core.create_sparse_table(tn.core.AdaGrad(), "", 4, False, "")
    rng = np.random.default_rng(run)
    ex = np.repeat(np.arange(batch), run)
    var = rng.standard_normal((rows, dim)).astype(np.float32)
    ids = rng.integers(0, rows, len(ex))
    wrong = ex.copy()
    wrong[moved * run:(moved + 2) * run] = np.repeat([moved + 1, moved], run)
    gvar, gids = [dev(var)] * slots, [dev(ids)] * slots
    good = [dev(ex)] * slots
    bound = tn.ops.BoundEmbeddingLookupSparse(gvar, gids, good[1:] + [dev(wrong)], batch, table, "sum")
    with pytest.raises(TensorNetError) as e:
        bound()
    assert e.value.code == 1 and "non-decreasing" in str(e.value)
    want = C.combine_forward(ids, ex, var, batch, C.SUM)
    want[moved + 1] = want[moved]  # (where its lookups stood)
    want[moved] = 0
    np.testing.assert_allclose(bound.out[slots - 1].cpu().numpy(), want, rtol=RTOL, atol=1e-6)
    out = tn.ops.embedding_lookup_sparse(gvar, gids, good, batch, table, "sum")
    want = C.combine_forward(ids, ex, var, batch, C.SUM)
    for o in out:
        np.testing.assert_allclose(o.cpu().numpy(), want, rtol=RTOL, atol=1e-6)
