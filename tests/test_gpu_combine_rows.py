"""The forward combiner keeps the rows of a workgroup's lookups in LDS where they fit (2048): one workgroup's lookups around that
number, a mapped id that is no row of its variable at either end of them, and many slots, whose workgroups take more examples."""
import numpy as np
import pytest
import torch

from oracle import combine as C
from tensornet_amd._lib import TensorNetError

from helpers import RTOL, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,lookups,slots,dim", [
    (50, 2047, 1, 16), (50, 2048, 1, 16), (50, 2049, 1, 16), (64, 6000, 2, 10), (1000, 3000, 200, 8), (600, 4800, 300, 4)])
def test_lookups_around_what_fits(tn, batch, lookups, slots, dim):
    table = tn.core.create_sparse_table(tn.core.AdaGrad(), "", 4, False, "")
    rng = np.random.default_rng(lookups)
    rows = 777
    var = [rng.standard_normal((rows, dim)).astype(np.float32) for _ in range(slots)]
    ids = [rng.integers(0, rows, lookups) for _ in range(slots)]
    ex = [np.sort(rng.integers(0, batch, lookups)) for _ in range(slots)]
    gvar, gids, gex = [dev(v) for v in var], [dev(i) for i in ids], [dev(e) for e in ex]
    out = tn.ops.embedding_lookup_sparse(gvar, gids, gex, batch, table, "sqrtn")
    for s in range(slots):
        # (sums in the oracle's order; a division apart)
        np.testing.assert_allclose(out[s].cpu().numpy(), C.combine_forward(ids[s], ex[s], var[s], batch, C.SQRTN), rtol=RTOL, atol=1e-6)
    for at in (0, lookups - 1):
        for bad in (-1, rows, 1 << 32):
            kept = int(gids[-1][at])
            gids[-1][at] = bad
            with pytest.raises(TensorNetError) as e:
                tn.ops.embedding_lookup_sparse(gvar, gids, gex, batch, table, "sqrtn")
            assert "not a row" in str(e.value)
            gids[-1][at] = kept
    again = tn.ops.embedding_lookup_sparse(gvar, gids, gex, batch, table, "sqrtn")
    assert all(torch.equal(a, b) for a, b in zip(out, again))
