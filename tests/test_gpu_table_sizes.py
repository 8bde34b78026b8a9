"""Table-level push at the numbers of buckets around which its counters' places in LDS jump, table-level pull of rows whose pieces
fill a workgroup's turns exactly, just not, or by one more, in pieces of four elements and of one, on either side of the two pieces of a
thread up to which they are copied one by one."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, dev, kernels_of

from test_gpu_table_level import HP, pushed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,opt,dim", [(128, "AdaGrad", 4), (129, "AdaGrad", 4), (1024, "AdaGrad", 4), (1025, "AdaGrad", 4),
                                       (8191, "AdaGrad", 4), (33000, "AdaGrad", 4), (262144, "AdaGrad", 4), (262145, "AdaGrad", 4),
                                       # the update kernel's chunks of four rounds above 768 buckets
                                       (98304, "Adam", 8), (98305, "Adam", 8), (98304, "Ftrl", 32), (98305, "Ftrl", 32)])
def test_push_of_so_many_buckets(tn, oracle, n, opt, dim):
    rng = np.random.default_rng(n)
    pair = Pair(tn, oracle, opt, dim, HP[opt], reserve=200000)
    base = pair.populate(synth.splitmix64(np.arange(1, 60001, dtype=np.uint64)))
    req = base[(rng.random(n) ** (2 if dim == 4 else 6) * len(base)).astype(np.int64)]
    out = []
    names = kernels_of(tn, lambda: out.append(pushed(tn, oracle, pair, req, rng)))
    many = n > 128 * (512 if opt == "AdaGrad" else 768)
    assert [k.endswith(", true)>") for k in names if k.startswith("k_table_apply<")] == [many]
    infos, grads = out[0]
    assert pair.o.push(infos, grads) == 0
    pair.assert_rows_match(base)


@pytest.mark.parametrize("dim", [1, 2, 3, 4, 8, 12, 32, 36, 64])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 16384, 16385, 17000])
def test_pull_of_rows(tn, oracle, dim, n):
    rng = np.random.default_rng(n + dim)
    pair = Pair(tn, oracle, "AdaGrad", dim, HP["AdaGrad"], reserve=10000)
    base = pair.populate(synth.splitmix64(np.arange(1, 3001, dtype=np.uint64)))
    req = base[rng.integers(0, len(base), n)]
    out = tn.ops.table_pull(pair.h, dev(req.view(np.int64)), dim).cpu().numpy()
    np.testing.assert_array_equal(out, pair.o.pull(req))
