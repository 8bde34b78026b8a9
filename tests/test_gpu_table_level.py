"""Table-level pull and push (tensornet_amd/csrc/table_level.h) at the sizes where their kernels change their work: one
record, edges of a tile, of the tile sizes and of what a bucket's workgroup groups at a time, signs with few records, with
many and with more than fit at once, unknown signs, new signs that a request repeats."""
import numpy as np
import pytest
import torch

import tensornet_amd
from tensornet_amd import synth

from helpers import Pair, dev, kernels_of

pytestmark = pytest.mark.gpu

HP = {"AdaGrad": dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8),
      "Adam": dict(learning_rate=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8),
      "Ftrl": dict(learning_rate=0.05, beta=1.0, lambda1=0.1, lambda2=1.0)}


def pushed(tn, oracle, pair, req, rng):
    n = len(req)
    infos = np.zeros(n, dtype=oracle.sign_info_dtype)
    infos["sign"] = req
    infos["batch_show"] = rng.integers(1, 5, n)
    infos["batch_click"] = rng.integers(0, 2, n)
    grads = (rng.standard_normal((n, pair.wf)) * 0.01).astype(np.float32)
    tn.ops.table_push(pair.h, tn.ops.make_sign_infos(dev(req.view(np.int64)), dev(infos["batch_show"].astype(np.int64)),
                                                     dev(infos["batch_click"].astype(np.int64))), dev(grads))
    return infos, grads


@pytest.mark.parametrize("opt,dim,cvm,n,spread", [
    ("AdaGrad", 8, False, 1, 1.0), ("Adam", 16, False, 256, 1.0), ("AdaGrad", 16, False, 257, 0.5),
    ("AdaGrad", 16, False, 5000, 0.0), ("Adam", 4, False, 1537, 0.0), ("Ftrl", 10, False, 9000, 0.01),
    ("AdaGrad", 10, True, 40000, 0.3), ("AdaGrad", 64, False, 40000, 0.05), ("Ftrl", 128, False, 3000, 0.02),
    ("Adam", 160, False, 2000, 0.2), ("Adam", 8, False, 131073, 0.4), ("AdaGrad", 16, False, 524289, 0.9)])
def test_push_and_pull(tn, oracle, opt, dim, cvm, n, spread):
    """n records of about spread * n signs, some of them far more often than the others."""
    rng = np.random.default_rng(n)
    keys = max(1, int(spread * n))
    pair = Pair(tn, oracle, opt, dim, HP[opt], use_cvm=cvm, reserve=2 * keys + 100)
    base = pair.populate(synth.splitmix64(np.arange(1, keys + 1, dtype=np.uint64)))
    req = base[(rng.random(n) ** 2 * keys).astype(np.int64)]
    for _ in range(2):
        infos, grads = pushed(tn, oracle, pair, req, rng)
        assert pair.o.push(infos, grads) == 0
    out = tn.ops.table_pull(pair.h, dev(req.view(np.int64)), pair.wf).cpu().numpy()
    np.testing.assert_allclose(out, pair.o.pull(req), rtol=1e-5, atol=1e-7)
    pair.assert_rows_match(base)


@pytest.mark.parametrize("opt", ["AdaGrad", "Adam", "Ftrl"])
@pytest.mark.parametrize("dim", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("cvm", [False, True])
def test_signs_with_many_records(tn, oracle, opt, dim, cvm):
    """As many records as a wavefront takes up, as a chunk of it holds, one less and one more, and more than are grouped at
    a time, among signs with one or two."""
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, opt, dim, HP[opt], use_cvm=cvm, reserve=2000)
    base = pair.populate(synth.splitmix64(np.arange(1, 601, dtype=np.uint64)))
    times = [15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 511, 512, 513, 1100]
    req = rng.permutation(np.concatenate([np.repeat(base[:len(times)], times), base[100:], base[100:200]]))
    for _ in range(2):
        infos, grads = pushed(tn, oracle, pair, req, rng)
        assert pair.o.push(infos, grads) == 0
    pair.assert_rows_match(base)


@pytest.mark.parametrize("n", [1, 64, 65, 1000, 65536])
def test_pull_of_new_signs(tn, oracle, n):
    """Most signs of the request are new and come up several times; every place gets the filled row."""
    rng = np.random.default_rng(n)
    pair = Pair(tn, oracle, "AdaGrad", 16, HP["AdaGrad"], reserve=200000)
    pool = synth.splitmix64(np.arange(1, max(2, n // 3) + 1, dtype=np.uint64))
    pair.populate(pool[::4])
    pool[-1] = np.uint64(0xFFFFFFFFFFFFFFFF)
    for _ in range(2):
        req = dev(pool[rng.integers(0, len(pool), n)].view(np.int64))
        out = tn.ops.table_pull(pair.h, req, 16)
        rows, _, found = tn.ops.table_export_rows(pair.h, req)  # (normally distributed: no new row is all zero)
        assert bool(found.all()) and bool((out == rows).all()) and bool((out != 0).any(1).all())


@pytest.mark.parametrize("n,fresh", [(300, 0), (60000, 0), (60000, 7)])
def test_pulled_rows_are_written_when_the_call_returns(tn, oracle, n, fresh):
    """Read on a stream that nothing orders behind the pull's.  (The rows are a moment behind the workgroups' reports, too
    short for a reader to show it: that the call ends with a launch behind the one that writes them is looked at.)"""
    rng = np.random.default_rng(n)
    pair = Pair(tn, oracle, "AdaGrad", 16, HP["AdaGrad"], reserve=200000)
    base = pair.populate(synth.splitmix64(np.arange(1, 20001, dtype=np.uint64)))
    req = base[rng.integers(0, len(base), n)]
    if fresh:
        req[:fresh] = synth.splitmix64(np.arange(10**6, 10**6 + fresh, dtype=np.uint64))
    signs = dev(req.view(np.int64))
    torch.cuda.synchronize()
    writer, reader = torch.cuda.Stream(), torch.cuda.Stream()
    host = torch.empty((n, 16), pin_memory=True)

    def pull():
        with torch.cuda.stream(writer):
            out = tn.ops.table_pull(pair.h, signs, 16)
        with torch.cuda.stream(reader):
            host.copy_(out, non_blocking=True)
            out.record_stream(reader)

    assert {"k_table_pull", "k_report"} <= kernels_of(tn, pull)
    torch.cuda.synchronize()
    want = tn.ops.table_export_rows(pair.h, signs)[0]
    assert bool((host == want.cpu()).all())


def test_push_of_unknown_signs(tn, oracle):
    """Reported when the table is next waited for, the other records applied; the next push is clean again."""
    rng = np.random.default_rng(5)
    pair = Pair(tn, oracle, "AdaGrad", 8, HP["AdaGrad"])
    base = pair.populate(synth.splitmix64(np.arange(1, 301, dtype=np.uint64)))
    req = np.concatenate([base[rng.integers(0, 300, 700)], synth.splitmix64(np.arange(1000, 1100, dtype=np.uint64))])
    req = req[rng.permutation(len(req))]
    infos, grads = pushed(tn, oracle, pair, req, rng)
    with pytest.raises(tensornet_amd.TensorNetError) as e:
        tn.ops.sparse_table_sync(pair.h)
    assert e.value.code == 5
    known = np.isin(req, base)
    assert pair.o.push(infos[known], grads[known]) == 0
    infos, grads = pushed(tn, oracle, pair, base, rng)
    tn.ops.sparse_table_sync(pair.h)
    assert pair.o.push(infos, grads) == 0
    pair.assert_rows_match(base)
