"""Table-level push with as many workgroups as the chip holds of the update kernel's variants for few of them, and with one more: rows
whose variant for many has chunks of four rounds or fewer registers, in 16-byte pieces and at any address, signs with many records."""
import numpy as np
import pytest

from tensornet_amd import synth

from helpers import Pair, dev, kernels_of

from test_gpu_table_level import HP, pushed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opt,dim", [("AdaGrad", d) for d in (8, 10, 12, 16, 32, 64, 100, 128)] + [("Adam", 64), ("Ftrl", 8), ("Ftrl", 16), ("Ftrl", 64)])
@pytest.mark.parametrize("more", [0, 1])
def test_push_by_many_workgroups(tn, oracle, opt, dim, more):
    n = 128 * (512 if opt == "AdaGrad" else 768) + more
    rng = np.random.default_rng(n + dim)
    pair = Pair(tn, oracle, opt, dim, HP[opt], reserve=100000)
    base = pair.populate(synth.splitmix64(np.arange(1, 30001, dtype=np.uint64)))
    req = base[(rng.random(n) ** 6 * len(base)).astype(np.int64)]
    out = []
    names = kernels_of(tn, lambda: out.append(pushed(tn, oracle, pair, req, rng)))
    assert [k.endswith(", true)>") for k in names if k.startswith("k_table_apply<")] == [bool(more)]  # (the variant for many workgroups)
    infos, grads = out[0]
    assert pair.o.push(infos, grads) == 0
    pair.assert_rows_match(base)


@pytest.mark.parametrize("dim", [16, 64])
def test_gradients_at_any_address(tn, oracle, dim):
    n = 128 * 512 + 1
    rng = np.random.default_rng(dim)
    pair = Pair(tn, oracle, "AdaGrad", dim, HP["AdaGrad"], reserve=100000)
    base = pair.populate(synth.splitmix64(np.arange(1, 30001, dtype=np.uint64)))
    req = base[(rng.random(n) ** 6 * len(base)).astype(np.int64)]
    infos = np.zeros(n, dtype=oracle.sign_info_dtype)
    infos["sign"], infos["batch_show"], infos["batch_click"] = req, rng.integers(1, 5, n), rng.integers(0, 2, n)
    grads = (rng.standard_normal((n, dim)) * 0.01).astype(np.float32)
    flat = dev(np.concatenate([np.zeros(1, np.float32), grads.reshape(-1)]))  # (rows four bytes behind a 16-byte boundary)
    records = tn.ops.make_sign_infos(dev(req.view(np.int64)), dev(infos["batch_show"].astype(np.int64)),
                                     dev(infos["batch_click"].astype(np.int64)))
    names = kernels_of(tn, lambda: tn.ops.table_push(pair.h, records, flat[1:].view(n, dim)))
    assert [k.endswith(", true)>") and ", true, " in k for k in names if k.startswith("k_table_apply<")] == [True]  # (any address)
    assert pair.o.push(infos, grads) == 0
    pair.assert_rows_match(base)
