"""The dense step takes a launch's worth of variables at once, four elements to a thread at any alignment: numbers of
variables around a launch's, lengths around a workgroup's 1024 elements, variables and gradients at odd offsets."""
import numpy as np
import pytest
import torch

from helpers import ATOL, RTOL, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opt", ["Adam", "AdaGrad"])
@pytest.mark.parametrize("sizes,shift", [([1023, 1024, 1025, 1, 3], 0), ([2047, 5, 2049], 1), ([7] * 64, 3), ([9] * 65, 0),
                                         ([1, 0, 2, 4096, 0] * 40, 2)])
def test_dense_segments(tn, oracle, opt, sizes, shift):
    total = sum(sizes)
    rng = np.random.default_rng(total)
    kind = {"Adam": oracle.ADAM, "AdaGrad": oracle.ADAGRAD}[opt]
    hp = {} if opt == "Adam" else dict(initial_g2sum=0.5, epsilon=1e-3, grad_decay_rate=0.9, mom_decay_rate=0.5)
    h = tn.core.create_dense_table(getattr(tn.core, opt)(**hp))
    d = oracle.Dense(kind, total, **hp)
    w0 = rng.uniform(-0.5, 0.5, total).astype(np.float32)
    d.set_weight(w0)

    def split(a):  # consecutive views that start `shift` elements into an allocation
        flat = torch.cat([torch.zeros(shift, device="cuda"), dev(a)])[shift:]
        return list(flat.split(sizes))

    vars_ = split(w0)
    tn.ops.dense_table_init(vars_, h)
    for _ in range(3):
        g = rng.standard_normal(total).astype(np.float32)
        d.apply(g, 1e-2)
        tn.ops.dense_table_push_pull(vars_, split(g), 1e-2, h)
        np.testing.assert_allclose(torch.cat(vars_).cpu().numpy(), d.get_weight(), rtol=RTOL, atol=ATOL)
    assert torch.equal(tn.ops.dense_table_get_weight(h), torch.cat(vars_))
