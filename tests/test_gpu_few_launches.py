"""The launches of a small batch at the sizes where they change: a pull's second half as one launch or two (up to eight
slots, buckets that want much LDS), rows copied one part per thread or two, rows that do not fill the lanes; and buckets
whose wavefronts share signs with one record, with a few and with many, pushed twice on one plan."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth

from helpers import Pair, all_signs, check_pull, dev, kernels_of

pytestmark = pytest.mark.gpu

HP = {"AdaGrad": dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8),
      "Adam": dict(learning_rate=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8),
      "Ftrl": dict(learning_rate=0.05, beta=1.0, lambda1=0.001, lambda2=1.0)}


@pytest.mark.parametrize("slots,per,opt,dim,one_launch", [
    (8, 50, "AdaGrad", 8, False), (9, 50, "AdaGrad", 8, True),     # up to eight slots: two launches
    (140, 60, "Adam", 4, True), (150, 60, "AdaGrad", 4, False),    # 29 and 43 KB of LDS a bucket
    (20, 218, "AdaGrad", 30, True), (20, 219, "AdaGrad", 30, True),  # 2^17 parts of rows: one a thread, then two
    (13, 900, "Ftrl", 128, True), (16, 1025, "AdaGrad", 1, True),  # 32 parts a row, one part a row
])
def test_rows_and_records(tn, oracle, slots, per, opt, dim, one_launch):
    rng = np.random.default_rng(slots * 1009 + per)
    pool = synth.splitmix64(np.arange(1, 4001, dtype=np.uint64)).view(np.int64)
    pair = Pair(tn, oracle, opt, dim, HP[opt], reserve=100000, zero_init=True)
    pair.populate(pool[:3000].view(np.uint64))
    values = []
    for s in range(slots):
        v = pool[(rng.random(per) ** 3 * len(pool)).astype(np.int64)]
        v[:min(6, per)] = pool[:min(6, per)]  # signs with a record in every slot
        values.append(v[:per - s % 3])  # (slots of several lengths)
    counts = check_pull(pair, values)
    gvars = [torch.zeros((len(v) + 1, pair.wf), device="cuda") for v in values]
    gvalues = [dev(v) for v in values]
    names = kernels_of(tn, lambda: tn.ops.sparse_table_pull(gvars, gvalues, pair.h))
    rest = {k for k in names if k.startswith("k_small_pull_rest")}
    assert "k_small_slots" in names and bool(rest) == one_launch and len(names) == (2 if one_launch else 3)
    for seed in range(2):
        grads = synth.make_grads(counts, pair.wf, 0.01, seed=seed)
        pair.push_op(values, grads, [(rng.random(len(v)) < 0.3).astype(np.int64) for v in values])
        assert pair.assert_rows_match(all_signs(values)) > 0.99
    check_pull(pair, values)
