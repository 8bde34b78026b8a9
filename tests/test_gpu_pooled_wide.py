"""Pooled gradients of more examples than 32 bits number: lookups of the first 2^32 are summed, those of examples behind them refused (they
were taken for the examples 2^32 earlier)."""
import numpy as np
import pytest
import torch

from tensornet_amd import synth
from tensornet_amd._lib import TensorNetError

from helpers import Pair, dev
from test_gpu_small_edges import HP

pytestmark = pytest.mark.gpu

LAST = 2 ** 32 - 1


@pytest.mark.parametrize("few_launches", [True, False])
def test_examples_beyond_32_bits(tn, oracle, few_launches):
    pair = Pair(tn, oracle, "AdaGrad", 1, HP, reserve=1000)
    tn.core.set_sparse_table_small_batch_path(pair.h, few_launches)
    base = pair.populate(synth.splitmix64(np.arange(1, 9, dtype=np.uint64)))
    signs = base.view(np.int64)
    grads = torch.empty((LAST + 17, 1), device="cuda")  # (17 GB, of which a few rows are read)
    rows = {3: 0.5, 5: 0.25, LAST: -0.125, LAST + 1 + 5: 8.0, LAST + 16: 16.0}
    for row, g in rows.items():
        grads[row] = g

    def push(examples):
        values = [signs[:len(examples)]]
        labels = [np.zeros(len(examples), np.int64)]
        pair.pull_op(values)
        tn.ops.sparse_table_push_pooled([dev(v) for v in values], [dev(np.array(examples))], [grads], [dev(l) for l in labels],
                                        pair.h, "sum")
        tn.ops.sparse_table_sync(pair.h)
        assert pair.o.push_op(values, [np.array([[rows[e]] for e in examples], np.float32)], labels)[0] == 0

    try:
        push([3, 5, 5, LAST])
        pair.assert_rows_match(base)
        for examples in ([5, LAST + 1 + 5], [LAST, LAST + 16], [3, 5, LAST + 16]):
            with pytest.raises(TensorNetError) as e:
                push(examples)
            assert e.value.code == 1
            pair.assert_rows_match(base)
        push([5, LAST])
        pair.assert_rows_match(base)
    finally:
        del grads
        torch.cuda.empty_cache()
