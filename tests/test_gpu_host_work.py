"""tn_while_waiting (csrc/host_work.h): which calls run the caller's work, how often, and what waits for it meanwhile."""
import ctypes
import threading
import time

import pytest
import torch

from tensornet_amd import _lib, synth

from helpers import Pair, dev

pytestmark = pytest.mark.gpu
HP = dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8)
Fn = ctypes.CFUNCTYPE(None, ctypes.c_void_p)


class Work:
    """A function to call while waiting, and how often it was."""

    def __init__(self, then=lambda: None):
        self.calls = 0

        def fn(arg):
            self.calls += 1
            assert arg == 7
            then()
        self.fn = Fn(fn)
        self.register = _lib.load().tn_while_waiting
        self.register.argtypes = [Fn, ctypes.c_void_p]

    def __enter__(self):
        self.register(self.fn, 7)
        return self

    def __exit__(self, *_):
        self.register(Fn(0), None)


def setup(tn, oracle, small=True):
    pair = Pair(tn, oracle, "AdaGrad", 8, HP, reserve=20000)
    pair.populate(synth.splitmix64(torch.arange(1, 2001).numpy().astype("uint64")))
    tn.core.set_sparse_table_small_batch_path(pair.h, small)
    values = [synth.splitmix64_torch(torch.arange(1, 1501, device="cuda")) for _ in range(3)]
    room = [torch.zeros((1501, 8), device="cuda") for _ in values]
    pull = tn.ops.BoundSparseTablePull(room, values, pair.h)
    return pair, values, room, pull


@pytest.mark.parametrize("small", [True, False])
def test_calls_that_wait_do_it_once(tn, oracle, small):
    pair, values, room, pull = setup(tn, oracle, small)
    with Work() as w:
        mapped = pull()
        assert w.calls == 1
        pull()
        assert w.calls == 1
    examples = [torch.arange(1500, device="cuda") for _ in values]
    combine = tn.ops.BoundEmbeddingLookupSparse(room, mapped, examples, 1500, pair.h, "sum")
    for call in (combine, lambda: tn.ops.table_pull(pair.h, values[0], 8)):
        with Work() as w:
            call()
            assert w.calls == 1


@pytest.mark.parametrize("small", [True, False])
def test_other_calls_leave_it(tn, oracle, small):
    pair, values, room, pull = setup(tn, oracle, small)
    pull()
    grads = [torch.zeros((1500, 8), device="cuda") for _ in values]
    labels = [torch.zeros_like(v) for v in values]
    push = tn.ops.BoundSparseTablePush(values, grads, labels, pair.h)
    no_such_table = tn.ops.BoundSparseTablePull(room, values, pair.h + 1000)
    with Work() as w:
        push()
        with pytest.raises(_lib.TensorNetError):
            no_such_table()
        tn.core.set_sparse_table_async(pair.h, True)
        pull()
        tn.core.set_sparse_table_async(pair.h, False)
        assert w.calls == 0
        pull()
        assert w.calls == 1
    with Work() as w:
        pass
    pull()  # taken back
    assert w.calls == 0


def test_another_threads_call_on_the_table_waits(tn, oracle):
    pair, values, room, pull = setup(tn, oracle)
    other, _, _, _ = setup(tn, oracle)
    pull()
    ended = {}

    def count(h):
        tn.core.sparse_table_key_count(h)
        ended[h] = time.monotonic()

    threads = [threading.Thread(target=count, args=(h,)) for h in (pair.h, other.h)]
    left = []

    def work():
        for t in threads:
            t.start()
        threads[1].join(10)  # another table's call does not wait
        time.sleep(0.05)
        left.append(time.monotonic())

    with Work(work) as w:
        pull()
    for t in threads:
        t.join(10)
    assert w.calls == 1 and ended[other.h] < left[0] < ended[pair.h]
