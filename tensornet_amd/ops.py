"""Operator surface of the hot path: the four TensorFlow ops of the reference
(core/ops/sparse_table_ops.cc:21-53, core/ops/dense_table_ops.cc:21-37, Python
wrappers tensornet/core/gen_sparse_table_ops.py / gen_dense_table_ops.py) with
the same names and argument order, taking torch tensors that live on the GPU.
Tensors are only used as device memory: every call goes through the C ABI with
raw device pointers and the current HIP stream.  The operators that run in every
step are marshalled by a native module (csrc/bind.cc), the others through ctypes.

A "resource" (tf.Variable handle in the reference) is here the variable's
torch tensor itself, updated in place.
"""
import ctypes as C

import torch

from . import _lib

_bind = _lib.load_bind()


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _require(t, dtype, what):
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise ValueError("%s must be a CUDA/HIP tensor" % what)
    if t.dtype != dtype:
        raise ValueError("%s must have dtype %s, got %s" % (what, dtype, t.dtype))
    if not t.is_contiguous():
        raise ValueError("%s must be contiguous" % what)


class BoundSparseTablePull:
    """SparseTablePull bound to fixed tensors, the way an op kernel of a built
    graph sees its inputs: arguments are validated and marshalled once, the
    mapped-id outputs allocated once; every call only crosses the C ABI (with the
    stream current at that moment).  Calling it returns the N mapped-id tensors."""

    def __init__(self, resources, values, table_handle):
        self._call = _bind.bind_pull(resources, values, table_handle)
        self.mapped = self._call.outputs

    def __call__(self):
        return self._call()


class BoundSparseTablePush:
    """SparseTablePush bound to fixed tensors (see BoundSparseTablePull)."""

    def __init__(self, values, grads, feature_labels, table_handle):
        self._call = _bind.bind_push(values, grads, feature_labels, table_handle)

    def __call__(self):
        self._call()


def sparse_table_pull(resources, values, table_handle):
    """SparseTablePull.  resources: N float32 variables [rows, dim] (updated in
    place: row j <- embedding of the j-th distinct sign of the slot);
    values: N int64 rank-1 tensors of signs.  Returns N int64 tensors of mapped
    ids (same shapes as values)."""
    return _bind.sparse_table_pull(resources, values, table_handle)


def sparse_table_push(values, grads, feature_labels, table_handle):
    """SparseTablePush.  grads[i] is [U_i, dim] with row j the gradient of the
    j-th distinct sign of values[i]; feature_labels[i] has one int64 label per
    lookup.  Returns nothing (the update is enqueued on the current stream)."""
    _bind.sparse_table_push(values, grads, feature_labels, table_handle)


COMBINERS = {"sum": 0, "mean": 1, "sqrtn": 2}


def _combiner(combiner):
    if combiner not in COMBINERS:
        raise ValueError("combiner must be one of 'sum', 'mean', 'sqrtn', got %r" % (combiner,))
    return COMBINERS[combiner]


def embedding_lookup_sparse(resources, mapped_values, example_ids, batch_size, table_handle, combiner="mean"):
    """What TensorFlow does with the pull's results for every slot
    (tf.nn.embedding_lookup_sparse behind embedding_column.get_dense_tensor,
    tensornet/layers/embedding_features.py:278-280): out[s][b] = combiner over
    the rows resources[s][mapped_values[s][i]] of the lookups i of example b.
    example_ids[s][i] is the example of lookup i (SparseTensor.indices[:, 0]).
    Returns N float32 tensors [batch_size, dim]."""
    return _bind.embedding_lookup_sparse(resources, mapped_values, example_ids, batch_size, table_handle, _combiner(combiner))


class BoundEmbeddingLookupSparse:
    """embedding_lookup_sparse bound to fixed tensors (see BoundSparseTablePull): the variables and mapped ids of a
    bound pull, the example ids, and outputs allocated once.  Calling it returns the N [batch_size, dim] tensors."""

    def __init__(self, resources, mapped_values, example_ids, batch_size, table_handle, combiner="mean"):
        self._call = _bind.bind_combine(resources, mapped_values, example_ids, batch_size, table_handle, _combiner(combiner))
        self.out = self._call.outputs

    def __call__(self):
        return self._call()


class BoundSparseTablePushPooled:
    """SparseTablePush fed with the gradients of the combiner's outputs
    (pooled_grads[s]: [batch_size, dim]) instead of per-distinct-sign rows; the
    reduction TensorFlow performs in between (gradient of embedding_lookup_sparse
    summed per distinct id) runs on the device.  Bound to fixed tensors like
    BoundSparseTablePush."""

    def __init__(self, values, example_ids, pooled_grads, feature_labels, table_handle, combiner="mean"):
        self._call = _bind.bind_push_pooled(values, example_ids, pooled_grads, feature_labels, table_handle,
                                            _combiner(combiner))

    def __call__(self):
        self._call()


def sparse_table_push_pooled(values, example_ids, pooled_grads, feature_labels, table_handle, combiner="mean"):
    _bind.sparse_table_push_pooled(values, example_ids, pooled_grads, feature_labels, table_handle, _combiner(combiner))


def sparse_table_sync(table_handle):
    """Waits for enqueued pushes of the table and raises their latched error."""
    _lib.check(_lib.load().tn_sparse_table_sync(table_handle))


def sparse_table_last_unique_counts(table_handle, n_slots):
    out = (C.c_int64 * n_slots)()
    _lib.check(_lib.load().tn_sparse_table_last_unique_counts(table_handle, n_slots, out))
    return [int(x) for x in out]


def dense_table_init(vars, table_handle):
    """DenseTableInit: the table takes the concatenation of the variables."""
    for i, v in enumerate(vars):
        _require(v, torch.float32, "vars[%d]" % i)
    rc = _lib.load().tn_dense_table_init(
        table_handle,
        len(vars),
        _lib.ptr_array([v.data_ptr() for v in vars]),
        _lib.i64_array([v.numel() for v in vars]),
        _stream(),
    )
    _lib.check(rc)


def dense_table_push_pull(vars, grads, learning_rate, table_handle):
    """DenseTablePushPull: optimizer step with the concatenated gradients, new
    weights written back into the variables (in place)."""
    _bind.dense_table_push_pull(vars, grads, learning_rate, table_handle)


# ------------------------------------------------------------ table level
def table_pull(table_handle, signs, dim):
    """SparseTable::Pull: signs int64/uint64-as-int64 [n] -> float32 [n, dim]."""
    return _bind.table_pull(table_handle, signs, dim)


def table_push(table_handle, sign_infos, grads):
    """SparseTable::Push: sign_infos is an int64 tensor [n, 2] holding the 16-byte
    records (sign, batch_show | batch_click << 32); grads float32 [n, dim]."""
    _bind.table_push(table_handle, sign_infos, grads)


def make_sign_infos(signs, shows, clicks):
    """Packs int64 signs and int32-valued shows/clicks into 16-byte records."""
    rec = torch.empty((signs.numel(), 2), dtype=torch.int64, device=signs.device)
    rec[:, 0] = signs
    rec[:, 1] = (shows.to(torch.int64) & 0xFFFFFFFF) | (clicks.to(torch.int64) << 32)
    return rec


def table_load_rows(table_handle, signs, w, state=None):
    _require(signs, torch.int64, "signs")
    _require(w, torch.float32, "w")
    if state is not None:
        _require(state, torch.float32, "state")
    rc = _lib.load().tn_sparse_table_load_rows(
        table_handle,
        signs.data_ptr(),
        w.data_ptr(),
        state.data_ptr() if state is not None else None,
        signs.numel(),
        _stream(),
    )
    _lib.check(rc)


def table_export_rows(table_handle, signs):
    from .core import sparse_table_row_layout

    _require(signs, torch.int64, "signs")
    wf, sf = sparse_table_row_layout(table_handle)
    n = signs.numel()
    w = torch.empty((n, wf), dtype=torch.float32, device=signs.device)
    st = torch.empty((n, sf), dtype=torch.float32, device=signs.device)
    found = torch.empty((n,), dtype=torch.uint8, device=signs.device)
    rc = _lib.load().tn_sparse_table_export_rows(
        table_handle, signs.data_ptr(), n, w.data_ptr(), st.data_ptr(), found.data_ptr(), _stream()
    )
    _lib.check(rc)
    return w, st, found


def table_delete_by_show(table_handle, signs):
    """Value::DeleteByShow for the rows of `signs` (uint8 tensor: 1 = the row would be left out of
    a saved table, 0 = kept or absent)."""
    _require(signs, torch.int64, "signs")
    out = torch.empty((signs.numel(),), dtype=torch.uint8, device=signs.device)
    _lib.check(_lib.load().tn_sparse_table_delete_by_show(table_handle, signs.data_ptr(), signs.numel(),
                                                          out.data_ptr(), _stream()))
    return out


def dense_table_range(table_handle):
    """(begin, end) of the table's elements this shard holds (optimizer_kernel.h:55-57)."""
    b, e = C.c_int64(), C.c_int64()
    _lib.check(_lib.load().tn_dense_table_range(table_handle, C.byref(b), C.byref(e)))
    return b.value, e.value


def dense_table_get_weight(table_handle, device="cuda"):
    b, e = dense_table_range(table_handle)
    w = torch.empty((e - b,), dtype=torch.float32, device=device)
    _lib.check(_lib.load().tn_dense_table_get_weight(table_handle, w.data_ptr(), _stream()))
    return w


def dense_table_get_state(table_handle, n_states=2, device="cuda"):
    b, e = dense_table_range(table_handle)
    outs = [torch.empty((e - b,), dtype=torch.float32, device=device) for _ in range(n_states)]
    ptrs = [o.data_ptr() for o in outs] + [None] * (3 - n_states)
    _lib.check(_lib.load().tn_dense_table_get_state(table_handle, ptrs[0], ptrs[1], ptrs[2], _stream()))
    return outs
