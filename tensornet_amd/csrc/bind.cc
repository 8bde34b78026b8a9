// Python binding of the operators (tensornet_amd/ops.py): reads the tensors' addresses and sizes, calls the C ABI of
// include/tensornet_amd.h and hands the outputs back.  Host code only.
//
// An operator of N slots looks at 3 to 4 N tensors a call and pull returns N of them.  Through ctypes a tensor cost
// 0.35 us to check and marshal and an output view 0.6 us -- 0.4 ms per pull + push of 100 slots, 1.2 ms for a step of
// 211 slots with the combiner, most of it while the device had nothing to do.  Here it is 10-20 ns per tensor and 0.15 us
// per output view, and a bound operator's call costs 0.2 us instead of 5.
//
// The interpreter's lock is released while the library runs, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <memory>
#include <string>
#include <vector>

#include "host_work.h"
#include "tensornet_amd.h"

namespace {

PyObject* g_error_class = nullptr;  // tensornet_amd._lib.TensorNetError

// A Python exception is set: unwinds to the entry point.
struct PyFailed {};

[[noreturn]] void value_error(const std::string& what) {
    PyErr_SetString(PyExc_ValueError, what.c_str());
    throw PyFailed{};
}

[[noreturn]] void status_error(int code, const std::string& what) {
    PyObject* args = Py_BuildValue("(is)", code, what.c_str());
    if (args) {
        PyErr_SetObject(g_error_class, args);
        Py_DECREF(args);
    }
    throw PyFailed{};
}

// The items of a sequence argument, in a tuple of their own: another thread may clear or refill the caller's list while
// the library runs without the interpreter's lock.
class Items {
public:
    explicit Items(PyObject* o) : items_(PySequence_Tuple(o)) {
        if (!items_) throw PyFailed{};
    }
    Items(const Items&) = delete;
    ~Items() { Py_DECREF(items_); }
    Py_ssize_t size() const { return PyTuple_GET_SIZE(items_); }
    PyObject* operator[](Py_ssize_t i) const { return PyTuple_GET_ITEM(items_, i); }
    // The tuple (a new reference).
    PyObject* tuple() const {
        Py_INCREF(items_);
        return items_;
    }

private:
    PyObject* items_;
};

// A contiguous device tensor of the given type, or a ValueError that names it.
const at::Tensor& require(PyObject* o, at::ScalarType type, const char* name, Py_ssize_t i = -1) {
    auto what = [&] { return i < 0 ? std::string(name) : std::string(name) + "[" + std::to_string(i) + "]"; };
    if (!THPVariable_Check(o)) value_error(what() + " must be a CUDA/HIP tensor");
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) value_error(what() + " must be a CUDA/HIP tensor");
    if (t.scalar_type() != type)
        value_error(what() + " must have dtype " + (type == at::kFloat ? "torch.float32" : "torch.int64") + ", got " +
                    "torch." + torch::getTHPDtype(t.scalar_type())->name);
    if (!t.is_contiguous()) value_error(what() + " must be contiguous");
    return t;
}

std::string shape_text(const at::Tensor& t) {
    std::string s = "(";
    for (int64_t d : t.sizes()) s += std::to_string(d) + ", ";
    if (t.dim() > 1) s.resize(s.size() - 2);
    return s + ")";
}

uint32_t handle_arg(PyObject* o) {
    PyObject* n = PyNumber_Index(o);
    if (!n) throw PyFailed{};
    const unsigned long v = PyLong_AsUnsignedLongMask(n);
    Py_DECREF(n);
    return (uint32_t)v;
}

int64_t int_arg(PyObject* o) {
    PyObject* n = PyNumber_Index(o);
    if (!n) throw PyFailed{};
    const long long v = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (v == -1 && PyErr_Occurred()) throw PyFailed{};
    return (int64_t)v;
}

void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// `columns` arrays of n words each in one allocation: what the C ABI takes as arrays of pointers and lengths.
class Words {
public:
    Words(int n, int columns) : n_(n), w_(new int64_t[(size_t)n * columns]) {}
    int64_t* lens(int column) { return w_.get() + (size_t)column * n_; }
    template <typename T>
    T** ptrs(int column) {
        static_assert(sizeof(T*) == sizeof(int64_t), "64-bit pointers");
        return reinterpret_cast<T**>(w_.get() + (size_t)column * n_);
    }

private:
    int n_;
    std::unique_ptr<int64_t[]> w_;
};

// One marshalled call of the library.
struct Call {
    virtual ~Call() { Py_XDECREF(outputs); }
    virtual int run(void* stream) = 0;
    PyObject* outputs = nullptr;  // what a bound operator returns, held by the call; nullptr: None
};

void finish(int rc) {
    if (rc != TN_OK) status_error(rc, tn_last_error());
}

// The interpreter's lock is released while this lives (an exception that passes it finds the lock held again).
class Unlocked {
public:
    Unlocked() : state_(PyEval_SaveThread()) {}
    Unlocked(const Unlocked&) = delete;
    ~Unlocked() { PyEval_RestoreThread(state_); }

private:
    PyThreadState* state_;
};

// A call of the library without the interpreter's lock; an error status becomes Python's exception.
template <typename F>
void call_library(F f) {
    int rc;
    {
        const Unlocked unlocked;
        rc = f();
    }
    finish(rc);
}

void run(Call& c) {
    void* stream = current_stream();
    call_library([&] { return c.run(stream); });
}

// n tensors that are consecutive parts of `flat` (as torch.split hands them out), without the dispatcher.  Half of what a view
// takes is the tensor, which needs no interpreter (build), the other half its Python object (take).
class Views {
public:
    Views(const at::Tensor& flat, Py_ssize_t n) : flat_(flat), n_((size_t)n) { made_.reserve(n_); }
    Views(const Views&) = delete;
    // sizes(i): the next view's; those that build() has not come to are made by take().
    template <typename Sizes>
    void build(Sizes sizes) {
        while (made_.size() < n_) {
            const auto dims = sizes(made_.size());
            auto impl = c10::make_intrusive<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(flat_.storage()),
                                                             flat_.key_set(), flat_.dtype());
            impl->set_storage_offset(offset_);
            impl->set_sizes_contiguous(dims);
            impl->set_version_counter(flat_.unsafeGetTensorImpl()->version_counter());
            offset_ += impl->numel();
            made_.emplace_back(std::move(impl));
        }
    }
    template <typename Sizes>
    PyObject* take(Sizes sizes) {
        build(sizes);
        PyObject* list = PyList_New((Py_ssize_t)n_);
        if (!list) throw PyFailed{};
        for (size_t i = 0; i < n_; i++) {
            PyObject* o = THPVariable_Wrap(std::move(made_[i]));
            if (!o) {
                Py_DECREF(list);
                throw PyFailed{};
            }
            PyList_SET_ITEM(list, (Py_ssize_t)i, o);
        }
        return list;
    }

private:
    const at::Tensor& flat_;
    const size_t n_;
    std::vector<at::Tensor> made_;
    int64_t offset_ = 0;
};

// A call with outputs: their tensors are made while it waits for the device, which has nothing to do once it has reported.
// (The tensors only, without the interpreter's lock: taking it in the middle of a call would have the call wait for other
// Python threads.)  Pull and combine of 26 slots 46.4 -> 44.3 us; with the pooled push, 211 slots, 361 -> 354.
template <typename C>
PyObject* run_for_views(C& c) {
    struct Work {
        C& call;
        Views views;
    } work{c, Views(c.flat, c.n)};
    tn_while_waiting(
        [](void* p) {
            Work& w = *static_cast<Work*>(p);
            try {
                w.views.build([&](size_t i) { return w.call.view_sizes(i); });
            } catch (...) {  // (out of memory: take() tries again, and reports it)
            }
        },
        &work);
    struct TakeBack {
        ~TakeBack() { tn_while_waiting(nullptr, nullptr); }
    } take_back;
    run(c);
    return work.views.take([&](size_t i) { return c.view_sizes(i); });
}

struct PullCall : Call {
    uint32_t handle;
    int n, dim = 0;
    Words w;
    at::Tensor flat;

    static int slots(const Items& resources, const Items& values) {
        const Py_ssize_t n = values.size();
        if (resources.size() != n)
            value_error("SparseTable pull num_inputs: " + std::to_string(resources.size() + n) +
                        " not equal: " + std::to_string(n * 2));
        if (n == 0) value_error("SparseTable pull needs at least one slot");
        return (int)n;
    }

    PullCall(const Items& resources, const Items& values, uint32_t h)
        : handle(h), n(slots(resources, values)), w(n, 5) {
        int64_t total = 0;
        for (int i = 0; i < n; i++) {
            const at::Tensor& r = require(resources[i], at::kFloat, "resources", i);
            const at::Tensor& v = require(values[i], at::kLong, "values", i);
            if (r.dim() != 2) value_error("sparse pull variable must Matrix(sign_id_cnt, dim), saw: " + shape_text(r));
            if (v.dim() != 1) value_error("values[" + std::to_string(i) + "] must have rank 1");
            if (i == 0)
                dim = (int)r.size(1);
            else if (dim != r.size(1))
                status_error(TN_ERR_DIM_MISMATCH, "all variables of one pull must have the same dim");
            w.ptrs<int64_t>(0)[i] = (int64_t*)v.data_ptr();
            w.lens(1)[i] = v.numel();
            w.ptrs<float>(2)[i] = (float*)r.data_ptr();
            w.lens(3)[i] = r.size(0);
            total += v.numel();
        }
        // one allocation for all mapped ids, handed out as per-slot views
        flat = at::empty({total}, THPVariable_Unpack(values[0]).options());
        int64_t* p = (int64_t*)flat.data_ptr();
        for (int i = 0; i < n; i++) {
            w.ptrs<int64_t>(4)[i] = p;
            p += w.lens(1)[i];
        }
    }
    std::array<int64_t, 1> view_sizes(size_t i) { return {w.lens(1)[i]}; }
    int run(void* stream) override {
        return tn_sparse_table_pull_op(handle, n, w.ptrs<const int64_t>(0), w.lens(1), w.ptrs<float>(2), w.lens(3), dim,
                                       w.ptrs<int64_t>(4), stream);
    }
};

struct PushCall : Call {
    uint32_t handle;
    int n, dim = 0;
    Words w;

    static int slots(const Items& values, const Items& grads, const Items& labels) {
        const Py_ssize_t n = values.size();
        if (grads.size() != n || labels.size() != n)
            value_error("SparseTable push num_inputs: " + std::to_string(n + grads.size() + labels.size()) +
                        " not equal: " + std::to_string(n * 3));
        if (n == 0) value_error("SparseTable push needs at least one slot");
        return (int)n;
    }

    PushCall(const Items& values, const Items& grads, const Items& labels, uint32_t h)
        : handle(h), n(slots(values, grads, labels)), w(n, 5) {
        for (int i = 0; i < n; i++) {
            const at::Tensor& v = require(values[i], at::kLong, "values", i);
            const at::Tensor& g = require(grads[i], at::kFloat, "grads", i);
            const at::Tensor& l = require(labels[i], at::kLong, "feature_labels", i);
            if (g.dim() != 2) value_error("sparse push grad must Matrix(sign_id_cnt, dim), saw: " + shape_text(g));
            if (l.numel() != v.numel())
                value_error("feature_labels[" + std::to_string(i) + "] must have one label per lookup");
            if (i == 0)
                dim = (int)g.size(1);
            else if (dim != g.size(1))
                status_error(TN_ERR_DIM_MISMATCH, "all gradients of one push must have the same dim");
            w.ptrs<int64_t>(0)[i] = (int64_t*)v.data_ptr();
            w.lens(1)[i] = v.numel();
            w.ptrs<float>(2)[i] = (float*)g.data_ptr();
            w.lens(3)[i] = g.size(0);
            w.ptrs<int64_t>(4)[i] = (int64_t*)l.data_ptr();
        }
    }
    int run(void* stream) override {
        return tn_sparse_table_push_op(handle, n, w.ptrs<const int64_t>(0), w.lens(1), w.ptrs<const float>(2), w.lens(3),
                                       dim, w.ptrs<const int64_t>(4), stream);
    }
};

struct CombineCall : Call {
    uint32_t handle;
    int n, dim = 0, combiner;
    int64_t batch;
    Words w;
    at::Tensor flat;

    static int slots(const Items& resources, const Items& mapped, const Items& examples) {
        const Py_ssize_t n = mapped.size();
        if (resources.size() != n || examples.size() != n || n == 0)
            value_error("embedding_lookup_sparse needs one variable, id tensor and example-id tensor per slot");
        return (int)n;
    }

    CombineCall(const Items& resources, const Items& mapped, const Items& examples, int64_t batch_size, uint32_t h, int comb)
        : handle(h), n(slots(resources, mapped, examples)), combiner(comb), batch(batch_size), w(n, 6) {
        for (int i = 0; i < n; i++) {
            const at::Tensor& r = require(resources[i], at::kFloat, "resources", i);
            const at::Tensor& m = require(mapped[i], at::kLong, "mapped_values", i);
            const at::Tensor& e = require(examples[i], at::kLong, "example_ids", i);
            if (e.numel() != m.numel())
                value_error("example_ids[" + std::to_string(i) + "] must have one entry per lookup");
            w.ptrs<int64_t>(0)[i] = (int64_t*)m.data_ptr();
            w.lens(1)[i] = m.numel();
            w.ptrs<int64_t>(2)[i] = (int64_t*)e.data_ptr();
            w.ptrs<float>(3)[i] = (float*)r.data_ptr();
            w.lens(4)[i] = r.size(0);
        }
        const at::Tensor& r0 = THPVariable_Unpack(resources[0]);
        dim = (int)r0.size(1);
        flat = at::empty({n, batch, dim}, r0.options().requires_grad(false));
        for (int i = 0; i < n; i++) w.ptrs<float>(5)[i] = (float*)flat.data_ptr() + (int64_t)i * batch * dim;
    }
    std::array<int64_t, 2> view_sizes(size_t) { return {batch, (int64_t)dim}; }
    int run(void* stream) override {
        return tn_sparse_table_combine_op(handle, n, w.ptrs<const int64_t>(0), w.lens(1), w.ptrs<const int64_t>(2),
                                          w.ptrs<const float>(3), w.lens(4), dim, batch, combiner, w.ptrs<float>(5), stream);
    }
};

struct PooledCall : Call {
    uint32_t handle;
    int n, dim = 0, combiner;
    int64_t batch = 0;
    Words w;

    static int slots(const Items& values, const Items& examples, const Items& grads, const Items& labels) {
        const Py_ssize_t n = values.size();
        if (examples.size() != n || grads.size() != n || labels.size() != n || n == 0)
            value_error("SparseTable push (pooled) needs values, example ids, gradients and labels per slot");
        return (int)n;
    }

    PooledCall(const Items& values, const Items& examples, const Items& grads, const Items& labels, uint32_t h, int comb)
        : handle(h), n(slots(values, examples, grads, labels)), combiner(comb), w(n, 5) {
        for (int i = 0; i < n; i++) {
            const at::Tensor& v = require(values[i], at::kLong, "values", i);
            const at::Tensor& e = require(examples[i], at::kLong, "example_ids", i);
            const at::Tensor& g = require(grads[i], at::kFloat, "pooled_grads", i);
            const at::Tensor& l = require(labels[i], at::kLong, "feature_labels", i);
            if (i == 0 && g.dim() == 2) {
                batch = g.size(0);
                dim = (int)g.size(1);
            }
            if (g.dim() != 2 || g.size(0) != batch || g.size(1) != dim)
                value_error("pooled_grads must all be Matrix(batch_size, dim)");
            if (e.numel() != v.numel() || l.numel() != v.numel())
                value_error("example_ids / feature_labels of slot " + std::to_string(i) + " must have one entry per lookup");
            w.ptrs<int64_t>(0)[i] = (int64_t*)v.data_ptr();
            w.lens(1)[i] = v.numel();
            w.ptrs<int64_t>(2)[i] = (int64_t*)e.data_ptr();
            w.ptrs<float>(3)[i] = (float*)g.data_ptr();
            w.ptrs<int64_t>(4)[i] = (int64_t*)l.data_ptr();
        }
    }
    int run(void* stream) override {
        return tn_sparse_table_push_pooled_op(handle, n, w.ptrs<const int64_t>(0), w.lens(1), w.ptrs<const int64_t>(2),
                                              w.ptrs<const float>(3), batch, dim, combiner, w.ptrs<const int64_t>(4), stream);
    }
};

// Every entry point: C++ exceptions (torch's among them) become Python's.
template <typename F>
PyObject* guarded(F f) {
    try {
        return f();
    } catch (const PyFailed&) {
        return nullptr;
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
        return nullptr;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// ------------------------------------------------------------ bound operators
// A call marshalled once: holds what it reads (the items it was marshalled from, as tuples) and its outputs.
struct Bound {
    PyObject_HEAD
    Call* call;
    PyObject* keep;
};

void bound_dealloc(PyObject* self) {
    Bound* b = reinterpret_cast<Bound*>(self);
    delete b->call;
    Py_XDECREF(b->keep);
    Py_TYPE(self)->tp_free(self);
}

PyObject* bound_call(PyObject* self, PyObject*, PyObject*) {
    return guarded([&] {
        Bound* b = reinterpret_cast<Bound*>(self);
        run(*b->call);
        PyObject* out = b->call->outputs ? b->call->outputs : Py_None;
        Py_INCREF(out);
        return out;
    });
}

PyObject* bound_outputs(PyObject* self, void*) {
    Bound* b = reinterpret_cast<Bound*>(self);
    PyObject* out = b->call->outputs ? b->call->outputs : Py_None;
    Py_INCREF(out);
    return out;
}

PyGetSetDef bound_getset[] = {{"outputs", bound_outputs, nullptr, "the tensors every call writes and returns", nullptr},
                              {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyTypeObject BoundType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// sequences: the items the call was marshalled from, which it needs as long as it lives.  (An argument may be an iterator:
// going over it again would find nothing.)
PyObject* make_bound(std::unique_ptr<Call> call, std::initializer_list<const Items*> sequences) {
    Bound* b = PyObject_New(Bound, &BoundType);
    if (!b) throw PyFailed{};
    b->call = call.release();
    b->keep = PyTuple_New((Py_ssize_t)sequences.size());  // (bound_dealloc takes nullptr, too)
    PyObject* self = reinterpret_cast<PyObject*>(b);
    try {
        if (!b->keep) throw PyFailed{};
        Py_ssize_t i = 0;
        for (const Items* s : sequences) PyTuple_SET_ITEM(b->keep, i++, s->tuple());
    } catch (const PyFailed&) {
        Py_DECREF(self);
        throw;
    }
    return self;
}

void arg_count(Py_ssize_t have, Py_ssize_t want, const char* name) {
    if (have == want) return;
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, want, have);
    throw PyFailed{};
}

PyObject* none() { Py_RETURN_NONE; }

PyObject* py_pull(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 3, "sparse_table_pull");
        const Items resources(a[0]), values(a[1]);
        PullCall c(resources, values, handle_arg(a[2]));
        return run_for_views(c);
    });
}

PyObject* py_bind_pull(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 3, "bind_pull");
        const Items resources(a[0]), values(a[1]);
        auto c = std::make_unique<PullCall>(resources, values, handle_arg(a[2]));
        c->outputs = Views(c->flat, c->n).take([&](size_t i) { return c->view_sizes(i); });
        return make_bound(std::move(c), {&resources, &values});
    });
}

PyObject* py_push(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 4, "sparse_table_push");
        const Items values(a[0]), grads(a[1]), labels(a[2]);
        PushCall c(values, grads, labels, handle_arg(a[3]));
        run(c);
        return none();
    });
}

PyObject* py_bind_push(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 4, "bind_push");
        const Items values(a[0]), grads(a[1]), labels(a[2]);
        return make_bound(std::make_unique<PushCall>(values, grads, labels, handle_arg(a[3])), {&values, &grads, &labels});
    });
}

PyObject* py_combine(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 6, "embedding_lookup_sparse");
        const Items resources(a[0]), mapped(a[1]), examples(a[2]);
        CombineCall c(resources, mapped, examples, int_arg(a[3]), handle_arg(a[4]), (int)int_arg(a[5]));
        return run_for_views(c);
    });
}

PyObject* py_bind_combine(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 6, "bind_combine");
        const Items resources(a[0]), mapped(a[1]), examples(a[2]);
        auto c = std::make_unique<CombineCall>(resources, mapped, examples, int_arg(a[3]), handle_arg(a[4]), (int)int_arg(a[5]));
        c->outputs = Views(c->flat, c->n).take([&](size_t i) { return c->view_sizes(i); });
        return make_bound(std::move(c), {&resources, &mapped, &examples});
    });
}

PyObject* py_push_pooled(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 6, "sparse_table_push_pooled");
        const Items values(a[0]), examples(a[1]), grads(a[2]), labels(a[3]);
        PooledCall c(values, examples, grads, labels, handle_arg(a[4]), (int)int_arg(a[5]));
        run(c);
        return none();
    });
}

PyObject* py_bind_push_pooled(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 6, "bind_push_pooled");
        const Items values(a[0]), examples(a[1]), grads(a[2]), labels(a[3]);
        return make_bound(std::make_unique<PooledCall>(values, examples, grads, labels, handle_arg(a[4]), (int)int_arg(a[5])),
                          {&values, &examples, &grads, &labels});
    });
}

PyObject* py_dense_push_pull(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 4, "dense_table_push_pull");
        const Items vars(a[0]), grads(a[1]);
        const double lr = PyFloat_AsDouble(a[2]);
        if (lr == -1.0 && PyErr_Occurred()) throw PyFailed{};
        const uint32_t handle = handle_arg(a[3]);
        if (vars.size() != grads.size())
            value_error("DenseTable pushpull num_inputs: " + std::to_string(vars.size() + grads.size() + 1) +
                        " not equal: " + std::to_string(2 * vars.size() + 1));
        const int n = (int)vars.size();
        Words w(n, 3);
        for (int i = 0; i < n; i++) {
            const at::Tensor& v = require(vars[i], at::kFloat, "vars", i);
            const at::Tensor& g = require(grads[i], at::kFloat, "grads", i);
            if (v.numel() != g.numel())
                value_error("DenseTable var tensor length: " + std::to_string(v.numel()) +
                            " not equal grad tensor length: " + std::to_string(g.numel()));
            w.ptrs<float>(0)[i] = (float*)v.data_ptr();
            w.ptrs<float>(1)[i] = (float*)g.data_ptr();
            w.lens(2)[i] = g.numel();
        }
        void* stream = current_stream();
        call_library([&] {
            return tn_dense_table_push_pull(handle, n, w.ptrs<float>(0), w.ptrs<const float>(1), w.lens(2), (float)lr, stream);
        });
        return none();
    });
}

PyObject* py_table_pull(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 3, "table_pull");
        const uint32_t handle = handle_arg(a[0]);
        const at::Tensor& signs = require(a[1], at::kLong, "signs");
        const int64_t n = signs.numel(), dim = int_arg(a[2]);
        at::Tensor out = at::empty({n, dim}, signs.options().dtype(at::kFloat));
        const uint64_t* s = (const uint64_t*)signs.data_ptr();
        float* o = (float*)out.data_ptr();
        void* stream = current_stream();
        call_library([&] { return tn_sparse_table_pull(handle, s, n, (int)dim, o, stream); });
        return THPVariable_Wrap(std::move(out));
    });
}

PyObject* py_table_push(PyObject*, PyObject* const* a, Py_ssize_t na) {
    return guarded([&] {
        arg_count(na, 3, "table_push");
        const uint32_t handle = handle_arg(a[0]);
        const at::Tensor& infos = require(a[1], at::kLong, "sign_infos");
        const at::Tensor& grads = require(a[2], at::kFloat, "grads");
        if (grads.dim() < 2) {
            PyErr_SetString(PyExc_IndexError, "grads must be [n, dim]");
            throw PyFailed{};
        }
        const tn_sign_info* si = (const tn_sign_info*)infos.data_ptr();
        const float* g = (const float*)grads.data_ptr();
        const int64_t n = grads.size(0), dim = grads.size(1);
        void* stream = current_stream();
        call_library([&] { return tn_sparse_table_push(handle, si, g, n, (int)dim, stream); });
        return none();
    });
}

#define TN_FAST(NAME, FN) {NAME, (PyCFunction)(void (*)(void))FN, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {TN_FAST("sparse_table_pull", py_pull),
                         TN_FAST("bind_pull", py_bind_pull),
                         TN_FAST("sparse_table_push", py_push),
                         TN_FAST("bind_push", py_bind_push),
                         TN_FAST("embedding_lookup_sparse", py_combine),
                         TN_FAST("bind_combine", py_bind_combine),
                         TN_FAST("sparse_table_push_pooled", py_push_pooled),
                         TN_FAST("bind_push_pooled", py_bind_push_pooled),
                         TN_FAST("dense_table_push_pull", py_dense_push_pull),
                         TN_FAST("table_pull", py_table_pull),
                         TN_FAST("table_push", py_table_push),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "tensornet_amd._bind", "Operators of tensornet_amd over its C ABI.", -1,
                          methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bind(void) {
    BoundType.tp_name = "tensornet_amd._bind.Bound";
    BoundType.tp_basicsize = sizeof(Bound);
    BoundType.tp_flags = Py_TPFLAGS_DEFAULT;
    BoundType.tp_dealloc = bound_dealloc;
    BoundType.tp_call = bound_call;
    BoundType.tp_getset = bound_getset;
    if (PyType_Ready(&BoundType) < 0) return nullptr;
    PyObject* lib = PyImport_ImportModule("tensornet_amd._lib");
    if (!lib) return nullptr;
    g_error_class = PyObject_GetAttrString(lib, "TensorNetError");
    Py_DECREF(lib);
    if (!g_error_class) return nullptr;
    return PyModule_Create(&module_def);
}
