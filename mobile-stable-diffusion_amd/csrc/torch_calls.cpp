// The calls of the Python package for plain tensors, in native code: checks, outputs, the current stream and the C ABI
// call without Python in between.  A LayerNorm of 154 rows is 2.2 us of GPU and 2.5 to 3.5 (by host) of the runtime's
// launch; the checks, the output and the call cost 3.6 more from Python and 1.1 from here.
//
// Every function takes the arguments of its namesake in the package, all of them, by position, and returns the result,
// or None where the call is not a plain one: an argument that is no dense contiguous device tensor of torch's own
// types, that does not fit the others, a call under a tensor or function mode or a transform.  The package then takes the
// call through its general path, which makes the same call or says what is wrong with it.
//
// Tensors are read through inline accessors, so the extension is good for the one Python and torch it was compiled for:
// `built_for` names them, and the package asks before it makes any other call here.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <vector>

#include "../../include/msd_hip.h"

namespace {

// The C ABI of the library the package has loaded (bind below).
#define MSD_CALLS(X)                                                                                                       \
    X(msd_groupnorm) X(msd_groupnorm_noalloc) X(msd_chunk_add_groupnorm) X(msd_groupnorm_tokens) X(msd_permute_0_2_1)      \
    X(msd_layernorm) X(msd_add_layernorm) X(msd_elemwise_add) X(msd_chunkwise_add) X(msd_geglu) X(msd_silu) X(msd_gelu)    \
    X(msd_quick_gelu) X(msd_timestep_embedding) X(msd_linear_rows) X(msd_linear_rows_grouped) X(msd_softmax)               \
    X(msd_ddim_update)
struct Abi {
#define X(name) decltype(&::name) name = nullptr;
    MSD_CALLS(X)
#undef X
} abi;
PyObject *raise_code = nullptr;  // the package's check(code)

// Gathers what a call is made of; `ok` turns false at the first thing that is not plain.
struct Call {
    bool ok = true;

    Call(Py_ssize_t given, Py_ssize_t wanted) {
        ok = given == wanted && abi.msd_layernorm != nullptr && !at::impl::torch_function_mode_enabled() &&
             !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
             !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
             !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) &&
             !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
    }
    // A dense contiguous tensor on a device, of torch's own class (or a Parameter).
    const at::Tensor *tensor(PyObject *o) {
        if (!ok) return nullptr;
        if (!THPVariable_CheckExact(o)) return fail();
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.defined()) return fail();
        const c10::DispatchKeySet keys = t.key_set();
        constexpr c10::DispatchKeySet kWrapped(
            {c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
             c10::DispatchKey::Python, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
        if (!t.is_cuda() || t.layout() != at::kStrided || keys.has_any(kWrapped) || !t.has_storage() || !t.is_contiguous())
            return fail();
        return &t;
    }
    // ... of float32 or float16; `code` receives which.
    const at::Tensor *data(PyObject *o, int *code) {
        const at::Tensor *t = tensor(o);
        if (t == nullptr) return nullptr;
        if (t->scalar_type() == at::kFloat) *code = MSD_DTYPE_F32;
        else if (t->scalar_type() == at::kHalf) *code = MSD_DTYPE_F16;
        else return fail();
        return t;
    }
    // dtype and device of `like`, `numel` elements
    const at::Tensor *same(PyObject *o, const at::Tensor &like, int64_t numel) {
        const at::Tensor *t = tensor(o);
        if (t == nullptr) return nullptr;
        if (t->scalar_type() != like.scalar_type() || t->get_device() != like.get_device() || t->numel() != numel) return fail();
        return t;
    }
    const float *affine(PyObject *o, int64_t n, const at::Tensor &like) {
        const at::Tensor *t = tensor(o);
        if (t == nullptr) return nullptr;
        if (t->scalar_type() != at::kFloat || t->numel() != n || t->get_device() != like.get_device()) {
            ok = false;
            return nullptr;
        }
        return static_cast<const float *>(t->data_ptr());
    }
    double number(PyObject *o) {
        if (!ok) return 0;
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return v;
    }
    int64_t integer(PyObject *o) {
        if (!ok) return 0;
        if (!PyLong_Check(o)) {  // (a bool is one)
            ok = false;
            return 0;
        }
        const long long v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return v;
    }
    // a C int; what does not fit one is the general path's to convert or refuse
    int code(PyObject *o) {
        const int64_t v = integer(o);
        if (v != (int)v) ok = false;
        return (int)v;
    }
    int truth(PyObject *o) {
        if (ok && !PyBool_Check(o)) ok = false;
        return o == Py_True;
    }
    const at::Tensor *fail() {
        ok = false;
        return nullptr;
    }
};

// A new tensor on the device of `like`, past the dispatcher, which has nothing to say about plain calls (Call): 0.4 us
// less than at::empty.
at::Tensor new_tensor(at::IntArrayRef shape, at::ScalarType type, const at::Tensor &like) {
    return at::Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt));
}

// Whether a contiguous tensor has the strides that a new one of its shape gets.  Those of axes of length one can be any
// (channels last with one position per channel), and torch.empty_like keeps them.
bool plain_strides(const at::Tensor &t) {
    const at::IntArrayRef sizes = t.sizes(), strides = t.strides();
    int64_t stride = 1;
    for (size_t i = sizes.size(); i-- > 0; stride *= std::max<int64_t>(sizes[i], 1))
        if (strides[i] != stride) return false;
    return true;
}

// An output: the caller's tensor, or a new one.
struct Out {
    PyObject *object = nullptr;  // the caller's
    at::Tensor fresh;
    void *data = nullptr;

    void take(Call &c, PyObject *o, const at::Tensor &like) {  // like `like`, or what the caller gave
        if (!c.ok) return;
        if (o == Py_None) {
            if (!plain_strides(like)) {
                c.ok = false;
                return;
            }
            make(new_tensor(like.sizes(), like.scalar_type(), like));
        } else if (const at::Tensor *t = c.same(o, like, like.numel())) {
            object = o;
            data = t->data_ptr();
        }
    }
    void make(at::Tensor t) {
        fresh = std::move(t);
        data = fresh.data_ptr();
    }
    PyObject *result() {
        if (object == nullptr) return THPVariable_Wrap(std::move(fresh));
        Py_INCREF(object);
        return object;
    }
};

// The current stream of the current device; the GIL is given up around the call, as ctypes does.
template <typename F>
int on_stream(F f) {
    void *stream = c10::hip::getCurrentHIPStream(c10::hip::current_device()).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(stream);
    Py_END_ALLOW_THREADS
    return rc;
}

// What `body` returns, None where it returns nullptr without an error set, and for C++ exceptions.
template <typename F>
PyObject *plainly(F body) {
    try {
        PyObject *r = body();
        if (r != nullptr || PyErr_Occurred()) return r;
    } catch (...) {
        PyErr_Clear();
    }
    Py_RETURN_NONE;
}

// nullptr with the package's exception set for a code other than 0
bool failed(int rc) {
    if (rc == 0) return false;
    PyObject *r = PyObject_CallFunction(raise_code, "i", rc);
    if (r != nullptr) {
        Py_DECREF(r);
        PyErr_SetString(PyExc_RuntimeError, "msd call failed");
    }
    return true;
}

PyObject *finish(int rc, Out &out) { return failed(rc) ? nullptr : out.result(); }

struct Planes {
    int64_t batch = 0, channels = 0, hw = 0;
    Planes(Call &c, const at::Tensor *x) {
        if (!c.ok) return;
        if (x->dim() < 2) {
            c.ok = false;
            return;
        }
        batch = x->size(0);
        channels = x->size(1);
        hw = batch * channels != 0 ? x->numel() / (batch * channels) : 0;
    }
};

typedef PyObject *const *Args;

PyObject *groupnorm(PyObject *, Args a, Py_ssize_t n) {  // x, gamma, beta, groups, eps, fuse_silu, out, noalloc
    return plainly([&]() -> PyObject * {
        Call c(n, 8);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const Planes p(c, x);
        if (!c.ok) return nullptr;
        const float *g = c.affine(a[1], p.channels, *x), *b = c.affine(a[2], p.channels, *x);
        const int64_t groups = c.integer(a[3]);
        const double eps = c.number(a[4]);
        const int silu = c.truth(a[5]), noalloc = c.truth(a[7]);
        Out out;
        out.take(c, a[6], *x);
        if (!c.ok || groups < 0) return nullptr;
        auto *call = noalloc ? abi.msd_groupnorm_noalloc : abi.msd_groupnorm;
        const void *xp = x->data_ptr();
        return finish(on_stream([&](void *s) {
            return call(xp, out.data, g, b, p.batch, p.channels, p.hw, groups, (float)eps, silu, code, s);
        }), out);
    });
}

PyObject *chunk_add_groupnorm(PyObject *, Args a, Py_ssize_t n) {  // x, chunk, gamma, beta, groups, eps, fuse_silu, out
    return plainly([&]() -> PyObject * {
        Call c(n, 8);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const Planes p(c, x);
        if (!c.ok) return nullptr;
        const at::Tensor *chunk = c.same(a[1], *x, p.batch * p.channels);
        const float *g = c.affine(a[2], p.channels, *x), *b = c.affine(a[3], p.channels, *x);
        const int64_t groups = c.integer(a[4]);
        const double eps = c.number(a[5]);
        const int silu = c.truth(a[6]);
        Out out;
        out.take(c, a[7], *x);
        if (!c.ok || groups < 0) return nullptr;
        const void *xp = x->data_ptr(), *cp = chunk->data_ptr();
        return finish(on_stream([&](void *s) {
            return abi.msd_chunk_add_groupnorm(xp, cp, out.data, g, b, p.batch, p.channels, p.hw, groups, (float)eps, silu, code, s);
        }), out);
    });
}

PyObject *groupnorm_tokens(PyObject *, Args a, Py_ssize_t n) {  // x, gamma, beta, groups, eps; never in a capture
    return plainly([&]() -> PyObject * {
        Call c(n, 5);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const Planes p(c, x);
        if (!c.ok) return nullptr;
        const float *g = c.affine(a[1], p.channels, *x), *b = c.affine(a[2], p.channels, *x);
        const int64_t groups = c.integer(a[3]);
        const double eps = c.number(a[4]);
        if (!c.ok || groups < 0) return nullptr;
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        const hipStream_t stream = c10::hip::getCurrentHIPStream(c10::hip::current_device()).stream();
        if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return nullptr;
        Out out;
        out.make(new_tensor({p.batch, p.hw, p.channels}, x->scalar_type(), *x));
        const void *xp = x->data_ptr();
        return finish(on_stream([&](void *s) {
            return abi.msd_groupnorm_tokens(xp, out.data, g, b, p.batch, p.channels, p.hw, groups, (float)eps, code, s);
        }), out);
    });
}

PyObject *permute_0_2_1(PyObject *, Args a, Py_ssize_t n) {  // x
    return plainly([&]() -> PyObject * {
        Call c(n, 1);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok || x->dim() != 3) return nullptr;
        const int64_t i = x->size(0), j = x->size(1), k = x->size(2);
        Out out;
        out.make(new_tensor({i, k, j}, x->scalar_type(), *x));
        const void *xp = x->data_ptr();
        return finish(on_stream([&](void *s) { return abi.msd_permute_0_2_1(xp, out.data, i, j, k, code, s); }), out);
    });
}

// rows and length of the last axis
struct Rows {
    int64_t rows = 0, dim = 0;
    Rows(Call &c, const at::Tensor *x) {
        if (!c.ok) return;
        if (x->dim() < 1) {
            c.ok = false;
            return;
        }
        dim = x->size(-1);
        rows = dim != 0 ? x->numel() / dim : 0;
    }
};

PyObject *layernorm(PyObject *, Args a, Py_ssize_t n) {  // x, gamma, beta, eps, out
    return plainly([&]() -> PyObject * {
        Call c(n, 5);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const Rows r(c, x);
        if (!c.ok) return nullptr;
        const float *g = c.affine(a[1], r.dim, *x), *b = c.affine(a[2], r.dim, *x);
        const double eps = c.number(a[3]);
        Out out;
        out.take(c, a[4], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr();
        return finish(on_stream([&](void *s) { return abi.msd_layernorm(xp, out.data, g, b, r.rows, r.dim, (float)eps, code, s); }), out);
    });
}

PyObject *add_layernorm(PyObject *, Args a, Py_ssize_t n) {  // a, b, gamma, beta, eps, sum_out, out
    return plainly([&]() -> PyObject * {
        Call c(n, 7);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const Rows r(c, x);
        if (!c.ok) return nullptr;
        const at::Tensor *res = c.same(a[1], *x, x->numel());
        const float *g = c.affine(a[2], r.dim, *x), *b = c.affine(a[3], r.dim, *x);
        const double eps = c.number(a[4]);
        Out sum, out;
        sum.take(c, a[5], *x);
        out.take(c, a[6], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr(), *rp = res->data_ptr();
        const int rc = on_stream([&](void *s) {
            return abi.msd_add_layernorm(xp, rp, sum.data, out.data, g, b, r.rows, r.dim, (float)eps, code, s);
        });
        if (failed(rc)) return nullptr;
        PyObject *pair = PyTuple_New(2);
        if (pair == nullptr) return nullptr;
        PyTuple_SET_ITEM(pair, 0, sum.result());
        PyTuple_SET_ITEM(pair, 1, out.result());
        return pair;
    });
}

PyObject *elemwise_add(PyObject *, Args a, Py_ssize_t n) {  // a, b, out
    return plainly([&]() -> PyObject * {
        Call c(n, 3);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok) return nullptr;
        const at::Tensor *b = c.same(a[1], *x, x->numel());
        Out out;
        out.take(c, a[2], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr(), *bp = b->data_ptr();
        const int64_t count = x->numel();
        return finish(on_stream([&](void *s) { return abi.msd_elemwise_add(xp, bp, out.data, count, code, s); }), out);
    });
}

PyObject *chunkwise_add(PyObject *, Args a, Py_ssize_t n) {  // a, chunk, chunk_size, out
    return plainly([&]() -> PyObject * {
        Call c(n, 4);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok) return nullptr;
        const int64_t size = c.integer(a[2]), count = x->numel();
        if (!c.ok || size <= 0 || count % size != 0) return nullptr;
        const at::Tensor *chunk = c.same(a[1], *x, count / size);
        Out out;
        out.take(c, a[3], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr(), *cp = chunk->data_ptr();
        return finish(on_stream([&](void *s) { return abi.msd_chunkwise_add(xp, cp, out.data, count, size, code, s); }), out);
    });
}

PyObject *geglu(PyObject *, Args a, Py_ssize_t n) {  // proj, out
    return plainly([&]() -> PyObject * {
        Call c(n, 2);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok || x->dim() < 1) return nullptr;
        const int64_t inner = x->size(-1) / 2, rows = inner != 0 ? x->numel() / (2 * inner) : 0;
        Out out;
        if (a[1] == Py_None) {
            std::vector<int64_t> shape(x->sizes().begin(), x->sizes().end());
            shape.back() = inner;
            at::Tensor fresh = new_tensor(shape, x->scalar_type(), *x);
            if (fresh.numel() != rows * inner) return nullptr;
            out.make(std::move(fresh));
        } else if (const at::Tensor *t = c.same(a[1], *x, rows * inner)) {
            out.object = a[1];
            out.data = t->data_ptr();
        }
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr();
        return finish(on_stream([&](void *s) { return abi.msd_geglu(xp, out.data, rows, inner, code, s); }), out);
    });
}

template <typename F>
PyObject *activation(F *call, Args a, Py_ssize_t n) {  // x, out
    return plainly([&]() -> PyObject * {
        Call c(n, 2);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok) return nullptr;
        Out out;
        out.take(c, a[1], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr();
        const int64_t count = x->numel();
        return finish(on_stream([&](void *s) { return call(xp, out.data, count, code, s); }), out);
    });
}
PyObject *silu(PyObject *, Args a, Py_ssize_t n) { return activation(abi.msd_silu, a, n); }
PyObject *gelu(PyObject *, Args a, Py_ssize_t n) { return activation(abi.msd_gelu, a, n); }
PyObject *quick_gelu(PyObject *, Args a, Py_ssize_t n) { return activation(abi.msd_quick_gelu, a, n); }

PyObject *timestep_embedding(PyObject *, Args a, Py_ssize_t n) {  // timesteps, dim, max_period, half (a bool)
    return plainly([&]() -> PyObject * {
        Call c(n, 4);
        const at::Tensor *t = c.tensor(c.ok ? a[0] : nullptr);
        if (!c.ok || t->scalar_type() != at::kLong) return nullptr;
        const int64_t dim = c.integer(a[1]), count = t->numel();
        const double period = c.number(a[2]);
        const int half = c.truth(a[3]);
        if (!c.ok || dim < 0) return nullptr;
        Out out;
        out.make(new_tensor({count, dim}, half ? at::kHalf : at::kFloat, *t));
        const int64_t *tp = static_cast<const int64_t *>(t->data_ptr());
        return finish(on_stream([&](void *s) {
            return abi.msd_timestep_embedding(tp, out.data, count, dim, (float)period, half ? MSD_DTYPE_F16 : MSD_DTYPE_F32, s);
        }), out);
    });
}

PyObject *linear_rows(PyObject *, Args a, Py_ssize_t n) {  // x, weight, bias, act_in, act_out, out
    return plainly([&]() -> PyObject * {
        Call c(n, 6);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const at::Tensor *w = c.tensor(c.ok ? a[1] : nullptr);
        if (!c.ok || x->dim() != 2 || w->dim() != 2) return nullptr;
        const int64_t m = x->size(0), k = x->size(1), cols = w->size(0);
        if (w->size(1) != k || w->scalar_type() != x->scalar_type() || w->get_device() != x->get_device()) return nullptr;
        const float *bias = a[2] == Py_None ? nullptr : c.affine(a[2], cols, *x);
        const int act_in = c.code(a[3]), act_out = c.code(a[4]);
        if (!c.ok) return nullptr;
        Out out;
        if (a[5] == Py_None) {
            out.make(new_tensor({m, cols}, x->scalar_type(), *x));
        } else if (const at::Tensor *t = c.same(a[5], *x, m * cols)) {
            out.object = a[5];
            out.data = t->data_ptr();
        }
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr(), *wp = w->data_ptr();
        return finish(on_stream([&](void *s) {
            return abi.msd_linear_rows(xp, wp, bias, out.data, m, cols, k, act_in, act_out, code, s);
        }), out);
    });
}

PyObject *linear_rows_grouped(PyObject *, Args a, Py_ssize_t n) {  // x, weights, biases, act_in, act_out
    return plainly([&]() -> PyObject * {
        Call c(n, 5);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok || x->dim() != 2 || !PyList_CheckExact(a[1]) || !(a[2] == Py_None || PyList_CheckExact(a[2]))) return nullptr;
        const Py_ssize_t count = PyList_GET_SIZE(a[1]);
        if (a[2] != Py_None && PyList_GET_SIZE(a[2]) < count) return nullptr;
        const int64_t m = x->size(0), k = x->size(1);
        const int act_in = c.code(a[3]), act_out = c.code(a[4]);
        std::vector<const void *> ws(count);
        std::vector<const float *> bs(count);
        std::vector<size_t> ns(count);
        for (Py_ssize_t i = 0; i < count; i++) {
            const at::Tensor *w = c.tensor(PyList_GET_ITEM(a[1], i));
            if (!c.ok || w->dim() != 2 || w->size(1) != k || w->scalar_type() != x->scalar_type() ||
                w->get_device() != x->get_device())
                return nullptr;
            ws[i] = w->data_ptr();
            ns[i] = (size_t)w->size(0);
            PyObject *b = a[2] == Py_None ? Py_None : PyList_GET_ITEM(a[2], i);
            bs[i] = b == Py_None ? nullptr : c.affine(b, w->size(0), *x);
        }
        if (!c.ok) return nullptr;
        std::vector<Out> outs(count);
        std::vector<void *> ys(count);
        for (Py_ssize_t i = 0; i < count; i++) {
            outs[i].make(new_tensor({m, (int64_t)ns[i]}, x->scalar_type(), *x));
            ys[i] = outs[i].data;
        }
        const void *xp = x->data_ptr();
        const int rc = on_stream([&](void *s) {
            return abi.msd_linear_rows_grouped(xp, ws.data(), bs.data(), ys.data(), ns.data(), count, m, k, act_in, act_out, code, s);
        });
        if (failed(rc)) return nullptr;
        PyObject *list = PyList_New(count);
        if (list == nullptr) return nullptr;
        for (Py_ssize_t i = 0; i < count; i++) PyList_SET_ITEM(list, i, outs[i].result());
        return list;
    });
}

PyObject *softmax(PyObject *, Args a, Py_ssize_t n) {  // x, stable, out
    return plainly([&]() -> PyObject * {
        Call c(n, 3);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        const Rows r(c, x);
        if (!c.ok) return nullptr;
        const int stable = c.truth(a[1]);
        Out out;
        out.take(c, a[2], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr();
        return finish(on_stream([&](void *s) { return abi.msd_softmax(xp, out.data, r.rows, r.dim, stable, code, s); }), out);
    });
}

PyObject *ddim_update(PyObject *, Args a, Py_ssize_t n) {  // x, e_t, a_t, a_prev, sqrt_one_minus_at, out
    return plainly([&]() -> PyObject * {
        Call c(n, 6);
        int code = 0;
        const at::Tensor *x = c.data(c.ok ? a[0] : nullptr, &code);
        if (!c.ok) return nullptr;
        const at::Tensor *e = c.same(a[1], *x, x->numel());
        const double a_t = c.number(a[2]), a_prev = c.number(a[3]), rest = c.number(a[4]);
        Out out;
        out.take(c, a[5], *x);
        if (!c.ok) return nullptr;
        const void *xp = x->data_ptr(), *ep = e->data_ptr();
        const int64_t count = x->numel();
        return finish(on_stream([&](void *s) {
            return abi.msd_ddim_update(xp, ep, out.data, count, (float)a_t, (float)a_prev, (float)rest, code, s);
        }), out);
    });
}

// bind(addresses by name, check): the library's entry points and what raises their error codes
PyObject *bind(PyObject *, PyObject *args) {
    PyObject *addresses = nullptr, *check = nullptr;
    if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &addresses, &check)) return nullptr;
    Abi bound;
#define X(name)                                                                                      \
    {                                                                                                \
        PyObject *at = PyDict_GetItemString(addresses, #name);                                       \
        void *p = at != nullptr ? PyLong_AsVoidPtr(at) : nullptr;                                    \
        if (p == nullptr) {                                                                          \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);                           \
            return nullptr;                                                                          \
        }                                                                                            \
        bound.name = reinterpret_cast<decltype(bound.name)>(p);                                      \
    }
    MSD_CALLS(X)
#undef X
    Py_INCREF(check);
    Py_XDECREF(raise_code);
    raise_code = check;
    abi = bound;
    Py_RETURN_NONE;
}

PyObject *names(PyObject *, PyObject *) {
    PyObject *list = PyList_New(0);
#define X(name)                                                    \
    if (list != nullptr) {                                         \
        PyObject *s = PyUnicode_FromString(#name);                 \
        if (s == nullptr || PyList_Append(list, s) != 0) Py_CLEAR(list); \
        Py_XDECREF(s);                                             \
    }
    MSD_CALLS(X)
#undef X
    return list;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FAST(groupnorm), FAST(chunk_add_groupnorm), FAST(groupnorm_tokens), FAST(permute_0_2_1), FAST(layernorm),
    FAST(add_layernorm), FAST(elemwise_add), FAST(chunkwise_add), FAST(geglu), FAST(silu), FAST(gelu), FAST(quick_gelu),
    FAST(timestep_embedding), FAST(linear_rows), FAST(linear_rows_grouped), FAST(softmax), FAST(ddim_update),
    {"bind", bind, METH_VARARGS, nullptr}, {"names", names, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "msd_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_msd_torch_calls(void) {
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "built_for", MSD_BUILT_FOR) != 0) Py_CLEAR(m);
    return m;
}
