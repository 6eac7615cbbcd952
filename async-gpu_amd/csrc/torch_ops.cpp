// The operators of ops.py in native code: argument checks, output allocation, context lookup and the call through the
// C ABI.  A decode-sized kernel runs 2 - 6 us; the same steps through ctypes took 9 us of host time per call, so a
// program that composes operators waited for the interpreter and not for the GPU.
//
// The library stays independent of torch: this module resolves the entry points at run time in the copy of
// libagpu_hip.so that _lib.py has loaded (bind()), and torch is only the allocator of the outputs, as in ops.py.
#include <Python.h>

#include <dlfcn.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <string>
#include <vector>

#include "../../include/agpu.h"

namespace {

// ---- the library, its errors and its contexts ---------------------------------------------

#define AGPU_OPS(X)                                                                                                          \
    X(agpu_int4_linear) X(agpu_ln_int4_linear) X(agpu_layer_norm) X(agpu_add_layer_norm_dual) X(agpu_gelu)                    \
    X(agpu_add_inplace) X(agpu_bias_add) X(agpu_softmax_rows) X(agpu_embedding) X(agpu_argmax_rows) X(agpu_split_qkv)         \
    X(agpu_concat_heads) X(agpu_attention) X(agpu_kv_append) X(agpu_gemm_f32) X(agpu_last_error_string)
struct Lib {
#define X(f) decltype(&f) f##_ = nullptr;
    AGPU_OPS(X)
#undef X
} lib;

PyObject *g_error = nullptr, *g_context = nullptr, *g_ptr = nullptr;  // AgpuError, ops.context, _lib.ptr

// One entry per (device, stream) that has been used; the Context object is kept alive by ops.py.
struct Ctx {
    int device;
    hipStream_t stream;
    agpu_ctx *handle;
};
std::vector<Ctx> g_ctx;  // under the GIL

struct PyFail {};  // a Python error is set

[[noreturn]] void shape_err(const std::string &expected, const std::string &actual) {
    const std::string m = "shape mismatch: expected " + expected + ", got " + actual;
    PyObject *e = PyObject_CallFunction(g_error, "is", AGPU_ERR_SHAPE_MISMATCH, m.c_str());
    if (e) PyErr_SetObject(g_error, e);
    Py_XDECREF(e);
    throw PyFail();
}

std::string str(int64_t v) { return std::to_string(v); }
std::string str(at::IntArrayRef s) {
    std::string r = "(";
    for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + str(s[i]);
    return r + (s.size() == 1 ? ",)" : ")");
}

agpu_ctx *context(const at::Tensor &t) {
    const int device = t.device().has_index() ? t.device().index() : 0;
    const hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();
    for (size_t i = 0; i < g_ctx.size(); ++i)
        if (g_ctx[i].device == device && g_ctx[i].stream == stream) {
            const Ctx c = g_ctx[i];
            if (i) std::swap(g_ctx[i], g_ctx[0]);
            return c.handle;
        }
    PyObject *c = PyObject_CallFunction(g_context, "i", device);
    PyObject *h = c ? PyObject_GetAttrString(c, "handle") : nullptr;
    PyObject *v = h ? PyObject_GetAttrString(h, "value") : nullptr;
    void *p = v ? PyLong_AsVoidPtr(v) : nullptr;
    Py_XDECREF(v);
    Py_XDECREF(h);
    Py_XDECREF(c);
    if (PyErr_Occurred()) throw PyFail();
    g_ctx.insert(g_ctx.begin(), Ctx{device, stream, static_cast<agpu_ctx *>(p)});
    return static_cast<agpu_ctx *>(p);
}

template <class F, class... A>
void call(F fn, agpu_ctx *c, A... a) {
    PyThreadState *s = PyEval_SaveThread();
    const int32_t rc = fn(c, a...);
    PyEval_RestoreThread(s);
    if (rc == AGPU_OK) return;
    PyObject *e = PyObject_CallFunction(g_error, "is", rc, lib.agpu_last_error_string_(c));
    if (e) PyErr_SetObject(g_error, e);
    Py_XDECREF(e);
    throw PyFail();
}

// ---- arguments and results ----------------------------------------------------------------

const at::Tensor &tensor(PyObject *o) {
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expects a torch tensor, got %s", Py_TYPE(o)->tp_name);
        throw PyFail();
    }
    return THPVariable_Unpack(o);
}

const at::Tensor &f32(PyObject *o) {
    const at::Tensor &t = tensor(o);
    if (t.scalar_type() != at::kFloat || !t.is_cuda() || !t.is_contiguous()) {
        PyErr_SetString(PyExc_AssertionError, "expects contiguous fp32 device tensors");
        throw PyFail();
    }
    return t;
}

// What _lib.ptr takes: a tensor, an address or None, and anything else through _lib.ptr itself.  A tensor that is written to is
// asked for a pointer to write through: one that shares its memory with a lazy clone gets memory of its own first.
void *address(PyObject *o, bool written = false) {
    if (o == Py_None) return nullptr;
    if (THPVariable_Check(o)) {
        const at::Tensor &t = THPVariable_Unpack(o);
        return written ? t.mutable_data_ptr() : const_cast<void *>(t.const_data_ptr());
    }
    if (PyLong_Check(o)) {
        void *p = PyLong_AsVoidPtr(o);
        if (PyErr_Occurred()) throw PyFail();
        return p;
    }
    PyObject *r = PyObject_CallFunctionObjArgs(g_ptr, o, nullptr);
    if (!r) throw PyFail();
    void *p = r == Py_None ? nullptr : PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    if (PyErr_Occurred()) throw PyFail();
    return p;
}
const float *fp(PyObject *o) { return static_cast<const float *>(address(o)); }
const float *data(const at::Tensor &t) { return static_cast<const float *>(t.const_data_ptr()); }
float *written(const at::Tensor &t) { return static_cast<float *>(t.mutable_data_ptr()); }

int64_t integer(PyObject *o) {
    PyObject *n = PyNumber_Index(o);
    if (!n) throw PyFail();
    const long long v = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (v == -1 && PyErr_Occurred()) throw PyFail();
    return v;
}
// An argument of 32 bits of the C ABI; what does not fit is an error and not cut off.
int32_t i32(int64_t v) {
    if (v < INT32_MIN || v > INT32_MAX) {
        PyErr_Format(PyExc_OverflowError, "%lld does not fit the library's 32-bit arguments", (long long)v);
        throw PyFail();
    }
    return (int32_t)v;
}
int32_t i32(PyObject *o) { return i32(integer(o)); }
float real(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PyFail();
    return (float)v;
}
int64_t last(const at::Tensor &t) {
    if (t.dim() == 0) shape_err("at least one dimension", "()");
    return t.size(-1);
}
void rank(const at::Tensor &t, int64_t dims, const char *what) {
    if (t.dim() != dims) shape_err(what, str(t.sizes()));
}

at::Tensor empty(at::IntArrayRef sizes, const at::Tensor &like, at::ScalarType type = at::kFloat) {
    return at::detail::empty_cuda(sizes, type, like.device(), std::nullopt);
}
PyObject *wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject *same(PyObject *o) {
    Py_INCREF(o);
    return o;
}

// ---- the operators: positional arguments in the order of ops.py ----------------------------

// x, packed, scales, bias, residual, group, flags, ln, out
PyObject *int4_linear(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]);
    const int64_t K = last(x);
    int64_t kp, N;
    if (THPVariable_Check(a[1])) {
        const at::Tensor &packed = THPVariable_Unpack(a[1]);
        rank(packed, 2, "packed weights [K/8, N]");
        kp = packed.size(0), N = packed.size(1);
    } else {
        PyObject *s = PyObject_GetAttrString(a[1], "shape");
        long long n0 = 0, n1 = 0;
        const bool ok = s && PyArg_ParseTuple(s, "LL", &n0, &n1);
        Py_XDECREF(s);
        if (!ok) throw PyFail();
        kp = n0, N = n1;
    }
    if (K != kp * 8) shape_err("last dim = " + str(kp * 8), "last dim = " + str(K));
    f32(a[0]);
    const int64_t M = x.numel() ? x.numel() / K : 0;
    agpu_ctx *c = context(x);
    PyObject *out = a[8];
    at::Tensor y;
    if (out == Py_None) {
        if (x.dim() <= 2) {
            y = empty({M, N}, x);
        } else {
            std::vector<int64_t> s = x.sizes().vec();
            s.back() = N;
            y = empty(s, x);
        }
    }
    float *yp = out == Py_None ? written(y) : static_cast<float *>(address(out, true));
    const auto *pk = static_cast<const uint32_t *>(address(a[1]));
    const int32_t m = i32(M), n = i32(N), k = i32(K), group = i32(a[5]);
    const uint32_t flags = (uint32_t)integer(a[6]);
    if (a[7] == Py_None) {
        call(lib.agpu_int4_linear_, c, data(x), pk, fp(a[2]), fp(a[3]), fp(a[4]), yp, m, n, k, group, flags);
    } else {
        PyObject *ln = PySequence_Fast(a[7], "ln is (gamma, beta, eps)");
        if (!ln) throw PyFail();
        struct Drop {
            PyObject *o;
            ~Drop() { Py_DECREF(o); }
        } drop{ln};
        if (PySequence_Fast_GET_SIZE(ln) < 3) {
            PyErr_SetString(PyExc_IndexError, "ln is (gamma, beta, eps)");
            throw PyFail();
        }
        PyObject **l = PySequence_Fast_ITEMS(ln);
        call(lib.agpu_ln_int4_linear_, c, data(x), fp(l[0]), fp(l[1]), real(l[2]), pk, fp(a[2]), fp(a[3]), fp(a[4]), yp, m, n, k, group,
             flags);
    }
    if (out == Py_None) return wrap(std::move(y));
    if (x.dim() <= 2) return same(out);
    std::vector<int64_t> s = x.sizes().vec();
    s.back() = N;
    return wrap(tensor(out).reshape(s));
}

// x, gamma, beta, eps
PyObject *layer_norm(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), &g = tensor(a[1]), &b = tensor(a[2]);
    const int64_t d = last(x);
    if (g.numel() != d || b.numel() != d) shape_err("gamma/beta of " + str(d), str(g.numel()) + "/" + str(b.numel()));
    f32(a[0]);
    at::Tensor y = empty(x.sizes(), x);
    call(lib.agpu_layer_norm_, context(x), data(x), data(g), data(b), written(y), i32(d ? x.numel() / d : 0), i32(d), real(a[3]));
    return wrap(std::move(y));
}

// a, b, gamma, beta, eps, want_sum
PyObject *add_layer_norm_dual(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), &r = tensor(a[1]);
    if (x.sizes() != r.sizes()) shape_err(str(x.sizes()), str(r.sizes()));
    f32(a[0]);
    f32(a[1]);
    const int64_t d = last(x);
    const int sum = PyObject_IsTrue(a[5]);
    if (sum < 0) throw PyFail();
    at::Tensor s, n = empty(x.sizes(), x);
    if (sum) s = empty(x.sizes(), x);
    call(lib.agpu_add_layer_norm_dual_, context(x), data(x), data(r), fp(a[2]), fp(a[3]), sum ? written(s) : nullptr, written(n),
         i32(d ? x.numel() / d : 0), i32(d), real(a[4]));
    if (!sum) return wrap(std::move(n));
    return Py_BuildValue("(NN)", wrap(std::move(s)), wrap(std::move(n)));
}

// x, mode
PyObject *gelu(PyObject *const *a) {
    const at::Tensor &x = f32(a[0]);
    at::Tensor y = empty(x.sizes(), x);
    call(lib.agpu_gelu_, context(x), data(x), written(y), (size_t)x.numel(), i32(a[1]));
    return wrap(std::move(y));
}

// a, b
PyObject *add_inplace(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), &r = tensor(a[1]);
    if (x.numel() != r.numel()) shape_err(str(x.sizes()), str(r.sizes()));
    f32(a[0]);
    f32(a[1]);
    float *xp = written(x);
    call(lib.agpu_add_inplace_, context(x), xp, data(r), (size_t)x.numel());
    return same(a[0]);
}

// data, bias
PyObject *bias_add(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), &b = tensor(a[1]);
    const int64_t n = last(x);
    if (b.numel() != n) shape_err("bias of " + str(n), str(b.numel()));
    f32(a[0]);
    float *xp = written(x);
    call(lib.agpu_bias_add_, context(x), xp, data(b), i32(n ? x.numel() / n : 0), i32(n));
    return same(a[0]);
}

// x
PyObject *softmax_rows(PyObject *const *a) {
    const at::Tensor &x = f32(a[0]);
    const int64_t n = last(x);
    at::Tensor y = empty(x.sizes(), x);
    call(lib.agpu_softmax_rows_, context(x), data(x), written(y), i32(n ? x.numel() / n : 0), i32(n));
    return wrap(std::move(y));
}

// tokens, wte, wpe, pos_offset
PyObject *embedding(PyObject *const *a) {
    const at::Tensor &tokens = tensor(a[0]), &wte = tensor(a[1]);
    rank(wte, 2, "wte [vocab, d]");
    const int64_t seq = tokens.numel(), d = wte.size(1);
    at::Tensor out = empty({seq, d}, wte);
    call(lib.agpu_embedding_, context(wte), static_cast<const uint32_t *>(address(a[0])), data(wte), fp(a[2]), written(out), i32(seq), i32(d),
         i32(a[3]));
    return wrap(std::move(out));
}

// x, last_index
PyObject *argmax_rows(PyObject *const *a) {
    const at::Tensor &x = f32(a[0]);
    const int64_t cols = last(x), rows = cols ? x.numel() / cols : 0;
    at::Tensor idx = empty({rows}, x, at::kInt);
    call(lib.agpu_argmax_rows_, context(x), data(x), static_cast<uint32_t *>(idx.data_ptr()), i32(rows), i32(cols), i32(a[1]));
    return wrap(std::move(idx));
}

// qkv, n_heads, d_head
PyObject *split_qkv(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]);
    const int64_t heads = integer(a[1]), dh = integer(a[2]);
    if (x.dim() != 2 || x.size(1) != 3 * heads * dh) shape_err("[seq, " + str(3 * heads * dh) + "]", str(x.sizes()));
    f32(a[0]);
    const int64_t seq = x.size(0);
    std::array<at::Tensor, 3> t;
    for (at::Tensor &o : t) o = empty({heads, seq, dh}, x);
    call(lib.agpu_split_qkv_, context(x), data(x), written(t[0]), written(t[1]), written(t[2]), i32(seq), i32(heads), i32(dh));
    return Py_BuildValue("(NNN)", wrap(std::move(t[0])), wrap(std::move(t[1])), wrap(std::move(t[2])));
}

// x
PyObject *concat_heads(PyObject *const *a) {
    const at::Tensor &x = f32(a[0]);
    rank(x, 3, "[heads, seq, d_head]");
    const int64_t heads = x.size(0), seq = x.size(1), dh = x.size(2);
    at::Tensor out = empty({seq, heads * dh}, x);
    call(lib.agpu_concat_heads_, context(x), data(x), written(out), i32(seq), i32(heads), i32(dh));
    return wrap(std::move(out));
}

void attend(PyObject *q, PyObject *k, PyObject *v, at::Tensor &o, int64_t heads, int64_t q_len, int64_t kv_len, int64_t q_offset,
            int64_t kv_stride, int64_t dh, int causal) {
    f32(k);
    f32(v);
    const at::Tensor &x = f32(q);
    o = empty(x.sizes(), x);
    call(lib.agpu_attention_, context(x), data(x), data(tensor(k)), data(tensor(v)), written(o), i32(heads), i32(q_len), i32(kv_len),
         i32(q_offset), i32(kv_stride), i32(dh), (int32_t)causal);
}

// q, k, v, kv_len, q_offset, causal
PyObject *attention(PyObject *const *a) {
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]);
    rank(q, 3, "q [heads, q_len, d_head]");
    if (k.dim() < 2) shape_err("k [heads, kv_stride, d_head]", str(k.sizes()));
    const int causal = PyObject_IsTrue(a[5]);
    if (causal < 0) throw PyFail();
    at::Tensor o;
    attend(a[0], a[1], a[2], o, q.size(0), q.size(1), a[3] == Py_None ? k.size(1) : integer(a[3]), integer(a[4]), k.size(1), q.size(2), causal);
    return wrap(std::move(o));
}

// q, k, v, seq_len, n_heads, d_head
PyObject *multi_head_flash_attention(PyObject *const *a) {
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    const int64_t seq = integer(a[3]), heads = integer(a[4]), dh = integer(a[5]);
    if (q.numel() != heads * seq * dh || k.sizes() != q.sizes() || v.sizes() != q.sizes())
        shape_err("q, k, v of " + str(heads * seq) + " x " + str(dh), str(q.sizes()) + ", " + str(k.sizes()) + ", " + str(v.sizes()));
    at::Tensor o;
    attend(a[0], a[1], a[2], o, heads, seq, seq, 0, seq, dh, 1);
    return wrap(std::move(o));
}

// src, cache, write_pos
PyObject *kv_append(PyObject *const *a) {
    const at::Tensor &src = f32(a[0]), &cache = f32(a[1]);
    rank(src, 3, "src [heads, rows, d_head]");
    if (cache.dim() < 2) shape_err("cache [heads, positions, d_head]", str(cache.sizes()));
    float *cp = written(cache);
    call(lib.agpu_kv_append_, context(src), data(src), cp, i32(src.size(0)), i32(src.size(1)), i32(cache.size(1)), i32(a[2]),
         i32(src.size(2)));
    return same(a[1]);
}

// a, b
PyObject *gemm_f32(PyObject *const *a) {
    const at::Tensor &x = tensor(a[0]), &b = tensor(a[1]);
    rank(x, 2, "A [M, K]");
    if (b.dim() != 2 || b.size(0) != x.size(1)) shape_err("B with " + str(x.size(1)) + " rows", str(b.sizes()));
    f32(a[0]);
    f32(a[1]);
    at::Tensor c = empty({x.size(0), b.size(1)}, x);
    call(lib.agpu_gemm_f32_, context(x), data(x), data(b), written(c), i32(x.size(0)), i32(b.size(1)), i32(x.size(1)));
    return wrap(std::move(c));
}

// ---- the module ---------------------------------------------------------------------------

template <PyObject *(*OP)(PyObject *const *), int NARGS>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != NARGS) return PyErr_Format(PyExc_TypeError, "expects %d arguments, got %zd", NARGS, n);
    if (!g_error) return PyErr_Format(PyExc_RuntimeError, "bind() has not been called");
    try {
        return OP(args);
    } catch (const PyFail &) {
        return nullptr;
    } catch (...) {  // torch's own (out of memory, a bad size): the Python error that torch makes of it
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// bind(library path, AgpuError, ops.context, _lib.ptr)
PyObject *bind(PyObject *, PyObject *args) {
    const char *path;
    PyObject *error, *context, *ptr;
    if (!PyArg_ParseTuple(args, "sOOO", &path, &error, &context, &ptr)) return nullptr;
    void *so = dlopen(path, RTLD_NOW | RTLD_LOCAL);  // the copy that is loaded already
    if (!so) return PyErr_Format(PyExc_OSError, "%s", dlerror());
#define X(f)                                                  \
    lib.f##_ = reinterpret_cast<decltype(&f)>(dlsym(so, #f)); \
    if (!lib.f##_) return PyErr_Format(PyExc_OSError, "%s lacks " #f, path);
    AGPU_OPS(X)
#undef X
    Py_INCREF(error);
    Py_INCREF(context);
    Py_INCREF(ptr);
    g_error = error, g_context = context, g_ptr = ptr;
    Py_RETURN_NONE;
}

// forget(address of a context that is about to be destroyed)
PyObject *forget(PyObject *, PyObject *handle) {
    const void *h = PyLong_AsVoidPtr(handle);
    if (PyErr_Occurred()) return nullptr;
    for (size_t i = g_ctx.size(); i-- > 0;)
        if (g_ctx[i].handle == h) g_ctx.erase(g_ctx.begin() + (long)i);
    Py_RETURN_NONE;
}

#define OP(name, n) {#name, (PyCFunction)(void (*)(void))entry<name, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    OP(int4_linear, 9), OP(layer_norm, 4), OP(add_layer_norm_dual, 6), OP(gelu, 2), OP(add_inplace, 2), OP(bias_add, 2), OP(softmax_rows, 1),
    OP(embedding, 4), OP(argmax_rows, 2), OP(split_qkv, 3), OP(concat_heads, 1), OP(attention, 6), OP(multi_head_flash_attention, 6),
    OP(kv_append, 3), OP(gemm_f32, 2),
    {"bind", bind, METH_VARARGS, nullptr}, {"forget", forget, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() { return PyModule_Create(&module); }
