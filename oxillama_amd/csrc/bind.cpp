// The device entry points' way from Python into liboxq_hip.so: arguments are taken from the call's vector, tensors give
// their data_ptr(), the stream is torch's current one, and the C ABI function is called without the interpreter lock.
// ctypes does the same in 1 us (a handful of arguments) to 3.5 us (pointer tables) a call, as long as the launch behind
// it; a one-token layer of a small model spent 11 of its 24 us there.
//
// Every function returns the C ABI's status; the callers in linear.py, moe.py and quant.py keep the public signatures
// and turn a status into an exception.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstdint>

#include "../../include/oxq.h"

namespace {

PyObject *s_data_ptr, *s_numel, *s_element_size;       // method names
PyObject *get_stream = nullptr, *get_device = nullptr;  // torch._C's functions

// The C ABI, by address from the library that capi.py loaded (it may not be the one beside this file).
#define OXQ_FUNCTIONS(X)                                                                                              \
    X(oxq_rmsnorm_quantize_q8_0_dev) X(oxq_linear_forward_dev) X(oxq_linear_forward_multi_dev) X(oxq_linear_forward_batch_dev) \
    X(oxq_swiglu_quantize_q8_0_dev) X(oxq_quantize_q8_0_dev) X(oxq_ffn_swiglu_dev) X(oxq_topk_dev) X(oxq_lm_head_topk_dev) \
    X(oxq_logits_edit_dev) X(oxq_sample_candidates_dev) X(oxq_moe_forward_dev) X(oxq_gemm_q8_dev) X(oxq_matvec_q8_fused_dev)
#define OXQ_DECLARE(f) decltype(&::f) p_##f = nullptr;
OXQ_FUNCTIONS(OXQ_DECLARE)
#undef OXQ_DECLARE

// One call's arguments; the first conversion that fails leaves a Python error and `ok` false.
struct Args {
    PyObject *const *v;
    bool ok = true;
    uint64_t number(PyObject *o) {
        if (!ok) return 0;
        uint64_t r;
        if (PyLong_Check(o)) {
            r = PyLong_AsUnsignedLongLongMask(o);
        } else {
            PyObject *i = PyNumber_Index(o);
            if (!i) return ok = false, 0;
            r = PyLong_AsUnsignedLongLongMask(i);
            Py_DECREF(i);
        }
        if (r == (uint64_t)-1 && PyErr_Occurred()) ok = false;
        return r;
    }
    uint64_t method(PyObject *o, PyObject *name) {
        if (!ok) return 0;
        PyObject *r = PyObject_VectorcallMethod(name, &o, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr);
        if (!r) return ok = false, 0;
        const uint64_t n = number(r);
        Py_DECREF(r);
        return n;
    }
    // A tensor that the call cannot do without: what has no data_ptr() -- None and integers among it -- is an
    // AttributeError here, as the C ABI launches with the addresses that it gets.
    template <class T> T *tensor_of(PyObject *o) { return (T *)(uintptr_t)method(o, s_data_ptr); }
    template <class T> T *tensor(int i) { return tensor_of<T>(v[i]); }
    // One that it can do without: None is a null pointer.
    template <class T> T *maybe_of(PyObject *o) { return o == Py_None ? nullptr : tensor_of<T>(o); }
    template <class T> T *maybe(int i) { return maybe_of<T>(v[i]); }
    // The address of a host structure, or None.
    template <class T> T *address(int i) { return v[i] == Py_None ? nullptr : (T *)(uintptr_t)number(v[i]); }
    size_t size(int i) { return (size_t)number(v[i]); }
    uint32_t u32(int i) { return (uint32_t)number(v[i]); }
    float real(PyObject *o) {
        if (!ok) return 0.0f;
        const double d = PyFloat_AsDouble(o);
        if (d == -1.0 && PyErr_Occurred()) ok = false;
        return (float)d;
    }
    float f32(int i) { return real(v[i]); }
    // Tensor types and eps are taken as int() and float() take them (a type as a number of any kind or as text).
    uint32_t type(int i) {
        if (!ok || PyLong_Check(v[i])) return u32(i);
        PyObject *o = PyNumber_Long(v[i]);
        if (!o) return ok = false, 0;
        const uint64_t r = number(o);
        Py_DECREF(o);
        return (uint32_t)r;
    }
    float eps(int i) {
        if (!ok || PyFloat_Check(v[i])) return f32(i);
        PyObject *o = PyNumber_Float(v[i]);
        if (!o) return ok = false, 0.0f;
        const float r = real(o);
        Py_DECREF(o);
        return r;
    }
    size_t numel(int i) { return v[i] == Py_None ? 0 : (size_t)method(v[i], s_numel); }
    size_t bytes(int i) { return v[i] == Py_None ? 0 : numel(i) * (size_t)method(v[i], s_element_size); }
    void *stream() {
        if (!ok) return nullptr;
        if (!get_stream) {
            PyObject *cuda = PyImport_ImportModule("torch.cuda"), *c = cuda ? PyImport_ImportModule("torch._C") : nullptr;
            PyObject *r = c ? PyObject_CallMethod(cuda, "init", nullptr) : nullptr;
            if (r) {
                get_device = PyObject_GetAttrString(c, "_cuda_getDevice");
                get_stream = get_device ? PyObject_GetAttrString(c, "_cuda_getCurrentRawStream") : nullptr;
            }
            Py_XDECREF(r), Py_XDECREF(c), Py_XDECREF(cuda);
            if (!get_stream) return ok = false, nullptr;
        }
        PyObject *d = PyObject_CallNoArgs(get_device);
        if (!d) return ok = false, nullptr;
        PyObject *s = PyObject_CallOneArg(get_stream, d);
        Py_DECREF(d);
        if (!s) return ok = false, nullptr;
        const uint64_t p = number(s);
        Py_DECREF(s);
        return (void *)(uintptr_t)p;
    }
};

// NAME(N arguments): CALL is the C ABI call, the rest takes the arguments.
#define OXQ_ENTRY(NAME, N, CALL, ...)                                                         \
    PyObject *NAME(PyObject *, PyObject *const *v, Py_ssize_t n) {                            \
        if (n != N) return PyErr_Format(PyExc_TypeError, #NAME " takes %d arguments", N);     \
        Args a{v};                                                                            \
        __VA_ARGS__ void *const stream = a.stream();                                          \
        if (!a.ok) return nullptr;                                                            \
        int st;                                                                               \
        Py_BEGIN_ALLOW_THREADS st = CALL;                                                     \
        Py_END_ALLOW_THREADS return PyLong_FromLong(st);                                      \
    }

OXQ_ENTRY(rmsnorm_quantize, 7,
          p_oxq_rmsnorm_quantize_q8_0_dev(x, w, eps, rows, cols, y, q8, stream),
          auto x = a.tensor<float>(0); auto w = a.tensor<float>(1); float eps = a.eps(2); size_t rows = a.size(3), cols = a.size(4);
          auto y = a.maybe<float>(5); auto q8 = a.maybe<uint8_t>(6);)

OXQ_ENTRY(linear_forward, 9,
          p_oxq_linear_forward_dev(t, w, x, acts, bias, lora, out, of, in, stream),
          uint32_t t = a.type(0); auto w = a.tensor<uint8_t>(1); auto x = a.maybe<float>(2); auto acts = a.maybe<uint8_t>(3);
          auto bias = a.maybe<float>(4); auto lora = a.address<oxq_lora>(5); auto out = a.tensor<float>(6);
          size_t of = a.size(7), in = a.size(8);)

OXQ_ENTRY(linear_forward_batch, 9,
          p_oxq_linear_forward_batch_dev(t, w, acts, bias, out, batch, of, in, ws, ws_n, stream),
          uint32_t t = a.type(0); auto w = a.tensor<uint8_t>(1); auto acts = a.tensor<uint8_t>(2); auto bias = a.maybe<float>(3);
          auto out = a.tensor<float>(4); size_t batch = a.size(5), of = a.size(6), in = a.size(7);
          auto ws = a.maybe<void>(8); size_t ws_n = a.numel(8);)

OXQ_ENTRY(gemm_q8, 9,
          p_oxq_gemm_q8_dev(t, w, acts, out, m, rows, k, acc, ws, ws_n, stream),
          uint32_t t = a.u32(0); auto w = a.tensor<uint8_t>(1); auto acts = a.tensor<uint8_t>(2); auto out = a.tensor<float>(3);
          size_t m = a.size(4), rows = a.size(5), k = a.size(6); int acc = (int)a.size(7); auto ws = a.maybe<void>(8);
          size_t ws_n = a.numel(8);)

OXQ_ENTRY(matvec_q8_fused, 7,
          p_oxq_matvec_q8_fused_dev(t, w, acts, out, rows, cols, acc, stream),
          uint32_t t = a.u32(0); auto w = a.tensor<uint8_t>(1); auto acts = a.tensor<uint8_t>(2); auto out = a.tensor<float>(3);
          size_t rows = a.size(4), cols = a.size(5); int acc = (int)a.size(6);)

OXQ_ENTRY(swiglu_quantize, 4,
          p_oxq_swiglu_quantize_q8_0_dev(g, u, total, h, q8, stream),
          auto g = a.tensor<float>(0); auto u = a.tensor<float>(1); size_t total = a.numel(0); auto h = a.maybe<float>(2);
          auto q8 = a.maybe<uint8_t>(3);)

OXQ_ENTRY(quantize_q8_0, 2,
          p_oxq_quantize_q8_0_dev(x, total, out, stream),
          auto x = a.tensor<float>(0); size_t total = a.numel(0); auto out = a.tensor<uint8_t>(1);)

OXQ_ENTRY(ffn_swiglu, 11,
          p_oxq_ffn_swiglu_dev(tg, g, tu, u, td, d, acts, out, hidden, inter, ws, ws_n, stream),
          uint32_t tg = a.type(0); auto g = a.tensor<uint8_t>(1); uint32_t tu = a.type(2); auto u = a.tensor<uint8_t>(3);
          uint32_t td = a.type(4); auto d = a.tensor<uint8_t>(5); auto acts = a.tensor<uint8_t>(6); auto out = a.tensor<float>(7);
          size_t hidden = a.size(8), inter = a.size(9); auto ws = a.tensor<void>(10); size_t ws_n = a.numel(10);)

OXQ_ENTRY(topk, 5,
          p_oxq_topk_dev(x, total, k, ov, oi, ws, ws_n, stream),
          auto x = a.tensor<float>(0); size_t total = a.numel(0), k = a.size(1); auto ov = a.tensor<float>(2);
          auto oi = a.tensor<uint32_t>(3); auto ws = a.tensor<void>(4); size_t ws_n = a.bytes(4);)

OXQ_ENTRY(lm_head_topk, 10,
          p_oxq_lm_head_topk_dev(t, w, acts, logits, rows, cols, k, ov, oi, ws, ws_n, stream),
          uint32_t t = a.u32(0); auto w = a.tensor<uint8_t>(1); auto acts = a.tensor<uint8_t>(2); auto logits = a.tensor<float>(3);
          size_t rows = a.size(4), cols = a.size(5), k = a.size(6); auto ov = a.tensor<float>(7); auto oi = a.tensor<uint32_t>(8);
          auto ws = a.tensor<void>(9); size_t ws_n = a.bytes(9);)

OXQ_ENTRY(logits_edit, 7,
          p_oxq_logits_edit_dev(x, total, ban, n_ban, bt, bv, n_bias, rec, n_rec, window, pen, stream),
          auto x = a.tensor<float>(0); size_t total = a.numel(0), n_ban = a.numel(1), n_bias = a.numel(2), n_rec = a.numel(4);
          auto ban = n_ban ? a.maybe<uint32_t>(1) : nullptr; auto bt = n_bias ? a.maybe<uint32_t>(2) : nullptr;
          auto bv = v[3] != Py_None && a.numel(3) ? a.maybe<float>(3) : nullptr; auto rec = n_rec ? a.maybe<uint32_t>(4) : nullptr;
          size_t window = a.size(5); float pen = a.f32(6);)

OXQ_ENTRY(sample_candidates, 9,
          p_oxq_sample_candidates_dev(x, idx, k, temp, min_p, top_p, rng, tok, probs, stream),
          auto x = a.tensor<float>(0); auto idx = a.tensor<uint32_t>(1); size_t k = a.size(2);
          float temp = a.f32(3), min_p = a.f32(4), top_p = a.f32(5); auto rng = a.tensor<uint64_t>(6);
          auto tok = a.tensor<uint32_t>(7); auto probs = a.maybe<float>(8);)

OXQ_ENTRY(moe_forward, 18,
          p_oxq_moe_forward_dev(tg, g, sg, tu, u, su, td, d, sd, n_exp, router, x, tokens, top_k, out, hidden, inter, ws, ws_n,
                                stream),
          uint32_t tg = a.type(0); auto g = a.tensor<uint8_t>(1); size_t sg = a.size(2); uint32_t tu = a.type(3);
          auto u = a.tensor<uint8_t>(4); size_t su = a.size(5); uint32_t td = a.type(6); auto d = a.tensor<uint8_t>(7);
          size_t sd = a.size(8), n_exp = a.size(9); auto router = a.tensor<float>(10); auto x = a.tensor<float>(11);
          size_t tokens = a.size(12), top_k = a.size(13); auto out = a.tensor<float>(14); size_t hidden = a.size(15);
          size_t inter = a.size(16); auto ws = a.tensor<void>(17); size_t ws_n = a.numel(17);)

// (type, weights, acts, biases or None, outs, rows of each, columns).  An output for every weight; a matrix past the end
// of the biases has none, one past the end of the row counts has no rows, which the C ABI refuses, as it does more than
// four matrices (the first MAX_MATS are looked at).
constexpr Py_ssize_t MAX_MATS = 64;
PyObject *linear_forward_multi(PyObject *, PyObject *const *v, Py_ssize_t n) {
    if (n != 7) return PyErr_Format(PyExc_TypeError, "linear_forward_multi takes 7 arguments");
    PyObject *seq[4] = {nullptr, nullptr, nullptr, nullptr};
    const int at[4] = {1, 3, 4, 5};
    const uint8_t *w[MAX_MATS];
    const float *bias[MAX_MATS];
    float *out[MAX_MATS];
    size_t rows[MAX_MATS];
    Args a{v};
    Py_ssize_t mats = 0;
    for (int i = 0; i < 4 && a.ok; i++) {
        if (i == 1 && v[3] == Py_None) continue;
        if (!(seq[i] = PySequence_Fast(v[at[i]], "a sequence with an entry per matrix"))) a.ok = false;
        else if (i == 0) mats = PySequence_Fast_GET_SIZE(seq[0]);
        const Py_ssize_t have = a.ok ? PySequence_Fast_GET_SIZE(seq[i]) : 0;
        if (a.ok && (have > mats || (i == 2 && have < mats))) {
            PyErr_SetString(PyExc_ValueError, "linear_forward_multi: one weight, output, row count (and bias) per matrix");
            a.ok = false;
        }
    }
    auto item = [&](int i, Py_ssize_t j) { return j < PySequence_Fast_GET_SIZE(seq[i]) ? PySequence_Fast_GET_ITEM(seq[i], j) : nullptr; };
    for (Py_ssize_t j = 0; j < mats && j < MAX_MATS && a.ok; j++) {
        w[j] = a.tensor_of<uint8_t>(item(0, j));
        PyObject *const b = seq[1] ? item(1, j) : nullptr, *const r = item(3, j);
        bias[j] = b ? a.maybe_of<float>(b) : nullptr;
        out[j] = a.tensor_of<float>(item(2, j));
        rows[j] = r ? (size_t)a.number(r) : 0;
    }
    const uint32_t t = a.type(0);
    auto acts = a.tensor<uint8_t>(2);
    const size_t cols = a.size(6);
    void *const stream = a.stream();
    int st = 0;
    if (a.ok) {
        Py_BEGIN_ALLOW_THREADS st = p_oxq_linear_forward_multi_dev(t, (size_t)mats, w, acts, seq[1] ? bias : nullptr, out, rows, cols, stream);
        Py_END_ALLOW_THREADS
    }
    for (PyObject *s : seq) Py_XDECREF(s);
    return a.ok ? PyLong_FromLong(st) : nullptr;
}

// attach({name: address}): the functions of the library that capi.py loaded
PyObject *attach(PyObject *, PyObject *addresses) {
    Args a{nullptr};
#define OXQ_TAKE(f)                                                                       \
    {                                                                                     \
        PyObject *o = PyDict_GetItemString(addresses, #f);                                \
        if (!o) return PyErr_Format(PyExc_KeyError, #f);                                  \
        p_##f = (decltype(p_##f))(uintptr_t)a.number(o);                                  \
        if (!a.ok) return nullptr;                                                        \
    }
    OXQ_FUNCTIONS(OXQ_TAKE)
#undef OXQ_TAKE
    Py_RETURN_NONE;
}

#define OXQ_M(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {OXQ_M(rmsnorm_quantize), OXQ_M(linear_forward), OXQ_M(linear_forward_multi), OXQ_M(linear_forward_batch),
                         OXQ_M(gemm_q8), OXQ_M(matvec_q8_fused), OXQ_M(swiglu_quantize), OXQ_M(quantize_q8_0), OXQ_M(ffn_swiglu),
                         OXQ_M(topk), OXQ_M(lm_head_topk), OXQ_M(logits_edit), OXQ_M(sample_candidates), OXQ_M(moe_forward),
                         {"attach", attach, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
#undef OXQ_M
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bind", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bind(void) {
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_numel = PyUnicode_InternFromString("numel");
    s_element_size = PyUnicode_InternFromString("element_size");
    return PyModule_Create(&module);
}
