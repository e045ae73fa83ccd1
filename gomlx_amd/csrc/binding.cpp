// The host path of gomlx_amd.nn in native code: argument checks, output allocation and the call into the C ABI for the
// operators of a decode loop.  In Python these steps took 11 us per call with its launch (attribute look-ups, ctypes conversions, one
// Tensor method call per property), longer than the kernels of a small projection; here 5 us.
//
// Every function returns None when it does not recognise its arguments or the library reports an error; gomlx_amd.nn then
// goes through the same call step by step in Python, which raises the exception that belongs to it.  The library's entry
// points come in as addresses (bind), so that whatever library _lib.py has loaded is the one that runs.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <initializer_list>

#include "../../include/gomlx_hipq.h"

namespace {

struct Entry {
    decltype(&gq_qdense_check) check;
    decltype(&gq_qdense_f32) dense_f32;
    decltype(&gq_qdense_bf16) dense_bf16;
    decltype(&gq_qdense_block_f32) block_f32;
    decltype(&gq_qdense_block_bf16) block_bf16;
    decltype(&gq_qdense_gated_f32) gated_f32;
    decltype(&gq_qdense_gated_bf16) gated_bf16;
    decltype(&gq_qdense_f32_batch) batch_f32;
    decltype(&gq_qdense_norm_f32_batch) norm_batch_f32;
    decltype(&gq_qdense_norm_bf16_batch) norm_batch_bf16;
    decltype(&gq_dequantize) dequantize;
    decltype(&gq_embedding_lookup) lookup;
    decltype(&gq_bytes_per_block) bytes_per_block;
    decltype(&gq_values_per_block) values_per_block;
} g;
constexpr int kEntries = 14;
bool g_bound = false;
PyTypeObject *g_activation = nullptr;  // nn.Activation
PyObject *s_scheme, *s_ggml_type, *s_gain, *s_epsilon, *s_scale_offset;

// activation.Type.ToBackend by the numeric value of nn.Activation
constexpr int kBackendAct[13] = {GQ_ACT_NONE, GQ_ACT_RELU, GQ_ACT_NONE, GQ_ACT_NONE, GQ_ACT_NONE, GQ_ACT_NONE, GQ_ACT_SILU,
                                 GQ_ACT_HARDSWISH, GQ_ACT_SILU, GQ_ACT_TANH, GQ_ACT_GELU, GQ_ACT_GELU, GQ_ACT_NONE};
constexpr long kSchemeGGML = 2;

bool to_long(PyObject *o, long &v) {
    if (!PyLong_Check(o)) return false;  // (IntEnum members are ints)
    v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return v >= INT_MIN && v <= INT_MAX;
}
bool attr_long(PyObject *o, PyObject *name, long &v) {
    PyObject *a = PyObject_GetAttr(o, name);
    if (!a) { PyErr_Clear(); return false; }
    const bool ok = to_long(a, v);
    Py_DECREF(a);
    return ok;
}
bool attr_double(PyObject *o, PyObject *name, double &v) {
    PyObject *a = PyObject_GetAttr(o, name);
    if (!a) { PyErr_Clear(); return false; }
    v = PyFloat_Check(a) || PyLong_Check(a) ? PyFloat_AsDouble(a) : -1.0;
    const bool ok = (PyFloat_Check(a) || PyLong_Check(a)) && !PyErr_Occurred();
    PyErr_Clear();
    Py_DECREF(a);
    return ok;
}
bool ggml_type_of(PyObject *quant, int &type) {
    long scheme, t;
    if (quant == Py_None || !attr_long(quant, s_scheme, scheme) || scheme != kSchemeGGML || !attr_long(quant, s_ggml_type, t)) return false;
    type = (int)t;
    return true;
}
// A member of nn.Activation itself: a bare number or a member of another enumeration says nothing about which function is meant.
bool backend_act(PyObject *act, int &v) {
    long a;
    if (Py_TYPE(act) != g_activation || !to_long(act, a) || a < 0 || a >= 13) return false;
    v = kBackendAct[a];
    return true;
}

// A plain contiguous GPU tensor, borrowed; null otherwise.
const at::Tensor *gpu_tensor(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.is_cuda() && t.is_contiguous() ? &t : nullptr;
}
// An optional vector of n floats: 1 = given, 0 = None, -1 = not that.
int vector_of(PyObject *o, int64_t n, const float *&p) {
    p = nullptr;
    if (o == Py_None) return 0;
    const at::Tensor *t = gpu_tensor(o);
    if (!t || t->scalar_type() != at::kFloat || t->dim() != 1 || t->size(0) != n) return -1;
    p = static_cast<const float *>(t->const_data_ptr());
    return 1;
}

struct Norm {
    gq_rmsnorm d;
    bool given = false;
    PyObject *gain = nullptr;  // owned: keeps the vector alive over the launch
    ~Norm() { Py_XDECREF(gain); }
    bool read(PyObject *o, int64_t K) {
        if (o == Py_None) return true;
        double eps, off;
        gain = PyObject_GetAttr(o, s_gain);
        if (!gain) { PyErr_Clear(); return false; }
        if (vector_of(gain, K, d.dGain) < 0 || !attr_double(o, s_epsilon, eps) || !attr_double(o, s_scale_offset, off)) return false;
        d.eps = (float)eps;
        d.gain_offset = (float)off;
        given = true;
        return true;
    }
    const gq_rmsnorm *ptr() const { return given ? &d : nullptr; }
};

// x [batch..., K] and W [N, bytes] of a GGML type: what nn checks before a dense call.
struct Operands {
    const at::Tensor *x, *w;
    int64_t M, K, N;
    bool bf16;
    bool read(PyObject *xo, PyObject *wo, int type, int act, int64_t bias_len) {
        x = gpu_tensor(xo);
        w = gpu_tensor(wo);
        if (!x || !w || w->scalar_type() != at::kByte || w->dim() != 2 || x->dim() < 1) return false;
        if (x->scalar_type() != at::kFloat && x->scalar_type() != at::kBFloat16) return false;
        bf16 = x->scalar_type() == at::kBFloat16;
        N = w->size(0);
        const int64_t k_in = x->size(-1);
        M = k_in ? x->numel() / k_in : 0;
        return g.check(type, bf16 ? GQ_BF16 : GQ_F32, M, k_in, N, w->size(1), bias_len, act, &K) == GQ_OK;
    }
    at::Tensor output() const {
        if (x->dim() == 2) return at::empty({x->size(0), N}, x->options().dtype(at::kFloat).requires_grad(false));
        std::vector<int64_t> shape(x->sizes().begin(), x->sizes().end());
        shape.back() = N;
        return at::empty(shape, x->options().dtype(at::kFloat).requires_grad(false));
    }
};
void *stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

PyObject *none() { Py_RETURN_NONE; }
template <class F> int without_gil(F f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}
// An exception of torch (out of memory, say) is left to the Python path, which meets it again in its own terms.
template <class F> PyObject *guarded(F f) {
    if (!g_bound) return none();
    try {
        return f();
    } catch (...) {
        return none();
    }
}

// dense(x, weights, quant, bias, activation, norm, residual)
PyObject *dense(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        int type, act;
        Operands o;
        Norm norm;
        if (n != 7 || !ggml_type_of(a[2], type) || !backend_act(a[4], act)) return none();
        const at::Tensor *w = gpu_tensor(a[1]);
        const float *bias, *residual = nullptr;
        if (!w || w->dim() != 2 || vector_of(a[3], w->size(0), bias) < 0) return none();
        if (!o.read(a[0], a[1], type, act, bias ? w->size(0) : -1) || !norm.read(a[5], o.K)) return none();
        at::Tensor y = o.output();
        if (a[6] != Py_None) {
            const at::Tensor *r = gpu_tensor(a[6]);
            if (!r || r->scalar_type() != at::kFloat || r->sizes() != y.sizes()) return none();
            residual = static_cast<const float *>(r->const_data_ptr());
        }
        const void *x = o.x->const_data_ptr(), *wp = o.w->const_data_ptr();
        float *yp = static_cast<float *>(y.mutable_data_ptr());
        void *s = stream_of(*o.x);
        const int rc = without_gil([&] {
            if (norm.given || residual)
                return o.bf16 ? g.block_bf16(type, static_cast<const uint16_t *>(x), o.M, o.K, norm.ptr(), wp, o.N, bias, act, residual, yp, s)
                              : g.block_f32(type, static_cast<const float *>(x), o.M, o.K, norm.ptr(), wp, o.N, bias, act, residual, yp, s);
            return o.bf16 ? g.dense_bf16(type, static_cast<const uint16_t *>(x), o.M, o.K, wp, o.N, bias, act, yp, s)
                          : g.dense_f32(type, static_cast<const float *>(x), o.M, o.K, wp, o.N, bias, act, yp, s);
        });
        return rc == GQ_OK ? THPVariable_Wrap(std::move(y)) : none();
    });
}

// gated(x, w_gate, w_up, quant, activation, bias_gate, bias_up, norm)
PyObject *gated(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        int type, act;
        Operands o;
        Norm norm;
        if (n != 8 || !ggml_type_of(a[3], type) || !backend_act(a[4], act)) return none();
        const at::Tensor *up = gpu_tensor(a[2]);
        if (!o.read(a[0], a[1], type, act, -1) || !up || up->scalar_type() != at::kByte || up->sizes() != o.w->sizes()) return none();
        const float *bg, *bu;
        if (vector_of(a[5], o.N, bg) < 0 || vector_of(a[6], o.N, bu) < 0 || !norm.read(a[7], o.K)) return none();
        at::Tensor y = o.output();
        const void *x = o.x->const_data_ptr(), *wg = o.w->const_data_ptr(), *wu = up->const_data_ptr();
        float *yp = static_cast<float *>(y.mutable_data_ptr());
        void *s = stream_of(*o.x);
        const int rc = without_gil([&] {
            return o.bf16 ? g.gated_bf16(type, static_cast<const uint16_t *>(x), o.M, o.K, norm.ptr(), wg, bg, wu, bu, o.N, act, yp, s)
                          : g.gated_f32(type, static_cast<const float *>(x), o.M, o.K, norm.ptr(), wg, bg, wu, bu, o.N, act, yp, s);
        });
        return rc == GQ_OK ? THPVariable_Wrap(std::move(y)) : none();
    });
}

// batch(problems, norm): up to eight (x, weights, quant, bias, activation | None) tuples
PyObject *batch(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        if (n != 2 || !(PyList_Check(a[0]) || PyTuple_Check(a[0]))) return none();
        const Py_ssize_t count = PySequence_Fast_GET_SIZE(a[0]);
        if (count < 1 || count > 8) return none();
        gq_dense_desc d[8];
        at::Tensor y[8];
        Operands o;
        bool bf16 = false;
        for (Py_ssize_t i = 0; i < count; i++) {
            PyObject *p = PySequence_Fast_GET_ITEM(a[0], i);
            int type, act = GQ_ACT_NONE;
            if (!PyTuple_Check(p) || PyTuple_GET_SIZE(p) != 5 || !ggml_type_of(PyTuple_GET_ITEM(p, 2), type)) return none();
            if (PyTuple_GET_ITEM(p, 4) != Py_None && !backend_act(PyTuple_GET_ITEM(p, 4), act)) return none();
            const float *bias;
            if (!o.read(PyTuple_GET_ITEM(p, 0), PyTuple_GET_ITEM(p, 1), type, act, -1) || vector_of(PyTuple_GET_ITEM(p, 3), o.N, bias) < 0) return none();
            if (i == 0) bf16 = o.bf16;
            if (o.bf16 != bf16 || (bf16 && a[1] == Py_None)) return none();
            y[i] = o.output();
            d[i] = gq_dense_desc{type, act, static_cast<const float *>(o.x->const_data_ptr()), o.M, o.K, o.w->const_data_ptr(), o.N, bias,
                                 static_cast<float *>(y[i].mutable_data_ptr())};
        }
        PyObject *p0 = PySequence_Fast_GET_ITEM(a[0], 0);
        const at::Tensor &x0 = THPVariable_Unpack(PyTuple_GET_ITEM(p0, 0));
        Norm norm;
        if (!norm.read(a[1], d[0].K)) return none();
        void *s = stream_of(x0);
        const int rc = without_gil([&] {
            if (!norm.given) return g.batch_f32((int)count, d, s);
            return bf16 ? g.norm_batch_bf16((int)count, d, &norm.d, s) : g.norm_batch_f32((int)count, d, &norm.d, s);
        });
        if (rc != GQ_OK) return none();
        PyObject *out = PyList_New(count);
        if (!out) return nullptr;
        for (Py_ssize_t i = 0; i < count; i++) PyList_SET_ITEM(out, i, THPVariable_Wrap(std::move(y[i])));
        return out;
    });
}

bool row_values(const at::Tensor &w, int type, int64_t &K) {
    const int bpb = g.bytes_per_block(type);
    if (w.scalar_type() != at::kByte || w.dim() != 2 || bpb <= 0 || w.size(1) % bpb) return false;
    K = w.size(1) / bpb * g.values_per_block(type);
    return true;
}

// dequantize(weights, ggml_type)
PyObject *dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        long type;
        int64_t K;
        const at::Tensor *w = n == 2 ? gpu_tensor(a[0]) : nullptr;
        if (!w || !to_long(a[1], type) || !row_values(*w, (int)type, K)) return none();
        at::Tensor y = at::empty({w->size(0), K}, w->options().dtype(at::kFloat).requires_grad(false));
        float *yp = static_cast<float *>(y.mutable_data_ptr());
        const void *wp = w->const_data_ptr();
        void *s = stream_of(*w);
        const int rc = without_gil([&] { return g.dequantize((int)type, wp, w->size(0), K, yp, s); });
        return rc == GQ_OK ? THPVariable_Wrap(std::move(y)) : none();
    });
}

// gather(table, indices int32 [batch..., 1], quant).  The kernel reports an index out of range in pinned host memory, which
// is read once the stream has drained: no clearing kernel and no copy back (28.4 -> 16.1 us for 512 rows of 4096 values).
PyObject *gather(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        int type;
        int64_t K;
        if (n != 3 || !ggml_type_of(a[2], type)) return none();
        const at::Tensor *t = gpu_tensor(a[0]), *idx = gpu_tensor(a[1]);
        if (!t || !idx || !row_values(*t, type, K) || idx->scalar_type() != at::kInt || idx->dim() < 1 || idx->size(-1) != 1 || idx->numel() < 1)
            return none();
        std::vector<int64_t> shape(idx->sizes().begin(), idx->sizes().end());
        shape.back() = K;
        at::Tensor y = at::empty(shape, t->options().dtype(at::kFloat).requires_grad(false));
        at::Tensor flag = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        int32_t *fp = flag.mutable_data_ptr<int32_t>();
        *fp = 0;
        float *yp = static_cast<float *>(y.mutable_data_ptr());
        const void *tp = t->const_data_ptr();
        const int32_t *ip = idx->const_data_ptr<int32_t>();
        const hipStream_t s = static_cast<hipStream_t>(stream_of(*t));
        const int rc = without_gil([&] {
            const int r = g.lookup(type, tp, t->size(0), K, ip, idx->numel(), yp, fp, s);
            return r == GQ_OK && hipStreamSynchronize(s) != hipSuccess ? (int)GQ_ERR_HIP : r;
        });
        return rc == GQ_OK && *static_cast<volatile int32_t *>(fp) == 0 ? THPVariable_Wrap(std::move(y)) : none();
    });
}

// bind(Activation, address, ...): the enumeration of nn.py, the entry points in the order of Entry
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != kEntries + 1 || !PyType_Check(a[0])) { PyErr_Format(PyExc_TypeError, "bind takes a type and %d addresses", kEntries); return nullptr; }
    void *p[kEntries];
    for (int i = 0; i < kEntries; i++) {
        p[i] = PyLong_AsVoidPtr(a[i + 1]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
            return nullptr;
        }
    }
    static_assert(sizeof(Entry) == sizeof p, "one pointer per entry point");
    std::memcpy(static_cast<void *>(&g), p, sizeof p);
    Py_INCREF(a[0]);
    Py_XDECREF(reinterpret_cast<PyObject *>(g_activation));
    g_activation = reinterpret_cast<PyTypeObject *>(a[0]);
    g_bound = true;
    return none();
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"dense", (PyCFunction)(void (*)(void))dense, METH_FASTCALL, nullptr},
    {"gated", (PyCFunction)(void (*)(void))gated, METH_FASTCALL, nullptr},
    {"batch", (PyCFunction)(void (*)(void))batch, METH_FASTCALL, nullptr},
    {"dequantize", (PyCFunction)(void (*)(void))dequantize, METH_FASTCALL, nullptr},
    {"gather", (PyCFunction)(void (*)(void))gather, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) {
    s_scheme = PyUnicode_InternFromString("scheme");
    s_ggml_type = PyUnicode_InternFromString("ggml_type");
    s_gain = PyUnicode_InternFromString("gain");
    s_epsilon = PyUnicode_InternFromString("epsilon");
    s_scale_offset = PyUnicode_InternFromString("scale_offset");
    return PyModule_Create(&module);
}
