// The calls of mojo_amd/ops.py as one native function each (extension module mojo_amd._call).
//
// What bounds a decode call of a small matrix is the host: the checks, the output and workspace tensors and the ctypes
// conversions of a call written in Python took 9 us around a 2.5 us launch and a 3 us kernel.  Here the same call costs
// the launch and about 1 us: tensors are read through their C++ objects, the output comes from the caching allocator without
// the dispatcher, the workspace is a block of that allocator without a tensor around it, and the stream is looked up once.
//
// Every function takes the plain, valid call and returns None for anything else (a wrong type or shape, a tensor subclass,
// a device that is not current, a status of the library): the Python code behind it then names the error, or serves the call.
#include <Python.h>

#include <ATen/EmptyTensor.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/Allocator.h>
#include <c10/hip/HIPFunctions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/qmm.h"

namespace {

constexpr int kEncodings = 7;
struct Encoding {
    PyObject* member;  // the enum member: compared by address (enum members are singletons)
    int code;
    int64_t elements, bytes;  // of a block; 0 for GPTQ
} g_encodings[kEncodings];
int g_encoding_count = 0;
PyObject *s_quant_method, *s_bits, *s_group_size, *s_desc_act, *s_sym, *s_gptq;

const Encoding* encoding_of(PyObject* o) {
    for (int i = 0; i < g_encoding_count; i++)
        if (g_encodings[i].member == o) return &g_encodings[i];
    return nullptr;
}

bool weight_encoding(const Encoding* e) { return e && e->code != QMM_Q8_0 && e->code != QMM_Q8_K; }

// A contiguous GPU tensor on `device` (-1: any), or null.
const at::Tensor* gpu_tensor(PyObject* o, int device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || !t.is_contiguous() || (device >= 0 && t.device().index() != device)) return nullptr;
    return &t;
}

// 0: float32, 1: bfloat16 (the enum qmm_dtype values), -1: neither
int float_code(at::ScalarType t) { return t == at::kFloat ? QMM_F32 : t == at::kBFloat16 ? QMM_BF16 : -1; }
int float_code(PyObject* dtype) { return THPDtype_Check(dtype) ? float_code(reinterpret_cast<THPDtype*>(dtype)->scalar_type) : -1; }

bool int_attr(PyObject* o, PyObject* name, int32_t& v) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (!a) {
        PyErr_Clear();
        return false;
    }
    const long x = PyLong_Check(a) ? PyLong_AsLong(a) : -1;  // (a bool is an int; other types go to the Python path)
    Py_DECREF(a);
    if (x < 0 || x > INT32_MAX) {
        PyErr_Clear();
        return false;
    }
    v = (int32_t)x;
    return true;
}

bool gptq_config(PyObject* config, qmm_gptq_config& c) {
    if (config == Py_None) return false;
    PyObject* method = PyObject_GetAttr(config, s_quant_method);
    if (!method) {
        PyErr_Clear();
        return false;
    }
    const bool gptq = method == s_gptq || (PyUnicode_Check(method) && PyUnicode_Compare(method, s_gptq) == 0);
    Py_DECREF(method);
    if (!gptq || !int_attr(config, s_bits, c.bits) || !int_attr(config, s_group_size, c.group_size) || !int_attr(config, s_desc_act, c.desc_act) ||
        !int_attr(config, s_sym, c.sym))
        return false;
    c.desc_act = c.desc_act != 0;
    c.sym = c.sym != 0;
    return true;
}

// The weight tensors of one product, checked against the encoding and K.
struct Weights {
    const void* ptrs[4];
    int count = 0;
    int64_t n = 0;
    qmm_gptq_config cfg;
    const qmm_gptq_config* cfg_p = nullptr;
};

bool matrix(const at::Tensor* t, at::ScalarType type, int64_t rows, int64_t cols) {
    return t && t->scalar_type() == type && t->dim() == 2 && t->size(0) == rows && t->size(1) == cols;
}

bool packed_matrix(const Encoding* e, const at::Tensor* t, int64_t k) {
    return t && t->scalar_type() == at::kByte && t->dim() == 2 && t->size(0) > 0 && e->elements > 0 && k > 0 && k % e->elements == 0 &&
           t->size(1) == k / e->elements * e->bytes;
}

bool read_weights(const Encoding* e, PyObject* config, PyObject* rhs, int64_t k, int device, Weights& w) {
    if (!PyTuple_CheckExact(rhs)) return false;
    const Py_ssize_t count = PyTuple_GET_SIZE(rhs);
    if (e->code != QMM_GPTQ) {
        if (count != 1) return false;
        const at::Tensor* t = gpu_tensor(PyTuple_GET_ITEM(rhs, 0), device);
        if (!packed_matrix(e, t, k)) return false;
        w.ptrs[0] = t->data_ptr();
        w.count = 1;
        w.n = t->size(0);
        return true;
    }
    if ((count != 3 && count != 4) || !gptq_config(config, w.cfg)) return false;
    const int64_t g = w.cfg.group_size;
    const at::Tensor* q = gpu_tensor(PyTuple_GET_ITEM(rhs, 0), device);
    if (!q || q->scalar_type() != at::kInt || q->dim() != 2 || q->size(0) * 8 != k || g <= 0 || k % g || q->size(1) <= 0) return false;
    w.n = q->size(1);
    const at::Tensor *s = gpu_tensor(PyTuple_GET_ITEM(rhs, 1), device), *z = gpu_tensor(PyTuple_GET_ITEM(rhs, 2), device);
    if (!matrix(s, at::kHalf, k / g, w.n) || !matrix(z, at::kInt, k / g, w.n / 8)) return false;
    w.ptrs[0] = q->data_ptr();
    w.ptrs[1] = s->data_ptr();
    w.ptrs[2] = z->data_ptr();
    w.ptrs[3] = nullptr;
    if (count == 4) {
        const at::Tensor* gi = gpu_tensor(PyTuple_GET_ITEM(rhs, 3), device);
        if (!gi || gi->scalar_type() != at::kInt || gi->dim() != 1 || gi->size(0) != k) return false;
        w.ptrs[3] = gi->data_ptr();
    } else if (w.cfg.desc_act) {
        return false;
    }
    w.count = (int)count;
    w.cfg_p = &w.cfg;
    return true;
}

// The activations of a call and where its results go.
struct Call {
    const at::Tensor* lhs;
    int dtype;
    int64_t m, k;
    int device;
    c10::Allocator* allocator;
    hipStream_t stream;

    bool open(const at::Tensor* t) {  // the device of `t` has to be current: the allocator and the launches go there
        device = t->device().index();
        if (device != c10::hip::current_device()) return false;
        allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
        stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
        return true;
    }
    bool open_lhs(PyObject* o) {
        lhs = gpu_tensor(o, -1);
        if (!lhs || lhs->dim() < 1) return false;
        dtype = float_code(lhs->scalar_type());
        k = lhs->size(-1);
        if (dtype < 0 || k <= 0) return false;
        m = lhs->numel() / k;
        return m > 0 && open(lhs);
    }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type) const {
        return at::Tensor(at::detail::empty_generic(sizes, allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt));
    }
    at::Tensor result(int64_t n, at::ScalarType type) const {  // the leading dimensions of the lhs, then N
        c10::SmallVector<int64_t, 6> sizes(lhs->sizes().begin(), lhs->sizes().end());
        sizes.back() = n;
        return empty(sizes, type);
    }
    // (freed when the call returns: the allocator hands it to later work of the same stream only)
    c10::DataPtr workspace(int64_t bytes) const { return bytes > 0 ? allocator->allocate((size_t)bytes) : c10::DataPtr(); }
};

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

PyObject* none() { Py_RETURN_NONE; }

// matmul(encoding, config, lhs, rhs, flags, out_dtype)
PyObject* py_matmul(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 6) return none();
    const Encoding* e = encoding_of(a[0]);
    Call c;
    Weights w;
    if (!weight_encoding(e) || !c.open_lhs(a[2]) || !read_weights(e, a[1], a[3], c.k, c.device, w)) return none();
    const int out_type = float_code(a[5]);
    if (out_type < 0) return none();
    const int flags = (int)PyLong_AsLong(a[4]) | (out_type == QMM_BF16 ? QMM_FLAG_OUT_BF16 : 0);
    at::Tensor out = c.result(w.n, out_type == QMM_BF16 ? at::kBFloat16 : at::kFloat);
    const int64_t need = qmm_preferred_workspace_bytes(QMM_OP_MATMUL, e->code, w.cfg_p, c.dtype, c.m, w.n, c.k, flags);
    c10::DataPtr ws = c.workspace(need);
    int rc;
    {
        NoGil go;
        rc = qmm_matmul(e->code, w.cfg_p, c.lhs->data_ptr(), c.dtype, c.m, c.k, w.ptrs, w.count, w.n, (float*)out.data_ptr(), ws.get(), need, flags,
                        c.stream);
    }
    if (rc != QMM_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// rmsnorm(encoding, config, x, gamma, eps, rhs, out_dtype)
PyObject* py_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 7) return none();
    const Encoding* e = encoding_of(a[0]);
    Call c;
    Weights w;
    if (!weight_encoding(e) || !c.open_lhs(a[2]) || !read_weights(e, a[1], a[5], c.k, c.device, w)) return none();
    const at::Tensor* gamma = gpu_tensor(a[3], c.device);
    const int out_type = float_code(a[6]);
    if (!gamma || gamma->scalar_type() != at::kFloat || gamma->dim() != 1 || gamma->size(0) != c.k || out_type < 0 || !PyFloat_Check(a[4])) return none();
    const double eps = PyFloat_AS_DOUBLE(a[4]);
    if (!(eps >= 0.0)) return none();
    const int flags = out_type == QMM_BF16 ? QMM_FLAG_OUT_BF16 : 0;
    at::Tensor out = c.result(w.n, out_type == QMM_BF16 ? at::kBFloat16 : at::kFloat);
    const int64_t need = qmm_preferred_workspace_bytes(QMM_OP_RMSNORM, e->code, w.cfg_p, c.dtype, c.m, w.n, c.k, flags);
    c10::DataPtr ws = c.workspace(need);
    int rc;
    {
        NoGil go;
        rc = qmm_matmul_rmsnorm(e->code, w.cfg_p, c.lhs->data_ptr(), c.dtype, (const float*)gamma->data_ptr(), (float)eps, c.m, c.k, w.ptrs, w.count, w.n,
                                (float*)out.data_ptr(), ws.get(), need, flags, c.stream);
    }
    if (rc != QMM_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// grouped(encoding, lhs, list of rhs)
PyObject* py_grouped(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    constexpr Py_ssize_t kMost = 16;
    if (count != 3 || !PyList_CheckExact(a[2])) return none();
    const Py_ssize_t mats = PyList_GET_SIZE(a[2]);
    const Encoding* e = encoding_of(a[0]);
    Call c;
    if (mats < 1 || mats > kMost || !weight_encoding(e) || e->code == QMM_GPTQ || !c.open_lhs(a[1])) return none();
    const void* rhs[kMost];
    void* outs[kMost];
    int64_t n[kMost];
    at::Tensor out[kMost];
    for (Py_ssize_t i = 0; i < mats; i++) {
        const at::Tensor* t = gpu_tensor(PyList_GET_ITEM(a[2], i), c.device);
        if (!packed_matrix(e, t, c.k)) return none();
        rhs[i] = t->data_ptr();
        n[i] = t->size(0);
    }
    for (Py_ssize_t i = 0; i < mats; i++) {
        out[i] = c.result(n[i], at::kFloat);
        outs[i] = out[i].data_ptr();
    }
    const int64_t need = qmm_matmul_grouped_workspace_bytes(e->code, c.dtype, c.m, c.k, (int)mats, n);
    c10::DataPtr ws = c.workspace(need);
    int rc;
    {
        NoGil go;
        rc = qmm_matmul_grouped(e->code, c.lhs->data_ptr(), c.dtype, c.m, c.k, (int)mats, rhs, n, (float* const*)outs, ws.get(), need, c.stream);
    }
    if (rc != QMM_OK) return none();
    PyObject* list = PyList_New(mats);
    if (!list) return nullptr;
    for (Py_ssize_t i = 0; i < mats; i++) PyList_SET_ITEM(list, i, THPVariable_Wrap(std::move(out[i])));
    return list;
    END_HANDLE_TH_ERRORS
}

// swiglu(encoding, lhs, gate, up)
PyObject* py_swiglu(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 4) return none();
    const Encoding* e = encoding_of(a[0]);
    Call c;
    if (!weight_encoding(e) || e->code == QMM_GPTQ || !c.open_lhs(a[1])) return none();
    const at::Tensor *gate = gpu_tensor(a[2], c.device), *up = gpu_tensor(a[3], c.device);
    if (!packed_matrix(e, gate, c.k) || !packed_matrix(e, up, c.k) || gate->size(0) != up->size(0)) return none();
    const int64_t n = gate->size(0);
    at::Tensor out = c.result(n, at::kFloat);
    const int64_t need = qmm_preferred_workspace_bytes(QMM_OP_SWIGLU, e->code, nullptr, c.dtype, c.m, n, c.k, 0);
    c10::DataPtr ws = c.workspace(need);
    int rc;
    {
        NoGil go;
        rc = qmm_matmul_swiglu(e->code, c.lhs->data_ptr(), c.dtype, c.m, c.k, gate->data_ptr(), up->data_ptr(), n, (float*)out.data_ptr(), ws.get(), need,
                               c.stream);
    }
    if (rc != QMM_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// repacked(encoding, config, lhs, n, k, packed, rhs)
PyObject* py_repacked(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 7 || !PyTuple_CheckExact(a[6])) return none();
    const Encoding* e = encoding_of(a[0]);
    Call c;
    Weights w;
    if (!weight_encoding(e) || !c.open_lhs(a[2]) || c.k != PyLong_AsLongLong(a[4])) return none();
    const int64_t n = PyLong_AsLongLong(a[3]);
    const at::Tensor* packed = gpu_tensor(a[5], c.device);
    if (!packed || n <= 0) return none();
    if (PyTuple_GET_SIZE(a[6]) > 0) {
        if (!read_weights(e, a[1], a[6], c.k, c.device, w) || w.n != n) return none();
    } else if (e->code == QMM_GPTQ) {
        if (!gptq_config(a[1], w.cfg)) return none();
        w.cfg_p = &w.cfg;
    }
    at::Tensor out = c.result(n, at::kFloat);
    const int64_t need = qmm_preferred_workspace_bytes(QMM_OP_REPACKED, e->code, w.cfg_p, c.dtype, c.m, n, c.k, 0);
    c10::DataPtr ws = c.workspace(need);
    int rc;
    {
        NoGil go;
        rc = qmm_matmul_repacked(e->code, w.cfg_p, c.lhs->data_ptr(), c.dtype, c.m, c.k, w.count ? w.ptrs : nullptr, w.count, packed->data_ptr(),
                                 packed->numel(), n, (float*)out.data_ptr(), ws.get(), need, 0, c.stream);
    }
    if (rc != QMM_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// dequantize(encoding, config, tensors, dtype)
PyObject* py_dequantize(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 4 || !PyTuple_CheckExact(a[2]) || PyTuple_GET_SIZE(a[2]) < 1) return none();
    const Encoding* e = encoding_of(a[0]);
    const int type = float_code(a[3]);
    if (!weight_encoding(e) || type < 0) return none();
    const at::Tensor* t = gpu_tensor(PyTuple_GET_ITEM(a[2], 0), -1);
    Call c;
    if (!t || t->dim() != 2 || !c.open(t)) return none();
    const bool gptq = e->code == QMM_GPTQ;
    const int64_t k = gptq ? t->size(0) * 8 : t->size(1) % e->bytes ? 0 : t->size(1) / e->bytes * e->elements;
    Weights w;
    if (k <= 0 || !read_weights(e, a[1], a[2], k, c.device, w)) return none();
    at::Tensor out = c.empty({w.n, k}, type == QMM_BF16 ? at::kBFloat16 : at::kFloat);
    int rc;
    {
        NoGil go;
        rc = gptq ? qmm_dequantize_gptq(w.cfg_p, w.ptrs[0], w.ptrs[1], w.ptrs[2], w.ptrs[3], w.n, k, out.data_ptr(), type, c.stream)
                  : qmm_dequantize(e->code, w.ptrs[0], w.n, k, out.data_ptr(), type, c.stream);
    }
    if (rc != QMM_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// quantize(encoding, x)
PyObject* py_quantize(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 2) return none();
    const Encoding* e = encoding_of(a[0]);
    const at::Tensor* x = gpu_tensor(a[1], -1);
    Call c;
    if (!e || e->elements <= 0 || !x || x->scalar_type() != at::kFloat || x->dim() != 2 || !c.open(x)) return none();
    const int64_t rows = x->size(0), k = x->size(1);
    if (rows <= 0 || k <= 0 || k % e->elements) return none();
    at::Tensor out = c.empty({rows, k / e->elements * e->bytes}, at::kByte);
    int rc;
    {
        NoGil go;
        rc = qmm_quantize(e->code, (const float*)x->data_ptr(), rows, k, out.data_ptr(), c.stream);
    }
    if (rc != QMM_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// quantize_gptq(config, w)
PyObject* py_quantize_gptq(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 2) return none();
    const at::Tensor* w = gpu_tensor(a[1], -1);
    Call c;
    qmm_gptq_config cfg;
    if (!w || w->scalar_type() != at::kFloat || w->dim() != 2 || !gptq_config(a[0], cfg) || !c.open(w)) return none();
    const int64_t n = w->size(0), k = w->size(1), g = cfg.group_size;
    if (n <= 0 || k <= 0 || g <= 0 || k % g || k % 8 || n % 8) return none();
    at::Tensor out[4] = {c.empty({k / 8, n}, at::kInt), c.empty({k / g, n}, at::kHalf), c.empty({k / g, n / 8}, at::kInt), c.empty({k}, at::kInt)};
    int rc;
    {
        NoGil go;
        rc = qmm_quantize_gptq(&cfg, (const float*)w->data_ptr(), n, k, out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), out[3].data_ptr(), c.stream);
    }
    if (rc != QMM_OK) return none();
    PyObject* tuple = PyTuple_New(4);
    if (!tuple) return nullptr;
    for (int i = 0; i < 4; i++) PyTuple_SET_ITEM(tuple, i, THPVariable_Wrap(std::move(out[i])));
    return tuple;
    END_HANDLE_TH_ERRORS
}

// setup([(member, code, elements, bytes), ...]): the members of QuantizationEncoding
PyObject* py_setup(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 1 || !PyList_Check(a[0]) || PyList_GET_SIZE(a[0]) > kEncodings) {
        PyErr_SetString(PyExc_TypeError, "setup takes one list of at most 7 encodings");
        return nullptr;
    }
    g_encoding_count = 0;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); i++) {
        PyObject* member;
        int code;
        long long elements, bytes;
        if (!PyArg_ParseTuple(PyList_GET_ITEM(a[0], i), "OiLL", &member, &code, &elements, &bytes)) return nullptr;
        Py_INCREF(member);
        g_encodings[g_encoding_count++] = Encoding{member, code, elements, bytes};
    }
    Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name, const char* doc) {
    return PyMethodDef{name, (PyCFunction)(void (*)(void))F, METH_FASTCALL, doc};
}

PyMethodDef g_methods[] = {
    method<py_setup>("setup", "setup(encodings)"),
    method<py_matmul>("matmul", "matmul(encoding, config, lhs, rhs, flags, out_dtype) -> tensor or None"),
    method<py_rmsnorm>("rmsnorm", "rmsnorm(encoding, config, x, gamma, eps, rhs, out_dtype) -> tensor or None"),
    method<py_grouped>("grouped", "grouped(encoding, lhs, rhs) -> list or None"),
    method<py_swiglu>("swiglu", "swiglu(encoding, lhs, gate, up) -> tensor or None"),
    method<py_repacked>("repacked", "repacked(encoding, config, lhs, n, k, packed, rhs) -> tensor or None"),
    method<py_dequantize>("dequantize", "dequantize(encoding, config, tensors, dtype) -> tensor or None"),
    method<py_quantize>("quantize", "quantize(encoding, x) -> tensor or None"),
    method<py_quantize_gptq>("quantize_gptq", "quantize_gptq(config, w) -> 4 tensors or None"),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_call", "The calls of mojo_amd.ops as native functions.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) {
    s_quant_method = PyUnicode_InternFromString("quant_method");
    s_bits = PyUnicode_InternFromString("bits");
    s_group_size = PyUnicode_InternFromString("group_size");
    s_desc_act = PyUnicode_InternFromString("desc_act");
    s_sym = PyUnicode_InternFromString("sym");
    s_gptq = PyUnicode_InternFromString("gptq");
    if (!s_quant_method || !s_bits || !s_group_size || !s_desc_act || !s_sym || !s_gptq) return nullptr;
    PyObject* const module = PyModule_Create(&g_module);
    // the build's torch and Python: the loader looks for these bytes in the file before it loads it
    if (module && PyModule_AddStringConstant(module, "compiled_for", QMM_CALL_STAMP) < 0) {
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
