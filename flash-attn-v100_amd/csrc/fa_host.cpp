// Host side of one forward / backward call as a CPython module: checks the
// layout of the tensors, allocates the outputs and the workspace with torch,
// fills the argument struct of include/fa_abi.h and calls the kernel library.
// The same steps through ctypes took 16 us (forward) and 25 us (backward) of
// Python per call, more than the kernels of a small call run; here 6 and 10 us
// (of which the launches take 3 and 6).
// The library's functions are bound by address (the Python layer has loaded
// and checked it).  Every call is self-contained: nothing is kept between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "fa_abi.h"

namespace {

decltype(&fa_fwd_workspace_size) p_fwd_ws_size;
decltype(&fa_fwd_ws) p_fwd_ws;
decltype(&fa_fwd_cols) p_fwd_cols;
decltype(&fa_bwd_workspace_size) p_bwd_ws_size;
decltype(&fa_bwd) p_bwd;
decltype(&fa_bwd_cols) p_bwd_cols;

int32_t dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return FA_DTYPE_F16;
        case at::kBFloat16: return FA_DTYPE_BF16;
        case at::kFloat: return FA_DTYPE_F32;
        default: return -1;  // the library refuses it
    }
}

// t, or a contiguous copy where the kernels' 16-byte loads need one: d stride
// 1, other strides non-negative multiples of 16 bytes, base 16-byte aligned
at::Tensor prepare(const at::Tensor& t) {
    const int64_t es = t.element_size(), n = t.dim();
    bool ok = n > 0 && t.stride(n - 1) == 1 && ((uintptr_t)t.data_ptr() & 15) == 0;
    for (int64_t d = 0; ok && d + 1 < n; ++d) ok = t.stride(d) >= 0 && (t.stride(d) * es) % 16 == 0;
    return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

void put_strides(int64_t (&dst)[4], const at::Tensor& t) {
    for (int d = 0; d < 4; ++d) dst[d] = t.stride(d);
}

// a tuple of four element strides
bool get_strides(PyObject* o, int64_t (&dst)[4]) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) {
        PyErr_SetString(PyExc_TypeError, "strides must be a tuple of four integers");
        return false;
    }
    for (int d = 0; d < 4; ++d) {
        dst[d] = PyLong_AsLongLong(PyTuple_GET_ITEM(o, d));
        if (dst[d] == -1 && PyErr_Occurred()) return false;
    }
    return true;
}

bool all_4d(std::initializer_list<const at::Tensor*> ts) {
    for (const at::Tensor* t : ts)
        if (t->dim() != 4) {
            PyErr_SetString(PyExc_ValueError, "tensors must be 4-dimensional [batch, seq_len, num_heads, head_dim]");
            return false;
        }
    return true;
}

bool check_args(Py_ssize_t n, Py_ssize_t want, PyObject* const* a, Py_ssize_t n_tensors) {
    if (n != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
        return false;
    }
    for (Py_ssize_t i = 0; i < n_tensors; ++i)
        if (!THPVariable_Check(a[i])) {
            PyErr_SetString(PyExc_TypeError, "expected a tensor");
            return false;
        }
    return true;
}

void* optional_ptr(PyObject* o) { return THPVariable_Check(o) ? THPVariable_Unpack(o).data_ptr() : nullptr; }

// the fields both structs share, from (causal, scale, dropout_p, seed, offset)
template <typename A>
bool put_common(A& a, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int32_t head_dim, PyObject* const* x) {
    a.q = q.data_ptr();
    a.k = k.data_ptr();
    a.v = v.data_ptr();
    put_strides(a.q_stride, q);
    put_strides(a.k_stride, k);
    put_strides(a.v_stride, v);
    a.batch = (int32_t)q.size(0);
    a.seqlen_q = (int32_t)q.size(1);
    a.seqlen_k = (int32_t)k.size(1);
    a.num_heads = (int32_t)q.size(2);
    a.num_heads_kv = (int32_t)k.size(2);
    a.head_dim = head_dim;
    a.dtype = dtype_code(q.scalar_type());
    a.causal = PyObject_IsTrue(x[0]);
    a.scale = (float)PyFloat_AsDouble(x[1]);
    a.dropout_p = (float)PyFloat_AsDouble(x[2]);
    a.seed = PyLong_AsUnsignedLongLongMask(x[3]);
    a.offset = PyLong_AsUnsignedLongLongMask(x[4]);
    return !PyErr_Occurred();
}

// bias tensor or None, its strides, its dtype code
template <typename A>
bool put_bias(A& a, PyObject* const* x) {
    a.bias = optional_ptr(x[0]);
    a.bias_stride[0] = a.bias_stride[1] = a.bias_stride[2] = 0;
    a.bias_stride[3] = 1;
    a.bias_dtype = a.dtype;
    if (!a.bias) return true;
    a.bias_dtype = (int32_t)PyLong_AsLong(x[2]);
    return get_strides(x[1], a.bias_stride) && !PyErr_Occurred();
}

PyObject* wrap_or_none(const at::Tensor& t) {
    if (t.defined()) return THPVariable_Wrap(t);
    Py_RETURN_NONE;
}

// fwd(q, k, v, causal, scale, dropout_p, seed, offset, bias, bias_strides,
//     bias_dtype, keep_bits, want_max, head_dim, cols, stream)
//   -> (status, o, lse, max or None)
PyObject* host_fwd(PyObject*, PyObject* const* x, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!check_args(n, 16, x, 3)) return nullptr;
    const at::Tensor &q0 = THPVariable_Unpack(x[0]), &k0 = THPVariable_Unpack(x[1]), &v0 = THPVariable_Unpack(x[2]);
    if (!all_4d({&q0, &k0, &v0})) return nullptr;
    const at::Tensor q = prepare(q0), k = prepare(k0), v = prepare(v0);
    const int32_t head_dim = (int32_t)PyLong_AsLong(x[13]), cols = (int32_t)PyLong_AsLong(x[14]);
    void* const stream = PyLong_AsVoidPtr(x[15]);
    const bool want_max = PyObject_IsTrue(x[12]) == 1;
    fa_fwd_args a;
    if (!put_common(a, q, k, v, head_dim, x + 3) || !put_bias(a, x + 8)) return nullptr;
    const at::Tensor o = at::empty(q.sizes(), q.options());
    const auto f32 = q.options().dtype(at::kFloat);
    const int64_t rows[3] = {q.size(0), q.size(2), q.size(1)};
    const at::Tensor lse = at::empty(rows, f32);
    const at::Tensor mx = want_max ? at::empty(rows, f32) : at::Tensor();
    a.o = o.data_ptr();
    put_strides(a.o_stride, o);
    a.lse = (float*)lse.data_ptr();
    a.max_vals = want_max ? (float*)mx.data_ptr() : nullptr;
    a.keep_bits = (uint32_t*)optional_ptr(x[11]);
    const size_t bytes = p_fwd_ws_size(&a);
    at::Tensor ws;
    if (bytes) ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    int32_t st;
    {
        void* const wp = bytes ? ws.data_ptr() : nullptr;
        pybind11::gil_scoped_release no_gil;
        st = cols ? p_fwd_cols(&a, cols, wp, bytes, stream) : p_fwd_ws(&a, wp, bytes, stream);
    }
    return Py_BuildValue("(iNNN)", (int)st, THPVariable_Wrap(o), THPVariable_Wrap(lse), wrap_or_none(mx));
    END_HANDLE_TH_ERRORS
}

// bwd(q, k, v, o, do, lse, causal, scale, dropout_p, seed, offset, bias,
//     bias_strides, bias_dtype, keep_bits, dbias, dbias_strides, dbias_dtype,
//     head_dim, cols, stream) -> (status, dq, dk, dv)
PyObject* host_bwd(PyObject*, PyObject* const* x, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!check_args(n, 21, x, 6)) return nullptr;
    const at::Tensor &q0 = THPVariable_Unpack(x[0]), &k0 = THPVariable_Unpack(x[1]), &v0 = THPVariable_Unpack(x[2]),
                     &o0 = THPVariable_Unpack(x[3]), &do0 = THPVariable_Unpack(x[4]);
    if (!all_4d({&q0, &k0, &v0, &o0, &do0})) return nullptr;
    const at::Tensor q = prepare(q0), k = prepare(k0), v = prepare(v0), o = prepare(o0), dout = prepare(do0);
    const at::Tensor lse = THPVariable_Unpack(x[5]).contiguous();
    const int32_t head_dim = (int32_t)PyLong_AsLong(x[18]), cols = (int32_t)PyLong_AsLong(x[19]);
    void* const stream = PyLong_AsVoidPtr(x[20]);
    fa_bwd_args a;
    if (!put_common(a, q, k, v, head_dim, x + 6) || !put_bias(a, x + 11)) return nullptr;
    const at::Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()),
                     dv = at::empty(v.sizes(), v.options());
    a.o = o.data_ptr();
    a.dout = dout.data_ptr();
    a.lse = (const float*)lse.data_ptr();
    a.dq = dq.data_ptr();
    a.dk = dk.data_ptr();
    a.dv = dv.data_ptr();
    put_strides(a.o_stride, o);
    put_strides(a.do_stride, dout);
    put_strides(a.dq_stride, dq);
    put_strides(a.dk_stride, dk);
    put_strides(a.dv_stride, dv);
    a.keep_bits = (const uint32_t*)optional_ptr(x[14]);
    a.dbias = optional_ptr(x[15]);
    a.dbias_stride[0] = a.dbias_stride[1] = a.dbias_stride[2] = 0;
    a.dbias_stride[3] = 1;
    a.dbias_dtype = FA_DTYPE_F32;
    if (a.dbias) {
        a.dbias_dtype = (int32_t)PyLong_AsLong(x[17]);
        if (!get_strides(x[16], a.dbias_stride) || PyErr_Occurred()) return nullptr;
    }
    const int64_t bytes = std::max<int64_t>((int64_t)p_bwd_ws_size(&a), 256);
    const at::Tensor ws = at::empty({bytes}, q.options().dtype(at::kByte));
    int32_t st;
    {
        void* const wp = ws.data_ptr();
        pybind11::gil_scoped_release no_gil;
        st = cols ? p_bwd_cols(&a, cols, wp, (size_t)bytes, stream) : p_bwd(&a, wp, (size_t)bytes, stream);
    }
    return Py_BuildValue("(iNNN)", (int)st, THPVariable_Wrap(dq), THPVariable_Wrap(dk), THPVariable_Wrap(dv));
    END_HANDLE_TH_ERRORS
}

// bind(fa_abi_version, sizeof(fa_fwd_args), sizeof(fa_bwd_args),
//      fa_fwd_workspace_size, fa_fwd_ws, fa_fwd_cols, fa_bwd_workspace_size,
//      fa_bwd, fa_bwd_cols): addresses in the loaded kernel library, and the
// struct sizes of the layer that binds it.  Refused where the library or that
// layer speaks another version than this module was compiled for: the structs
// carry device pointers.
PyObject* host_bind(PyObject*, PyObject* const* x, Py_ssize_t n) {
    if (n != 9) {
        PyErr_SetString(PyExc_TypeError, "bind takes seven addresses and two sizes");
        return nullptr;
    }
    void* p[7];
    for (int i = 0; i < 7; ++i) {
        p[i] = PyLong_AsVoidPtr(x[i == 0 ? 0 : i + 2]);
        if (PyErr_Occurred()) return nullptr;
        if (!p[i]) {
            PyErr_SetString(PyExc_ValueError, "bind: null address");
            return nullptr;
        }
    }
    const size_t sizes[2] = {PyLong_AsSize_t(x[1]), PyLong_AsSize_t(x[2])};
    if (PyErr_Occurred()) return nullptr;
    const int32_t version = ((decltype(&fa_abi_version))p[0])();
    if (version != FA_ABI_VERSION || sizes[0] != sizeof(fa_fwd_args) || sizes[1] != sizeof(fa_bwd_args)) {
        PyErr_Format(PyExc_RuntimeError,
                     "fa_host was built for ABI version %d with argument structs of %zu and %zu bytes; the library has "
                     "version %d, the binding %zu and %zu bytes",
                     FA_ABI_VERSION, sizeof(fa_fwd_args), sizeof(fa_bwd_args), (int)version, sizes[0], sizes[1]);
        return nullptr;
    }
    p_fwd_ws_size = (decltype(p_fwd_ws_size))p[1];
    p_fwd_ws = (decltype(p_fwd_ws))p[2];
    p_fwd_cols = (decltype(p_fwd_cols))p[3];
    p_bwd_ws_size = (decltype(p_bwd_ws_size))p[4];
    p_bwd = (decltype(p_bwd))p[5];
    p_bwd_cols = (decltype(p_bwd_cols))p[6];
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void*)host_bind, METH_FASTCALL, nullptr},
    {"fwd", (PyCFunction)(void*)host_fwd, METH_FASTCALL, nullptr},
    {"bwd", (PyCFunction)(void*)host_bwd, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "fa_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_fa_host(void) { return PyModule_Create(&module); }
