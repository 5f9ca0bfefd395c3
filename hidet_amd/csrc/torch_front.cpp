// Native front of the operators: the argument checks, the output allocation and the call of the library's
// entry point in one step of compiled code.  A decode loop makes one such call per linear layer and token, and the kernel
// of a 4096 x 4096 layer runs 6 us; the same work in Python with a ctypes call took 10 us of host time (16 x 4096 x 4096 on
// K-contiguous codes, calls back to back: 11.5 -> 5.6 us).
//
// Every function here takes torch tensors and either does the whole call or returns None, without an effect, when the
// arguments are not exactly what it handles (another dtype or layout, a subclass, something to be copied, an error to be
// reported): the Python operators then run their complete path.  Nothing is remembered about a tensor between calls; the
// workspaces are those of hidet_amd.ffi, looked up by (device, stream) on every call.
#include <ATen/ATen.h>
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "../../include/hidet_qmm.h"

namespace {

// Entry points of libhidet_qmm.so, handed over by hidet_amd.ffi (which opened the library), and what errors need.
struct Library {
    decltype(&hidet_get_last_error) get_last_error;
    decltype(&hidet_symmetric_quant_matmul_f16_i8) w8a16;
    decltype(&hidet_symmetric_quant_matmul_f16_i8_bias) w8a16_bias;
    decltype(&hidet_symmetric_quant_matmul_f16_i8_nk) w8a16_nk;
    decltype(&hidet_symmetric_quant_matmul_f16_i8_nk_bias) w8a16_nk_bias;
    decltype(&hidet_symmetric_quant_matmul_w4a16) w4a16;
    decltype(&hidet_symmetric_quant_matmul_w4a16_bias) w4a16_bias;
    decltype(&hidet_fp8_quantize_per_tensor) fp8_quantize;
    decltype(&hidet_matmul_f8) matmul_f8;
    decltype(&hidet_matmul_f8_scaled) matmul_f8_scaled;
    decltype(&hidet_symmetric_quantize) quantize;
    decltype(&hidet_symmetric_dequantize) dequantize;
    decltype(&hidet_group_quantize_int4) quantize_int4;
    decltype(&hidet_symmetric_quant_matmul_w4a16_nk) w4a16_nk;
} lib;
PyObject *workspaces = nullptr;      // hidet_amd.ffi._WORKSPACES: (device, stream) -> uint8 tensor
PyObject *new_workspace = nullptr;   // hidet_amd.ffi.workspace(device): makes the entry
PyObject *failure = nullptr;         // hidet_amd.ffi.failure(entry point, arguments, error): the exception to raise

const at::Tensor *tensor(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

// A GPU tensor of that type (an argument of these functions: anything else is left to Python).
const at::Tensor *gpu_tensor(PyObject *o, at::ScalarType type) {
    const at::Tensor *t = tensor(o);
    return t != nullptr && t->is_cuda() && t->scalar_type() == type && t->layout() == at::kStrided ? t : nullptr;
}

bool same_device(const at::Tensor &a, const at::Tensor &b) { return a.get_device() == b.get_device(); }

struct Rows {
    int64_t m, stride;
};
// The leading axes of `a` folded into rows of `k` contiguous elements, where that needs no copy.
bool as_rows(const at::Tensor &a, int64_t k, Rows *r) {
    if (a.dim() < 2 || k == 0 || a.size(-1) != k) return false;
    r->m = a.numel() / k;
    r->stride = k;
    if (r->m == 0) return false;
    if (a.is_contiguous()) return true;
    if (a.dim() != 2 || a.stride(1) != 1 || a.stride(0) < k) return false;
    if (r->m > 1) r->stride = a.stride(0);
    return true;
}

struct Workspace {
    void *stream, *ptr;
    int64_t bytes;
};
// The current stream of the tensor's device and its workspace; false with a Python error set.
bool stream_and_workspace(const at::Tensor &t, Workspace *w) {
    const auto device = t.get_device();
    w->stream = c10::hip::getCurrentHIPStream(device).stream();
    PyObject *key = Py_BuildValue("(iL)", int(device), static_cast<long long>(reinterpret_cast<intptr_t>(w->stream)));
    if (key == nullptr) return false;
    PyObject *ws = PyDict_GetItemWithError(workspaces, key);  // borrowed
    Py_DECREF(key);
    PyObject *made = nullptr;
    if (ws == nullptr) {
        if (PyErr_Occurred()) return false;
        PyObject *dev = THPDevice_New(t.device());
        if (dev == nullptr) return false;
        ws = made = PyObject_CallFunctionObjArgs(new_workspace, dev, nullptr);
        Py_DECREF(dev);
        if (made == nullptr) return false;
    }
    const at::Tensor &buffer = THPVariable_Unpack(ws);
    w->ptr = buffer.data_ptr();
    w->bytes = buffer.numel();
    Py_XDECREF(made);  // the dictionary holds it
    return true;
}

at::Tensor output(const at::Tensor &a, int64_t n, at::ScalarType type) {
    auto sizes = a.sizes().vec();
    sizes.back() = n;
    return at::empty(sizes, a.options().dtype(type).requires_grad(false));
}

// The result, or the library's error as an exception that names the entry point and describes the arguments.
PyObject *finish(const char *name, PyObject *const *args, Py_ssize_t nargs, PyObject *result) {
    const char *error = lib.get_last_error();
    if (error == nullptr) return result;
    Py_XDECREF(result);
    PyObject *list = PyTuple_New(nargs);
    if (list == nullptr) return nullptr;
    for (Py_ssize_t i = 0; i < nargs; ++i) {
        Py_INCREF(args[i]);
        PyTuple_SET_ITEM(list, i, args[i]);
    }
    PyObject *exception = PyObject_CallFunction(failure, "sOs", name, list, error);
    Py_DECREF(list);
    if (exception == nullptr) return nullptr;
    PyErr_SetObject(reinterpret_cast<PyObject *>(Py_TYPE(exception)), exception);
    Py_DECREF(exception);
    return nullptr;
}

PyObject *pair(at::Tensor first, at::Tensor second) {
    PyObject *p = PyTuple_New(2);
    if (p == nullptr) return nullptr;
    PyTuple_SET_ITEM(p, 0, THPVariable_Wrap(std::move(first)));
    PyTuple_SET_ITEM(p, 1, THPVariable_Wrap(std::move(second)));
    return p;
}

// Dtype codes of the ABI; -1: none.
int float_code(at::ScalarType type) {
    switch (type) {
        case at::kFloat: return HIDET_QMM_F32;
        case at::kHalf: return HIDET_QMM_F16;
        case at::kBFloat16: return HIDET_QMM_BF16;
        default: return -1;
    }
}
int output_code(at::ScalarType type) { return type == at::kFloat8_e4m3fn ? HIDET_QMM_E4M3 : float_code(type); }

template <typename F>
PyObject *guarded(F &&f) {
    try {
        return f();
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// a, weight, scale, bias or None
PyObject *w8a16(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *a = nargs == 4 ? gpu_tensor(args[0], at::kHalf) : nullptr;
        const at::Tensor *w = a ? gpu_tensor(args[1], at::kChar) : nullptr;
        const at::Tensor *scale = w ? gpu_tensor(args[2], at::kHalf) : nullptr;
        const bool biased = nargs == 4 && args[3] != Py_None;
        const at::Tensor *bias = scale && biased ? gpu_tensor(args[3], at::kHalf) : nullptr;
        Rows rows;
        if (scale == nullptr || (biased && bias == nullptr) || w->dim() != 2 || !same_device(*a, *w) || !same_device(*a, *scale)) Py_RETURN_NONE;
        const int64_t k = w->size(0), n = w->size(1);
        if (n == 0 || k % 2 != 0 || n % 2 != 0 || !as_rows(*a, k, &rows) || scale->dim() != 1 || scale->size(0) != n || !scale->is_contiguous()) Py_RETURN_NONE;
        if (biased && (bias->dim() != 1 || bias->size(0) != n || !bias->is_contiguous() || !same_device(*a, *bias))) Py_RETURN_NONE;
        const bool row_major = w->is_contiguous();
        const int64_t ldw = w->stride(1);
        // the same operand held K-contiguous: up to 16 rows (more rows and everything else: the Python operator)
        if (!row_major && !(rows.m <= 16 && w->stride(0) == 1 && ldw >= k && ldw % 16 == 0 && k % 16 == 0 && reinterpret_cast<uintptr_t>(w->data_ptr()) % 16 == 0))
            Py_RETURN_NONE;
        Workspace ws;
        if (!stream_and_workspace(*a, &ws)) return nullptr;
        at::Tensor c = output(*a, n, at::kHalf);
        const void *ap = a->data_ptr(), *wp = w->data_ptr(), *sp = scale->data_ptr(), *bp = biased ? bias->data_ptr() : nullptr;
        void *cp = c.data_ptr();
        if (row_major) {
            if (biased) lib.w8a16_bias(ap, wp, sp, bp, cp, rows.m, k, n, rows.stride, 0, ws.ptr, ws.bytes, ws.stream);
            else lib.w8a16(ap, wp, sp, cp, rows.m, k, n, rows.stride, 0, ws.ptr, ws.bytes, ws.stream);
        } else {
            if (biased) lib.w8a16_nk_bias(ap, wp, sp, bp, cp, rows.m, k, n, rows.stride, ldw, ws.ptr, ws.bytes, ws.stream);
            else lib.w8a16_nk(ap, wp, sp, cp, rows.m, k, n, rows.stride, ldw, ws.ptr, ws.bytes, ws.stream);
        }
        const char *name = row_major ? (biased ? "hidet_symmetric_quant_matmul_f16_i8_bias" : "hidet_symmetric_quant_matmul_f16_i8")
                                     : (biased ? "hidet_symmetric_quant_matmul_f16_i8_nk_bias" : "hidet_symmetric_quant_matmul_f16_i8_nk");
        return finish(name, args, nargs, THPVariable_Wrap(std::move(c)));
    });
}

// A group size; false where it is no int, not positive or more than the ABI's type holds.
bool group_of(PyObject *o, int64_t *group) {
    if (!PyLong_CheckExact(o)) return false;
    *group = PyLong_AsLong(o);
    if (*group == -1) PyErr_Clear();  // (set where no long holds it)
    return *group > 0 && *group <= INT32_MAX;
}

// a, packed, scales, group size, bias or None
PyObject *w4a16(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *a = nargs == 5 ? tensor(args[0]) : nullptr;
        if (a == nullptr || !a->is_cuda() || (a->scalar_type() != at::kHalf && a->scalar_type() != at::kBFloat16)) Py_RETURN_NONE;
        const at::Tensor *w = gpu_tensor(args[1], at::kByte), *scales = w ? gpu_tensor(args[2], a->scalar_type()) : nullptr;
        const bool biased = args[4] != Py_None;
        const at::Tensor *bias = scales && biased ? gpu_tensor(args[4], a->scalar_type()) : nullptr;
        int64_t group;
        if (scales == nullptr || (biased && bias == nullptr) || !group_of(args[3], &group)) Py_RETURN_NONE;
        if (w->dim() != 2 || scales->dim() != 2 || !w->is_contiguous() || !scales->is_contiguous() || !same_device(*a, *w) || !same_device(*a, *scales)) Py_RETURN_NONE;
        const int64_t k = w->size(0), n = w->size(1) * 2;
        Rows rows;
        if (n == 0 || k % group != 0 || scales->size(0) != k / group || scales->size(1) != n || !as_rows(*a, k, &rows)) Py_RETURN_NONE;
        if (biased && (bias->dim() != 1 || bias->size(0) != n || !bias->is_contiguous() || !same_device(*a, *bias))) Py_RETURN_NONE;
        Workspace ws;
        if (!stream_and_workspace(*a, &ws)) return nullptr;
        at::Tensor c = output(*a, n, a->scalar_type());
        const int dtype = a->scalar_type() == at::kHalf ? HIDET_QMM_F16 : HIDET_QMM_BF16;
        if (biased)
            lib.w4a16_bias(a->data_ptr(), w->data_ptr(), scales->data_ptr(), bias->data_ptr(), c.data_ptr(), rows.m, k, n, rows.stride, int(group), dtype, 0,
                           ws.ptr, ws.bytes, ws.stream);
        else
            lib.w4a16(a->data_ptr(), w->data_ptr(), scales->data_ptr(), c.data_ptr(), rows.m, k, n, rows.stride, int(group), dtype, 0, ws.ptr, ws.bytes, ws.stream);
        return finish(biased ? "hidet_symmetric_quant_matmul_w4a16_bias" : "hidet_symmetric_quant_matmul_w4a16", args, nargs, THPVariable_Wrap(std::move(c)));
    });
}

// x -> (codes, scale)
PyObject *fp8_quantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *x = nargs == 1 ? tensor(args[0]) : nullptr;
        if (x == nullptr || !x->is_cuda() || !x->is_contiguous()) Py_RETURN_NONE;
        const int dtype = float_code(x->scalar_type());
        if (dtype < 0) Py_RETURN_NONE;
        Workspace ws;
        if (!stream_and_workspace(*x, &ws)) return nullptr;
        at::Tensor codes = at::empty(x->sizes(), x->options().dtype(at::kFloat8_e4m3fn).requires_grad(false));
        at::Tensor scale = at::empty({1}, x->options().dtype(at::kFloat).requires_grad(false));
        lib.fp8_quantize(x->data_ptr(), codes.data_ptr(), scale.data_ptr(), x->numel(), dtype, ws.ptr, ws.bytes, ws.stream);
        return finish("hidet_fp8_quantize_per_tensor", args, nargs, pair(std::move(codes), std::move(scale)));
    });
}

// a, b [N, K] (both float8_e4m3), scale_a, scale_b (float32, one element; both None: unscaled), output dtype
PyObject *matmul_f8(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *a = nargs == 5 ? gpu_tensor(args[0], at::kFloat8_e4m3fn) : nullptr, *b = a ? gpu_tensor(args[1], at::kFloat8_e4m3fn) : nullptr;
        if (b == nullptr || !THPDtype_Check(args[4]) || b->dim() != 2 || !same_device(*a, *b)) Py_RETURN_NONE;
        const at::Tensor *scale[2] = {nullptr, nullptr};
        if ((args[2] == Py_None) != (args[3] == Py_None)) Py_RETURN_NONE;
        for (int i = 0; i < 2; ++i) {
            if (args[2 + i] == Py_None) continue;
            scale[i] = gpu_tensor(args[2 + i], at::kFloat);
            if (scale[i] == nullptr || scale[i]->numel() != 1 || !same_device(*a, *scale[i])) Py_RETURN_NONE;
        }
        const at::ScalarType type = reinterpret_cast<THPDtype *>(args[4])->scalar_type;
        const int out = output_code(type);
        if (out < 0) Py_RETURN_NONE;
        const int64_t n = b->size(0), k = b->size(1);
        Rows rows;
        if (n == 0 || !as_rows(*a, k, &rows) || (k > 1 && b->stride(1) != 1) || (n > 1 && b->stride(0) < k)) Py_RETURN_NONE;
        Workspace ws;
        if (!stream_and_workspace(*a, &ws)) return nullptr;
        at::Tensor c = output(*a, n, type);
        lib.matmul_f8(a->data_ptr(), b->data_ptr(), c.data_ptr(), rows.m, n, k, rows.stride, n > 1 ? b->stride(0) : k, out, scale[0] ? scale[0]->data_ptr() : nullptr,
                      scale[1] ? scale[1]->data_ptr() : nullptr, ws.ptr, ws.bytes, ws.stream);
        return finish("hidet_matmul_f8", args, nargs, THPVariable_Wrap(std::move(c)));
    });
}

// a [M, K], b [N, K], scale_a [K / 128, M], scale_b [N / 128, K / 128], output dtype: two-dimensional and dense
PyObject *matmul_f8_scaled(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *a = nargs == 5 ? gpu_tensor(args[0], at::kFloat8_e4m3fn) : nullptr, *b = a ? gpu_tensor(args[1], at::kFloat8_e4m3fn) : nullptr;
        const at::Tensor *sa = b ? gpu_tensor(args[2], at::kFloat) : nullptr, *sb = sa ? gpu_tensor(args[3], at::kFloat) : nullptr;
        if (sb == nullptr || !THPDtype_Check(args[4])) Py_RETURN_NONE;
        const at::ScalarType type = reinterpret_cast<THPDtype *>(args[4])->scalar_type;
        const int out = output_code(type);
        for (const at::Tensor *t : {a, b, sa, sb})
            if (t->dim() != 2 || !t->is_contiguous() || !same_device(*a, *t)) Py_RETURN_NONE;
        const int64_t m = a->size(0), k = a->size(1), n = b->size(0);
        if (out < 0 || m == 0 || n == 0 || k == 0 || k % 128 != 0 || n % 128 != 0 || b->size(1) != k) Py_RETURN_NONE;
        if (sa->size(0) != k / 128 || sa->size(1) != m || sb->size(0) != n / 128 || sb->size(1) != k / 128) Py_RETURN_NONE;
        Workspace ws;
        if (!stream_and_workspace(*a, &ws)) return nullptr;
        at::Tensor c = output(*a, n, type);
        lib.matmul_f8_scaled(a->data_ptr(), b->data_ptr(), sa->data_ptr(), sb->data_ptr(), c.data_ptr(), m, n, k, out, ws.ptr, ws.bytes, ws.stream);
        return finish("hidet_matmul_f8_scaled", args, nargs, THPVariable_Wrap(std::move(c)));
    });
}

// One reduced axis: an int, or a list or tuple of one. The view of the quantizers is [outer, reduce, inner].
struct View {
    int64_t axis, outer, reduce, inner;
};
bool view_of(const at::Tensor &t, PyObject *dims, View *v) {
    if (PyList_CheckExact(dims) && PyList_GET_SIZE(dims) == 1) dims = PyList_GET_ITEM(dims, 0);
    if (!PyLong_CheckExact(dims)) return false;
    v->axis = PyLong_AsLong(dims);
    if (v->axis == -1 && PyErr_Occurred()) {  // no long holds it
        PyErr_Clear();
        return false;
    }
    if (v->axis < 0) v->axis += t.dim();
    if (v->axis < 0 || v->axis >= t.dim()) return false;
    v->outer = v->inner = 1;
    for (int64_t d = 0; d < v->axis; ++d) v->outer *= t.size(d);
    for (int64_t d = v->axis + 1; d < t.dim(); ++d) v->inner *= t.size(d);
    v->reduce = t.size(v->axis);
    return true;
}

// w, code dtype (torch.int8 or torch.int16), axis -> (codes, scale)
PyObject *quantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *w = nargs == 3 ? tensor(args[0]) : nullptr;
        View v;
        if (w == nullptr || !w->is_cuda() || !w->is_contiguous() || !THPDtype_Check(args[1]) || !view_of(*w, args[2], &v)) Py_RETURN_NONE;
        const int dtype = float_code(w->scalar_type());
        const at::ScalarType type = reinterpret_cast<THPDtype *>(args[1])->scalar_type;
        Workspace ws;
        if (dtype < 0 || (type != at::kChar && type != at::kShort) || w->numel() == 0) Py_RETURN_NONE;
        if (!stream_and_workspace(*w, &ws)) return nullptr;
        if (ws.bytes / 16 < v.outer * v.inner) Py_RETURN_NONE;  // (a larger workspace is ffi.workspace's business)
        auto kept = w->sizes().vec();
        kept.erase(kept.begin() + v.axis);
        at::Tensor codes = at::empty(w->sizes(), w->options().dtype(type).requires_grad(false));
        at::Tensor scale = at::empty(kept, w->options().requires_grad(false));
        lib.quantize(w->data_ptr(), codes.data_ptr(), scale.data_ptr(), v.outer, v.reduce, v.inner, dtype, type == at::kChar ? HIDET_QMM_I8 : HIDET_QMM_I16, ws.ptr,
                     ws.bytes, ws.stream);
        return finish("hidet_symmetric_quantize", args, nargs, pair(std::move(codes), std::move(scale)));
    });
}

// codes, scale, axis
PyObject *dequantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *q = nargs == 3 ? tensor(args[0]) : nullptr, *scale = q ? tensor(args[1]) : nullptr;
        View v;
        if (scale == nullptr || !q->is_cuda() || !scale->is_cuda() || !same_device(*q, *scale) || !q->is_contiguous() || !scale->is_contiguous() ||
            (q->scalar_type() != at::kChar && q->scalar_type() != at::kShort) || !view_of(*q, args[2], &v))
            Py_RETURN_NONE;
        const int dtype = float_code(scale->scalar_type());
        auto kept = q->sizes().vec();
        kept.erase(kept.begin() + v.axis);
        if (dtype < 0 || q->numel() == 0 || scale->sizes() != at::IntArrayRef(kept)) Py_RETURN_NONE;
        at::Tensor w = at::empty(q->sizes(), scale->options().requires_grad(false));
        lib.dequantize(q->data_ptr(), scale->data_ptr(), w.data_ptr(), v.outer, v.reduce, v.inner, q->scalar_type() == at::kChar ? HIDET_QMM_I8 : HIDET_QMM_I16, dtype,
                       c10::hip::getCurrentHIPStream(q->get_device()).stream());
        return finish("hidet_symmetric_dequantize", args, nargs, THPVariable_Wrap(std::move(w)));
    });
}

// w float32 [K, N], group size, scale dtype -> (packed, scales)
PyObject *quantize_int4(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *w = nargs == 3 ? gpu_tensor(args[0], at::kFloat) : nullptr;
        int64_t group;
        if (w == nullptr || w->dim() != 2 || !w->is_contiguous() || w->numel() == 0 || !group_of(args[1], &group) || !THPDtype_Check(args[2])) Py_RETURN_NONE;
        const at::ScalarType type = reinterpret_cast<THPDtype *>(args[2])->scalar_type;
        const int64_t k = w->size(0), n = w->size(1);
        if (k % group != 0 || n % 2 != 0 || (type != at::kHalf && type != at::kBFloat16)) Py_RETURN_NONE;
        at::Tensor packed = at::empty({k, n / 2}, w->options().dtype(at::kByte).requires_grad(false));
        at::Tensor scales = at::empty({k / group, n}, w->options().dtype(type).requires_grad(false));
        lib.quantize_int4(w->data_ptr(), packed.data_ptr(), scales.data_ptr(), k, n, int(group), HIDET_QMM_F32, type == at::kHalf ? HIDET_QMM_F16 : HIDET_QMM_BF16,
                          c10::hip::getCurrentHIPStream(w->get_device()).stream());
        return finish("hidet_group_quantize_int4", args, nargs, pair(std::move(packed), std::move(scales)));
    });
}

// a, packed [N, K / 2] (the decode layout), scales, group size
PyObject *w4a16_decode(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject * {
        const at::Tensor *a = nargs == 4 ? tensor(args[0]) : nullptr;
        if (a == nullptr || !a->is_cuda() || (a->scalar_type() != at::kHalf && a->scalar_type() != at::kBFloat16)) Py_RETURN_NONE;
        const at::Tensor *w = gpu_tensor(args[1], at::kByte), *scales = w ? gpu_tensor(args[2], a->scalar_type()) : nullptr;
        int64_t group;
        if (scales == nullptr || !group_of(args[3], &group) || w->dim() != 2 || scales->dim() != 2 || !w->is_contiguous() || !scales->is_contiguous() ||
            !same_device(*a, *w) || !same_device(*a, *scales))
            Py_RETURN_NONE;
        const int64_t n = w->size(0), k = w->size(1) * 2;
        Rows rows;
        if (n == 0 || k % group != 0 || scales->size(0) != k / group || scales->size(1) != n || !as_rows(*a, k, &rows)) Py_RETURN_NONE;
        if (rows.stride % 8 != 0 || reinterpret_cast<uintptr_t>(a->data_ptr()) % 16 != 0) Py_RETURN_NONE;
        at::Tensor c = output(*a, n, a->scalar_type());
        lib.w4a16_nk(a->data_ptr(), w->data_ptr(), scales->data_ptr(), c.data_ptr(), rows.m, k, n, rows.stride, k / 2, int(group),
                     a->scalar_type() == at::kHalf ? HIDET_QMM_F16 : HIDET_QMM_BF16, c10::hip::getCurrentHIPStream(a->get_device()).stream());
        return finish("hidet_symmetric_quant_matmul_w4a16_nk", args, nargs, THPVariable_Wrap(std::move(c)));
    });
}

// dict of entry point addresses, workspaces, workspace function, function that makes exceptions
PyObject *bind(PyObject *, PyObject *args) {
    PyObject *addresses;
    if (!PyArg_ParseTuple(args, "O!O!OO", &PyDict_Type, &addresses, &PyDict_Type, &workspaces, &new_workspace, &failure)) return nullptr;
    Py_INCREF(workspaces);
    Py_INCREF(new_workspace);
    Py_INCREF(failure);
    auto get = [&](auto &slot, const char *name) {
        PyObject *v = PyDict_GetItemString(addresses, name);
        void *p = v != nullptr ? PyLong_AsVoidPtr(v) : nullptr;
        slot = reinterpret_cast<std::decay_t<decltype(slot)>>(p);
        if (p == nullptr && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "no address for %s", name);
        return p != nullptr;
    };
    const bool ok = get(lib.get_last_error, "hidet_get_last_error") && get(lib.w8a16, "hidet_symmetric_quant_matmul_f16_i8") &&
                    get(lib.w8a16_bias, "hidet_symmetric_quant_matmul_f16_i8_bias") && get(lib.w8a16_nk, "hidet_symmetric_quant_matmul_f16_i8_nk") &&
                    get(lib.w8a16_nk_bias, "hidet_symmetric_quant_matmul_f16_i8_nk_bias") && get(lib.w4a16, "hidet_symmetric_quant_matmul_w4a16") &&
                    get(lib.w4a16_bias, "hidet_symmetric_quant_matmul_w4a16_bias") && get(lib.fp8_quantize, "hidet_fp8_quantize_per_tensor") &&
                    get(lib.matmul_f8, "hidet_matmul_f8") && get(lib.matmul_f8_scaled, "hidet_matmul_f8_scaled") &&
                    get(lib.quantize, "hidet_symmetric_quantize") && get(lib.dequantize, "hidet_symmetric_dequantize") &&
                    get(lib.quantize_int4, "hidet_group_quantize_int4") && get(lib.w4a16_nk, "hidet_symmetric_quant_matmul_w4a16_nk");
    if (!ok) return nullptr;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"w8a16", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(w8a16)), METH_FASTCALL, nullptr},
    {"w4a16", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(w4a16)), METH_FASTCALL, nullptr},
    {"fp8_quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fp8_quantize)), METH_FASTCALL, nullptr},
    {"matmul_f8", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(matmul_f8)), METH_FASTCALL, nullptr},
    {"matmul_f8_scaled", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(matmul_f8_scaled)), METH_FASTCALL, nullptr},
    {"quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(quantize)), METH_FASTCALL, nullptr},
    {"dequantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(dequantize)), METH_FASTCALL, nullptr},
    {"quantize_int4", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(quantize_int4)), METH_FASTCALL, nullptr},
    {"w4a16_decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(w4a16_decode)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_front", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front() { return PyModule_Create(&module); }
