// The host side of a linear between the Python entry points and the library: what they ask of their tensors, the output, the workspace and
// the library call, as one native call.  A linear of few rows waits for the host (64 x 1024 -> 1024: 14.6 us of Python and ctypes in front of a
// kernel of 5), most of it attribute reads, argument conversion and two allocations through the interpreter.
//
// Every function here serves plain operands only -- fp16, contiguous, on the current device, of torch's own tensor class, outside
// any mode or transform that intercepts operations -- and returns None for everything else, before it has done anything: the
// caller's general code, which converts, copies and reports errors, then runs as if it had not been asked.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/version.h>

#include "vdmq.h"

namespace {

decltype(&vdmq_linear_bf6_ex) linear_bf6_ex;
decltype(&vdmq_linear_bf6_workspace) linear_bf6_workspace;
decltype(&vdmq_pack_weight) pack_weight;

constexpr int kInterface = 2; /* of the functions below; the package compares it with its own */
constexpr int64_t kMaxK = 16384; /* what the quantizers that write bf6 blocks take */

// Nothing intercepts operations: no __torch_function__ mode, no __torch_dispatch__ mode, no functorch transform.
bool plain_calls() {
    const auto included = c10::impl::tls_local_dispatch_key_set().included_;
    return at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !included.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                                  c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::Functionalize,
                                                  c10::DispatchKey::Tracer}));
}

// The tensor behind `obj` where that is torch's own class over ordinary device memory, else null.
const at::Tensor *plain(PyObject *obj) {
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(obj);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t._is_zerotensor() || t.is_neg() ||
        t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                 c10::DispatchKey::Functionalize, c10::DispatchKey::Fake})))
        return nullptr;
    return &t;
}

const at::Tensor *plain_half(PyObject *obj, c10::Device device) {
    const at::Tensor *t = plain(obj);
    return t != nullptr && t->scalar_type() == at::kHalf && t->device() == device && t->is_contiguous() ? t : nullptr;
}

// A packed weight of rows of K elements, as the checkpoint holds it: u8 [N, K / 2] and fp16 [N, K / 64].
bool packed_pair(PyObject *qweight, PyObject *wscales, c10::Device device, int64_t K, int64_t &N) {
    const at::Tensor *q = plain(qweight), *s = plain_half(wscales, device);
    if (q == nullptr || s == nullptr || q->scalar_type() != at::kByte || q->device() != device || !q->is_contiguous()) return false;
    if (q->dim() != 2 || s->dim() != 2 || q->size(1) != K / 2 || q->size(0) % 128 != 0 || s->size(0) != q->size(0) || s->size(1) != K / 64) return false;
    N = q->size(0);
    return N > 0;
}

// linear(prepare, x, shape, qweight, wscales, prepared, check_q, check_s, bias, clip, act, ln_mode, eps, a, b, rows_per_vec, residual, gate,
//        split_cols, views)
//
// `shape`: what x stands for, a tuple, or None where that is its own shape.
// `prepare(qweight, wscales, device index)` gives (blocks, scales, stream), or None where the device is not the current one.  It may make the
// weight's form, so everything else is checked in front of it.
// `prepared`: None, or qweight is a prepared weight (without `wscales`) and this its (N, K).  The row length of x is what the library multiplies
// by: a weight of another is read beyond its end.
// check_q, check_s: a packed pair whose shapes the call checks besides, or None.
// Returns the output [..., N], with split_cols [N / split_cols, ..., split_cols], with views the tuple of its parts of that many
// columns; None: not served; an int: the library's error code.
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 20) {
        PyErr_SetString(PyExc_TypeError, "linear takes 20 arguments");
        return nullptr;
    }
    PyObject *const prepare = args[0];
    const at::Tensor *const x = plain(args[1]);
    if (x == nullptr || x->scalar_type() != at::kHalf || !x->is_contiguous() || x->dim() < 1 || !plain_calls()) Py_RETURN_NONE;
    const c10::Device device = x->device();
    const int64_t K = x->size(-1), M = K > 0 ? x->numel() / K : 0;
    c10::SmallVector<int64_t, 8> lead; /* the outputs' shape but for the channels */
    if (args[2] == Py_None) {
        lead.assign(x->sizes().begin(), x->sizes().end() - 1);
    } else {
        if (!PyTuple_CheckExact(args[2])) Py_RETURN_NONE;
        int64_t rows = 1;
        for (Py_ssize_t i = 0; i + 1 < PyTuple_GET_SIZE(args[2]); ++i) {
            lead.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(args[2], i)));
            rows *= lead.back();
        }
        if (PyErr_Occurred()) PyErr_Clear(), rows = -1;
        if (rows != M) Py_RETURN_NONE;
    }
    if (M <= 0 || K % 64 != 0 || K < VDMQ_LINEAR_BF6_MIN_K || K > kMaxK) Py_RETURN_NONE;
    int64_t N = 0, checked = 0;
    const bool packed = args[5] == Py_None;
    if (packed) {
        if (!packed_pair(args[3], args[4], device, K, N)) Py_RETURN_NONE;
    } else {
        long long n = 0, k = 0;
        if (!PyArg_ParseTuple(args[5], "LL", &n, &k)) return nullptr;
        if (k != K || n <= 0) Py_RETURN_NONE;
        N = n;
    }
    if (args[6] != Py_None && !packed_pair(args[6], args[7], device, K, checked)) Py_RETURN_NONE;
    const double clip = PyFloat_AsDouble(args[9]), eps = PyFloat_AsDouble(args[12]);
    const long act = PyLong_AsLong(args[10]), ln_mode = PyLong_AsLong(args[11]);
    const int64_t rows_per_vec = PyLong_AsLongLong(args[15]), split_cols = PyLong_AsLongLong(args[18]), views = PyLong_AsLongLong(args[19]);
    if (PyErr_Occurred()) { /* (the general code says what is wrong with it) */
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const at::Tensor *bias = nullptr, *a = nullptr, *b = nullptr, *residual = nullptr, *gate = nullptr;
    if (args[8] != Py_None && ((bias = plain_half(args[8], device)) == nullptr || bias->dim() != 1)) Py_RETURN_NONE;
    if (ln_mode != 0 && ((a = plain_half(args[13], device)) == nullptr || (b = plain_half(args[14], device)) == nullptr)) Py_RETURN_NONE;
    if (args[16] != Py_None && (residual = plain_half(args[16], device)) == nullptr) Py_RETURN_NONE;
    if (args[17] != Py_None && ((gate = plain_half(args[17], device)) == nullptr || gate->dim() < 1 || gate->numel() == 0)) Py_RETURN_NONE;
    if (bias != nullptr && bias->numel() != N) Py_RETURN_NONE;
    if (gate != nullptr && (gate->size(-1) != N || M % (gate->numel() / N) != 0)) Py_RETURN_NONE;
    if (residual != nullptr) {
        if (residual->dim() != static_cast<int64_t>(lead.size()) + 1 || residual->size(-1) != N) Py_RETURN_NONE;
        for (size_t i = 0; i < lead.size(); ++i)
            if (residual->size(static_cast<int64_t>(i)) != lead[i]) Py_RETURN_NONE;
    }
    if (split_cols != 0 && (split_cols < 0 || split_cols % 64 != 0 || N % split_cols != 0 || residual != nullptr || gate != nullptr)) Py_RETURN_NONE;
    if (views < 0 || (views != 0 && N % views != 0)) Py_RETURN_NONE;
    PyObject *const index = PyLong_FromLong(device.index());
    if (index == nullptr) return nullptr;
    PyObject *const question[3] = {args[3], args[4], index};
    THPObjectPtr prepared(PyObject_Vectorcall(prepare, question, 3, nullptr));
    Py_DECREF(index);
    if (!prepared) return nullptr;
    if (prepared.get() == Py_None) Py_RETURN_NONE;
    PyObject *blocks_obj, *wscale_obj;
    unsigned long long stream = 0;
    if (!PyArg_ParseTuple(prepared.get(), "O!O!K", THPVariableClass, &blocks_obj, THPVariableClass, &wscale_obj, &stream)) return nullptr;
    const at::Tensor &blocks = THPVariable_Unpack(blocks_obj), &wscale = THPVariable_Unpack(wscale_obj);

    c10::SmallVector<int64_t, 8> shape;
    if (split_cols != 0) shape.push_back(N / split_cols);
    shape.append(lead.begin(), lead.end());
    shape.push_back(split_cols != 0 ? split_cols : N);
    at::Tensor out, workspace;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        out = at::empty(shape, x->options());
        const int64_t rows_per_gate = gate != nullptr ? M / (gate->numel() / N) : 1, ldr = residual != nullptr ? N : 0;
        const int64_t nbytes = linear_bf6_workspace(M, N, K, static_cast<int>(act), static_cast<int>(ln_mode), gate != nullptr ? rows_per_gate : 0, ldr, VDMQ_OUT_F16);
        if (nbytes > 0) workspace = at::empty({nbytes}, x->options().dtype(at::kByte));
        rc = linear_bf6_ex(x->const_data_ptr(), M, K, K, static_cast<float>(clip), static_cast<int>(act), static_cast<int>(ln_mode), static_cast<float>(eps),
                           a != nullptr ? a->const_data_ptr() : nullptr, b != nullptr ? b->const_data_ptr() : nullptr, a != nullptr ? K : 0, rows_per_vec,
                           blocks.const_data_ptr(), wscale.const_data_ptr(), bias != nullptr ? bias->const_data_ptr() : nullptr,
                           gate != nullptr ? gate->const_data_ptr() : nullptr, gate != nullptr ? N : 0, rows_per_gate,
                           residual != nullptr ? residual->const_data_ptr() : nullptr, ldr, split_cols, split_cols != 0 ? M * split_cols : 0, out.mutable_data_ptr(),
                           VDMQ_OUT_F16, N, split_cols != 0 ? split_cols : N, nbytes > 0 ? workspace.mutable_data_ptr() : nullptr, nbytes,
                           reinterpret_cast<vdmq_stream_t>(stream));
    }
    if (rc != VDMQ_OK) return PyLong_FromLong(rc);
    if (views == 0) return THPVariable_Wrap(out);
    const std::vector<at::Tensor> parts = out.split(views, -1);
    THPObjectPtr tuple(PyTuple_New(static_cast<Py_ssize_t>(parts.size())));
    if (!tuple) return nullptr;
    for (size_t i = 0; i < parts.size(); ++i) {
        PyObject *const part = THPVariable_Wrap(parts[i]);
        if (part == nullptr) return nullptr;
        PyTuple_SET_ITEM(tuple.get(), static_cast<Py_ssize_t>(i), part);
    }
    return tuple.release();
    END_HANDLE_TH_ERRORS
}

// pack(weight, scale or None, current device index, stream): (qweight, packed scales, scales) of an fp16 weight that the bf6 path serves; None:
// not served; an int: the library's error code.
PyObject *pack(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 4) {
        PyErr_SetString(PyExc_TypeError, "pack takes 4 arguments");
        return nullptr;
    }
    const at::Tensor *const w = plain(args[0]);
    if (w == nullptr || w->scalar_type() != at::kHalf || !w->is_contiguous() || w->dim() != 2 || !plain_calls()) Py_RETURN_NONE;
    const int64_t N = w->size(0), K = w->size(1);
    if (N <= 0 || N % 128 != 0 || K < VDMQ_LINEAR_BF6_MIN_K || K % 64 != 0 || w->device().index() != PyLong_AsLong(args[2])) Py_RETURN_NONE;
    const at::Tensor *scale = nullptr;
    if (args[1] != Py_None && ((scale = plain_half(args[1], w->device())) == nullptr || scale->dim() != 1 || scale->numel() != N)) Py_RETURN_NONE;
    const unsigned long long stream = PyLong_AsUnsignedLongLong(args[3]);
    at::Tensor qweight, packed, derived;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        qweight = at::empty({N, K / 2}, w->options().dtype(at::kByte));
        packed = at::empty({N, K / 64}, w->options());
        if (scale == nullptr) derived = at::empty({N}, w->options());
        rc = pack_weight(w->const_data_ptr(), scale != nullptr ? scale->const_data_ptr() : nullptr, qweight.mutable_data_ptr(), packed.mutable_data_ptr(),
                         scale == nullptr ? derived.mutable_data_ptr() : nullptr, nullptr, N, K, reinterpret_cast<vdmq_stream_t>(stream));
    }
    if (rc != VDMQ_OK) return PyLong_FromLong(rc);
    THPObjectPtr q(THPVariable_Wrap(qweight)), p(THPVariable_Wrap(packed)), d(scale == nullptr ? THPVariable_Wrap(derived) : Py_NewRef(args[1]));
    if (!q || !p || !d) return nullptr;
    return PyTuple_Pack(3, q.get(), p.get(), d.get());
    END_HANDLE_TH_ERRORS
}

// plain(tensors...): whether tensor operations on them can be replaced by a kernel without anybody noticing: torch's own class over ordinary device
// memory, nothing that intercepts operations, and no tangent of forward-mode differentiation on any of them.
PyObject *plain_tensors(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!plain_calls()) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < nargs; ++i) {
        const at::Tensor *const t = plain(args[i]);
        if (t == nullptr || t->_fw_grad(0).defined()) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

PyObject *init(PyObject *, PyObject *args) {
    unsigned long long linear_at, workspace_at, pack_at;
    if (!PyArg_ParseTuple(args, "KKK", &linear_at, &workspace_at, &pack_at)) return nullptr;
    pack_weight = reinterpret_cast<decltype(pack_weight)>(pack_at);
    linear_bf6_ex = reinterpret_cast<decltype(linear_bf6_ex)>(linear_at);
    linear_bf6_workspace = reinterpret_cast<decltype(linear_bf6_workspace)>(workspace_at);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"init", init, METH_VARARGS, "addresses of vdmq_linear_bf6_ex, vdmq_linear_bf6_workspace and vdmq_pack_weight"},
                         {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear)), METH_FASTCALL, "a linear on plain operands, or None"},
                         {"plain", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(plain_tensors)), METH_FASTCALL, "whether a kernel may stand in for operations on these tensors"},
                         {"pack", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(pack)), METH_FASTCALL, "a weight's packed buffers, or None"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_vdmq_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__vdmq_host(void) {
    PyObject *const m = PyModule_Create(&module);
    if (m != nullptr && (PyModule_AddIntConstant(m, "interface", kInterface) != 0 || PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
