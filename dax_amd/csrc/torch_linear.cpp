// The whole forward of a W8A8 linear behind one call from Python: checks, allocations and the C entry points of
// libdaxq.so (dax_amd/lib/_daxq_torch.so).
//
// What bounds it: the host alone.  A small linear's kernels take 6 us (1 x 1536 x 1536) while the custom op in
// Python took 24 (its wrappers 10, the checks and the ctypes call with its 24 arguments 6, two launches 7), and a module
// that is not bf16 per-token paid two custom ops (48 us at 2900 x 1000 x 3080 fp16, whose kernels take 22).  A forward through
// here costs the host 9 us.  Forwards back to back, us, before -> after: 1 x 1536 x 1536 22.7 -> 10.6, 17 x 5120 x 5120 e4m3
// 22.7 -> 10.6, 2900 x 1000 x 3080 fp16 48.5 -> 23.5, static 4725 x 5120 x 5120 e4m3 113.4 -> 108.6 (its kernels' time).
//
// linear() covers calls that the dispatcher would hand to the CUDA kernel without anything in between.  Everything
// else (gradients, forward-mode tangents, function modes, dispatch modes, functorch, autocast, tracing, a profiler's
// callbacks, an argument that a check refuses) returns None and the caller takes the custom op, which records, dispatches or
// raises as before.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/daxq.h"

namespace {

constexpr int64_t kAlign = DAXQ_K_ALIGN;
constexpr int64_t kRowPad = 128;          // as Q_ROW_PAD of ops.py: rows of whole kilobytes are kept a line apart
constexpr float kEps = 1.1920928955078125e-07f;

enum Scheme { kToken = 0, kTensor = 1, kStatic = 2 };

int float_kind(at::ScalarType t) {
    return t == at::kBFloat16 ? DAXQ_BF16 : t == at::kHalf ? DAXQ_F16 : t == at::kFloat ? DAXQ_F32 : -1;
}

const at::Tensor* unpack(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// The dispatcher would go to the plain CUDA kernel, and nobody differentiates through any of these tensors
// (`detached` ones enter the general forward as plain values, too, whatever they require)
bool plain(std::initializer_list<const at::Tensor*> ts, std::initializer_list<const at::Tensor*> detached) {
    if (at::impl::torch_function_mode_enabled() || at::hasCallbacks()) return false;
    const auto tls = c10::impl::tls_local_dispatch_key_set();
    c10::DispatchKeySet ks = tls.included_;
    for (auto* t : ts)
        if (t) ks = ks | t->key_set();
    for (auto* t : detached)
        if (t) ks = ks | t->key_set();
    const auto top = (ks - tls.excluded_).highestPriorityTypeId();
    if (top != c10::DispatchKey::AutogradCUDA && top != c10::DispatchKey::ADInplaceOrView && top != c10::DispatchKey::CUDA) return false;
    const bool grad = c10::GradMode::is_enabled();
    for (auto* t : ts) {
        if (!t) continue;
        if (grad && t->requires_grad()) return false;
        if (t->_fw_grad(0).defined()) return false;
    }
    // the dispatcher's fallbacks materialise these (their keys rank below autograd's); the bytes here are not the values
    for (auto& list : {ts, detached})
        for (auto* t : list)
            if (t && (t->is_neg() || t->_is_zerotensor())) return false;
    return true;
}

// linear(x, wq, sw, bias, in_scale, k, x_fmt, w_fmt, out_kind, scheme, scale_fp32, kernel)
//   x [..., k]; wq [n, pad128(k)] in its stored type or as bytes; sw fp32 [n], any shape; bias [n] of the output's type or None; in_scale fp32 [1] (static) or None
// -> the output [..., n], None (not a plain call), or the non-zero status of a C entry point.
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 12) {
        PyErr_SetString(PyExc_TypeError, "linear() takes 12 arguments");
        return nullptr;
    }
    const at::Tensor *x = unpack(a[0]), *wq = unpack(a[1]), *sw = unpack(a[2]);
    const at::Tensor *bias = a[3] == Py_None ? nullptr : unpack(a[3]), *in_scale = a[4] == Py_None ? nullptr : unpack(a[4]);
    if (!x || !wq || !sw || (a[3] != Py_None && !bias) || (a[4] != Py_None && !in_scale)) Py_RETURN_NONE;
    const int64_t k = PyLong_AsLongLong(a[5]);
    const int x_fmt = (int)PyLong_AsLong(a[6]), w_fmt = (int)PyLong_AsLong(a[7]), out_kind = (int)PyLong_AsLong(a[8]);
    const int scheme = (int)PyLong_AsLong(a[9]), scale_fp32 = PyObject_IsTrue(a[10]), kernel = (int)PyLong_AsLong(a[11]);
    if (PyErr_Occurred()) return nullptr;
    if (!plain({x, sw, in_scale}, {wq, bias})) Py_RETURN_NONE;

    const auto dev = x->device();
    const int x_kind = float_kind(x->scalar_type());
    if (!dev.is_cuda() || x_kind < 0 || x->layout() != at::kStrided || wq->device() != dev || sw->device() != dev) Py_RETURN_NONE;
    if ((bias && bias->device() != dev) || (scheme == kStatic) != (in_scale != nullptr)) Py_RETURN_NONE;
    const auto out_type = out_kind == DAXQ_BF16 ? at::kBFloat16 : out_kind == DAXQ_F16 ? at::kHalf : at::kFloat;
    const auto w_type = wq->scalar_type();  // the stored FP8 type, or its bytes
    if (w_fmt == DAXQ_FMT_I8 ? w_type != at::kChar : w_type != at::kByte && w_type != (w_fmt == DAXQ_FMT_E4M3 ? at::kFloat8_e4m3fn : at::kFloat8_e5m2)) Py_RETURN_NONE;
    if (wq->dim() != 2 || !wq->is_contiguous()) Py_RETURN_NONE;
    const int64_t n = wq->size(0), kp = wq->size(1);
    if (k <= 0 || n <= 0 || kp != (k + kAlign - 1) / kAlign * kAlign || x->dim() < 1 || x->size(-1) != k || x->numel() == 0) Py_RETURN_NONE;
    if (sw->scalar_type() != at::kFloat || sw->numel() != n || !sw->is_contiguous()) Py_RETURN_NONE;
    if (bias && (bias->scalar_type() != out_type || bias->numel() != n || !bias->is_contiguous())) Py_RETURN_NONE;
    if (in_scale && (in_scale->device() != dev || in_scale->scalar_type() != at::kFloat || in_scale->numel() != 1)) Py_RETURN_NONE;
    if (scheme != kToken && k > DAXQ_MAX_TENSOR_K) Py_RETURN_NONE;
    // rows: a matrix of contiguous rows at any distance, or a contiguous tensor of any shape
    int64_t m = x->numel() / k, ld_x = k;
    if (!x->is_contiguous()) {
        if (x->dim() != 2 || x->stride(1) != 1 || (m > 1 && x->stride(0) < k)) Py_RETURN_NONE;
        if (m > 1) ld_x = x->stride(0);
    }
    // a handful of rows, or some more short ones: one launch that quantises for itself
    const bool few = kernel == 0 && m <= 64 && (m <= 8 ? daxq_linear_few_applies : daxq_linear_short_rows_applies)(x_kind, x_fmt, w_fmt, out_kind, scheme, scale_fp32 ? 0 : 1, m, n, k);
    // rows that the buffers hold: 64 or 128 where that many in a tiled kernel are faster than m (what the rows beyond m hold is
    // never looked at, their outputs are cut off); a kernel chosen by name runs on the rows there are
    const int64_t rows = kernel == 0 ? daxq_linear_launch_rows(x_fmt, m, n, k) : m;

    at::Tensor out;
    int rc = 0;
    {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(dev);
        auto shape = x->sizes().vec();
        shape.back() = n;
        const auto opt = at::TensorOptions().device(dev);
        if (few) {
            out = at::empty(shape, opt.dtype(out_type));
            rc = (m <= 8 ? daxq_linear_few : daxq_linear_short_rows)(x_kind, x_fmt, w_fmt, out_kind, scheme, scale_fp32 ? 0 : 1, x->const_data_ptr(), ld_x,
                                 in_scale ? in_scale->const_data_ptr<float>() : nullptr, wq->const_data_ptr(), kp, sw->const_data_ptr<float>(),
                                 bias ? bias->const_data_ptr() : nullptr, out.mutable_data_ptr(), n, m, n, k,
                                 c10::hip::getCurrentHIPStream(dev.index()).stream());
        } else {
            const int64_t ld_q = kp + (kp % 1024 == 0 ? kRowPad : 0);
            // the quantised rows, their scales (the row length is a multiple of 128: aligned), 1 KiB for the abs-max of a tensor
            const int64_t scales = rows * ld_q, partial = (scales + 4 * rows + 15) / 16 * 16;
            const at::Tensor scratch = at::empty({partial + (scheme == kTensor ? 1024 : 0)}, opt.dtype(at::kByte));
            out = rows == m ? at::empty(shape, opt.dtype(out_type)) : at::empty({rows, n}, opt.dtype(out_type));
            uint8_t* q = static_cast<uint8_t*>(scratch.mutable_data_ptr());
            float* sx = reinterpret_cast<float*>(q + scales);
            void* st = c10::hip::getCurrentHIPStream(dev.index()).stream();
            const void *xp = x->const_data_ptr(), *wp = wq->const_data_ptr(), *bp = bias ? bias->const_data_ptr() : nullptr;
            const float* swp = sw->const_data_ptr<float>();
            void* op = out.mutable_data_ptr();
            const float qmax = x_fmt == DAXQ_FMT_I8 ? 127.0f : x_fmt == DAXQ_FMT_E4M3 ? 448.0f : 57344.0f;
            if (scheme == kToken)
                rc = daxq_act_quant_rows_ex(xp, x_kind, x_fmt, m, k, ld_x, q, ld_q, sx, qmax, kEps, scale_fp32 ? 0 : 1, st);
            else if (scheme == kTensor)
                rc = daxq_act_quant_tensor(xp, x_kind, x_fmt, m, k, ld_x, q, ld_q, sx, nullptr, q + partial, qmax, kEps, scale_fp32 ? 0 : 1, st);
            else
                rc = daxq_quantize_tensor(xp, x_kind, x_fmt, m, k, ld_x, in_scale->const_data_ptr<float>(), q, ld_q, sx, st);
            if (!rc) rc = daxq_linear_w8a8(x_fmt, w_fmt, out_kind, q, ld_q, sx, wp, kp, swp, bp, op, n, nullptr, n, rows, n, kp, kernel, st);
        }
        if (!few && rows != m) {
            const at::AutoDispatchBelowADInplaceOrView below;  // (the cut is no view of another tensor for the caller)
            out = out.narrow(0, 0, m).view(shape);
        }
    }
    if (rc) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// holds_its_values(t): False for a tensor whose memory is not what it stands for, and which the dispatcher therefore rewrites or unwraps
// before a kernel sees it: lazily negated, zero without storage, wrapped by a function transform, a subclass's.  (The three questions
// asked from Python cost a conversion 1 us.)
PyObject* holds_its_values(PyObject*, PyObject* a) {
    HANDLE_TH_ERRORS
    const at::Tensor* t = unpack(a);
    if (!t) Py_RETURN_FALSE;
    const auto top = (t->key_set() - c10::autograd_dispatch_keyset_with_ADInplaceOrView - c10::autocast_dispatch_keyset).highestPriorityTypeId();
    return PyBool_FromLong(top == c10::DispatchKey::CUDA || top == c10::DispatchKey::CPU);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"holds_its_values", holds_its_values, METH_O, "whether a tensor's memory is what it stands for"},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(linear)), METH_FASTCALL, "forward of a quantised linear, or None where the call is not a plain one"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_daxq_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__daxq_torch() {
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    // the rules that ops.py applies as well
    if (PyModule_AddIntConstant(m, "K_ALIGN", kAlign) || PyModule_AddIntConstant(m, "ROW_PAD", kRowPad) ||
        PyModule_AddIntConstant(m, "MAX_TENSOR_K", DAXQ_MAX_TENSOR_K) || PyModule_AddObject(m, "EPS", PyFloat_FromDouble(kEps))) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
