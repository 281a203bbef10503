// Native form of the tensor-level entry points (catccos_amd/ops.py) for the calls that programs make in earnest: plain GPU
// tensors of the right types, shapes and layouts.  A decode step's kernels take 3 to 10 us and the same call through Python
// and ctypes 10 us of host time (checks, allocations, argument conversion, stream look-up), so that the host was what such a step
// waited for.  Measured, host time of a call: mx_quant 11.6 -> 4.3 us, mx_matmul 10.3 -> 4.1, dynamic_quant_i8 9.9 -> 4.1,
// moe_init_routing 11.9 -> 5.2, moe_ffn_mxfp8 56 -> 17.5 (of which three quarters are allocations and launches).
//
// Every function here answers Py_NotImplemented to a call it does not recognise as one of those, or that the library refuses,
// before or without any effect that outlives the call: the caller (ops.py) then takes the general path, which makes inputs
// contiguous, converts, and raises.  So nothing is accepted, refused or reported here that is not so there.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <cstring>

#include "catccos_hip.h"

namespace {

int64_t ScaleCols(int64_t k) { return 2 * ((k + 63) / 64); }   // E8M0 bytes per row: block count padded to even
bool IsFp4(int fmt) { return fmt == CCH_FMT_E2M1 || fmt == CCH_FMT_E1M2; }

PyObject *Decline()
{
    Py_INCREF(Py_NotImplemented);
    return Py_NotImplemented;
}

// No tracing, functorch transform, dispatch mode or function mode is active (autocast and the gradient modes leave these calls alone).
bool PlainThread()
{
    const auto usual = c10::default_included_set | c10::autocast_dispatch_keyset;
    return usual.has_all(c10::impl::tls_local_dispatch_key_set().included_) && !at::impl::torch_function_mode_enabled();
}

// A torch.Tensor (no subclass) in GPU memory, contiguous, with elements, of this type and rank, without a lazy negation,
// wrapper or the like.
bool Plain(PyObject *o, at::ScalarType type, int64_t dim)
{
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor &t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet usual =
        c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA});
    return t.defined() && t.is_cuda() && usual.has_all(t.key_set()) && t.scalar_type() == type && (dim < 0 || t.dim() == dim) && t.numel() > 0 &&
           t.is_contiguous();
}
const at::Tensor &T(PyObject *o) { return THPVariable_Unpack(o); }

bool Int(PyObject *o, int64_t &v)   // a Python int (or bool)
{
    if (!PyLong_Check(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0 && v >= -(int64_t)0x7FFFFFFF && v <= 0x7FFFFFFF;
}
bool Flag(PyObject *o, int &v)   // 0 or 1
{
    int64_t x;
    if (!Int(o, x) || x < 0 || x > 1) return false;
    v = (int)x;
    return true;
}
bool Format(PyObject *o, int &fmt)
{
    if (PyUnicode_Check(o)) {
        const char *s = PyUnicode_AsUTF8(o);
        if (s == nullptr) {
            PyErr_Clear();
            return false;
        }
        fmt = !strcmp(s, "e4m3") ? CCH_FMT_E4M3 : !strcmp(s, "e5m2") ? CCH_FMT_E5M2 : !strcmp(s, "e2m1") ? CCH_FMT_E2M1 : -1;
        return fmt >= 0;
    }
    int64_t v;
    if (!Int(o, v) || (v != CCH_FMT_E4M3 && v != CCH_FMT_E5M2 && v != CCH_FMT_E2M1)) return false;
    fmt = (int)v;
    return true;
}
bool OutType(PyObject *o, at::ScalarType &type)
{
    if (!THPDtype_Check(o)) return false;
    type = reinterpret_cast<THPDtype *>(o)->scalar_type;
    return type == at::kBFloat16 || type == at::kHalf;
}
int OutCode(at::ScalarType type) { return type == at::kHalf ? CCH_OUT_FP16 : CCH_OUT_BF16; }

at::Tensor New(const at::Tensor &like, at::IntArrayRef shape, at::ScalarType type) { return at::empty(shape, like.options().dtype(type).requires_grad(false)); }
void *Stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }   // of the current device, as in ops.py

PyObject *Pair(const at::Tensor &a, const at::Tensor &b)
{
    PyObject *x = THPVariable_Wrap(a), *y = x ? THPVariable_Wrap(b) : nullptr;
    PyObject *t = y ? PyTuple_New(2) : nullptr;
    if (t == nullptr) {
        Py_XDECREF(x);
        Py_XDECREF(y);
        return nullptr;
    }
    PyTuple_SET_ITEM(t, 0, x);
    PyTuple_SET_ITEM(t, 1, y);
    return t;
}

// mx_quant(x, fmt, rounding)
PyObject *MxQuant(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    int fmt;
    int64_t rounding;
    if (n != 3 || !PlainThread() || !(Plain(a[0], at::kBFloat16, 2) || Plain(a[0], at::kHalf, 2)) || !Format(a[1], fmt) || !Int(a[2], rounding)) return Decline();
    const at::Tensor &x = T(a[0]);
    const int64_t m = x.size(0), k = x.size(1);
    at::Tensor payload, scales;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        payload = New(x, {m, IsFp4(fmt) ? (k + 1) / 2 : k}, at::kByte);
        scales = New(x, {m, ScaleCols(k)}, at::kByte);
        rc = (x.scalar_type() == at::kHalf ? cch_mx_quant_rows_f16 : cch_mx_quant_rows)(x.data_ptr(), payload.data_ptr(), scales.data_ptr(), m, k, fmt,
                                                                                       (int)rounding, Stream());
    }
    return rc == CCH_OK ? Pair(payload, scales) : Decline();
    END_HANDLE_TH_ERRORS
}

// dynamic_quant_i8(x, src_rows, topk, mode)
PyObject *DynamicQuantI8(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    int64_t topk, mode;
    if (n != 4 || !PlainThread() || !Plain(a[0], at::kBFloat16, 2) || (a[1] != Py_None && !Plain(a[1], at::kInt, 1)) || !Int(a[2], topk) || !Int(a[3], mode))
        return Decline();
    const at::Tensor &x = T(a[0]);
    const int32_t *src = a[1] != Py_None ? static_cast<const int32_t *>(T(a[1]).data_ptr()) : nullptr;
    const int64_t rows_in = x.size(0), k = x.size(1), t = src ? T(a[1]).size(0) : rows_in;
    at::Tensor q, scale;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        q = New(x, {t, k}, at::kChar);
        scale = New(x, {t}, at::kFloat);
        rc = cch_dyn_quant_i8_rows(x.data_ptr(), src, q.data_ptr(), static_cast<float *>(scale.data_ptr()), rows_in, t, k, (int)topk, (int)mode, Stream());
    }
    return rc == CCH_OK ? Pair(q, scale) : Decline();
    END_HANDLE_TH_ERRORS
}

// moe_init_routing(expert_idx, num_experts, cumsum)
PyObject *MoeInitRouting(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    int64_t experts;
    if (n != 3 || !PlainThread() || !Plain(a[0], at::kInt, -1) || !Int(a[1], experts) || experts < 1 || !PyBool_Check(a[2])) return Decline();
    const at::Tensor &idx = T(a[0]);
    const int64_t rows = idx.numel();
    at::Tensor d2s, s2d, tokens;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        d2s = New(idx, {rows}, at::kInt);
        s2d = New(idx, {rows}, at::kInt);
        tokens = New(idx, {experts}, at::kInt);
        const int64_t bytes = std::max<int64_t>(cch_moe_init_routing_workspace_bytes(rows, (int)experts), 4);
        const at::Tensor ws = New(idx, {bytes}, at::kByte);
        rc = cch_moe_init_routing(static_cast<const int32_t *>(idx.data_ptr()), rows, (int)experts, static_cast<int32_t *>(d2s.data_ptr()),
                                  static_cast<int32_t *>(s2d.data_ptr()), static_cast<int32_t *>(tokens.data_ptr()), a[2] == Py_True ? 1 : 0, ws.data_ptr(), bytes,
                                  Stream());
    }
    if (rc != CCH_OK) return Decline();
    PyObject *o[3] = {THPVariable_Wrap(d2s), THPVariable_Wrap(s2d), THPVariable_Wrap(tokens)};
    PyObject *t = o[0] && o[1] && o[2] ? PyTuple_New(3) : nullptr;
    for (int i = 0; i < 3; i++) {
        if (t) PyTuple_SET_ITEM(t, i, o[i]);
        else Py_XDECREF(o[i]);
    }
    return t;
    END_HANDLE_TH_ERRORS
}

// w8a8_matmul_dequant(a, b, per_tok, per_ch, trans_b, out_dtype)
PyObject *W8A8(PyObject *, PyObject *const *v, Py_ssize_t nv)
{
    HANDLE_TH_ERRORS
    int trans_b;
    at::ScalarType type;
    if (nv != 6 || !PlainThread() || !Plain(v[0], at::kChar, 2) || !Plain(v[1], at::kChar, 2) || !Plain(v[2], at::kFloat, -1) || !Plain(v[3], at::kFloat, -1) ||
        !Flag(v[4], trans_b) || !OutType(v[5], type))
        return Decline();
    const at::Tensor &a = T(v[0]), &b = T(v[1]), &per_tok = T(v[2]), &per_ch = T(v[3]);
    const int64_t m = a.size(0), k = a.size(1), n = b.size(trans_b ? 0 : 1);
    if (b.size(trans_b ? 1 : 0) != k || per_tok.numel() != m || per_ch.numel() != n) return Decline();
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        out = New(a, {m, n}, type);
        rc = cch_gemm_i8_dequant_out(a.data_ptr(), b.data_ptr(), static_cast<const float *>(per_tok.data_ptr()), static_cast<const float *>(per_ch.data_ptr()),
                                     out.data_ptr(), m, n, k, trans_b, OutCode(type), Stream());
    }
    return rc == CCH_OK ? THPVariable_Wrap(out) : Decline();
    END_HANDLE_TH_ERRORS
}

// gmm_i8(x, w, group_sizes, per_tok, per_ch, trans_b, swiglu, out_dtype)
PyObject *GmmI8(PyObject *, PyObject *const *v, Py_ssize_t nv)
{
    HANDLE_TH_ERRORS
    int trans_b, swiglu;
    at::ScalarType type;
    if (nv != 8 || !PlainThread() || !Plain(v[0], at::kChar, 2) || !Plain(v[1], at::kChar, 3) || !Plain(v[2], at::kInt, 1) || !Plain(v[3], at::kFloat, -1) ||
        !Plain(v[4], at::kFloat, 2) || !Flag(v[5], trans_b) || !Flag(v[6], swiglu) || !OutType(v[7], type))
        return Decline();
    const at::Tensor &x = T(v[0]), &w = T(v[1]), &gs = T(v[2]), &per_tok = T(v[3]), &per_ch = T(v[4]);
    const int64_t t = x.size(0), k = x.size(1), e = w.size(0), n = w.size(trans_b ? 1 : 2);
    if (w.size(trans_b ? 2 : 1) != k || gs.numel() != e || per_tok.numel() != t || per_ch.size(0) != e || per_ch.size(1) != n) return Decline();
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        out = New(x, {t, swiglu ? n / 2 : n}, type);
        rc = (swiglu ? cch_gmm_i8_dequant_swiglu_out : cch_gmm_i8_dequant_out)(
            x.data_ptr(), w.data_ptr(), static_cast<const int32_t *>(gs.data_ptr()), static_cast<const float *>(per_tok.data_ptr()),
            static_cast<const float *>(per_ch.data_ptr()), out.data_ptr(), e, t, n, k, trans_b, OutCode(type), Stream());
    }
    return rc == CCH_OK ? THPVariable_Wrap(out) : Decline();
    END_HANDLE_TH_ERRORS
}

// mx_matmul(a, sa, b, sb, fmt, trans_b, out_dtype), mx_grouped_matmul(a, sa, b, sb, group_sizes, fmt, trans_b, out_dtype)
PyObject *MxProduct(PyObject *const *v, bool grouped)
{
    int fmt, trans_b;
    at::ScalarType type;
    const int g = grouped ? 1 : 0;
    if (!PlainThread() || !Plain(v[0], at::kByte, 2) || !Plain(v[1], at::kByte, 2) || !Plain(v[2], at::kByte, 2 + g) || !Plain(v[3], at::kByte, -1) ||
        (grouped && !Plain(v[4], at::kInt, 1)) || !Format(v[4 + g], fmt) || !Flag(v[5 + g], trans_b) || !OutType(v[6 + g], type))
        return Decline();
    const at::Tensor &a = T(v[0]), &sa = T(v[1]), &b = T(v[2]), &sb = T(v[3]);
    const int64_t pack = IsFp4(fmt) ? 2 : 1, m = a.size(0), k = a.size(1) * pack, e = grouped ? b.size(0) : 1;
    const int64_t n = trans_b ? b.size(g) : b.size(g + 1) * pack, kb = trans_b ? b.size(g + 1) * pack : b.size(g);
    if (kb != k || sa.size(0) != m || sa.size(1) != ScaleCols(k) || sb.numel() != e * ScaleCols(k) * n || (grouped && T(v[4]).numel() != e)) return Decline();
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        out = New(a, {m, n}, type);
        if (!grouped) {
            rc = cch_mx_gemm_out(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), out.data_ptr(), m, n, k, fmt, trans_b, OutCode(type), Stream());
        } else {
            const int32_t *gs = static_cast<const int32_t *>(T(v[4]).data_ptr());
            rc = type == at::kHalf ? cch_mx_gmm_mapped(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), gs, nullptr, out.data_ptr(), m, CCH_OUT_FP16, e, m,
                                                       n, k, fmt, trans_b, Stream())
                                   : cch_mx_gmm(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), gs, out.data_ptr(), e, m, n, k, fmt, trans_b, Stream());
        }
    }
    return rc == CCH_OK ? THPVariable_Wrap(out) : Decline();
}
PyObject *MxMatmul(PyObject *, PyObject *const *v, Py_ssize_t nv)
{
    HANDLE_TH_ERRORS
    return nv == 7 ? MxProduct(v, false) : Decline();
    END_HANDLE_TH_ERRORS
}
PyObject *MxGroupedMatmul(PyObject *, PyObject *const *v, Py_ssize_t nv)
{
    HANDLE_TH_ERRORS
    return nv == 8 ? MxProduct(v, true) : Decline();
    END_HANDLE_TH_ERRORS
}

// moe_ffn_mxfp8(x, expert_idx, probs, w1, sw1, w2, sw2, trans_b): what lies between the launches is one allocation
PyObject *MoeFfnMxfp8(PyObject *, PyObject *const *v, Py_ssize_t nv)
{
    HANDLE_TH_ERRORS
    int trans_b;
    if (nv != 8 || !PlainThread() || !Plain(v[0], at::kBFloat16, 2) || !Plain(v[1], at::kInt, 2) || !Plain(v[2], at::kFloat, 2) || !Plain(v[3], at::kByte, 3) ||
        !Plain(v[4], at::kByte, -1) || !Plain(v[5], at::kByte, 3) || !Plain(v[6], at::kByte, -1) || !Flag(v[7], trans_b))
        return Decline();
    const at::Tensor &x = T(v[0]), &idx = T(v[1]), &probs = T(v[2]), &w1 = T(v[3]), &sw1 = T(v[4]), &w2 = T(v[5]), &sw2 = T(v[6]);
    const int64_t m = x.size(0), k = x.size(1), top_k = idx.size(1), e = w1.size(0), n = w1.size(trans_b ? 1 : 2), h = n / 2;
    if (idx.size(0) != m || probs.sizes() != idx.sizes() || top_k > 8 || w1.size(trans_b ? 2 : 1) != k || n % 2 || h == 0 || w2.size(0) != e ||
        w2.size(trans_b ? 2 : 1) != h || w2.size(trans_b ? 1 : 2) != k || sw1.numel() != e * ScaleCols(k) * n || sw2.numel() != e * ScaleCols(h) * k)
        return Decline();
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        const int64_t bytes = cch_moe_ffn_mxfp8_workspace_bytes(m, k, (int)top_k, e, n);
        const at::Tensor ws = New(x, {bytes}, at::kByte);
        out = New(x, {m, k}, at::kBFloat16);
        rc = cch_moe_ffn_mxfp8(x.data_ptr(), static_cast<const int32_t *>(idx.data_ptr()), static_cast<const float *>(probs.data_ptr()), w1.data_ptr(),
                               sw1.data_ptr(), w2.data_ptr(), sw2.data_ptr(), out.data_ptr(), m, k, (int)top_k, e, n, trans_b, ws.data_ptr(), bytes, Stream());
    }
    return rc == CCH_OK ? THPVariable_Wrap(out) : Decline();
    END_HANDLE_TH_ERRORS
}

#define CCH_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr
PyMethodDef methods[] = {
    {"mx_quant", CCH_FAST(MxQuant)},
    {"dynamic_quant_i8", CCH_FAST(DynamicQuantI8)},
    {"moe_init_routing", CCH_FAST(MoeInitRouting)},
    {"w8a8_matmul_dequant", CCH_FAST(W8A8)},
    {"gmm_i8", CCH_FAST(GmmI8)},
    {"mx_matmul", CCH_FAST(MxMatmul)},
    {"mx_grouped_matmul", CCH_FAST(MxGroupedMatmul)},
    {"moe_ffn_mxfp8", CCH_FAST(MoeFfnMxfp8)},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_direct", "native form of the tensor-level entry points", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__direct() { return PyModule_Create(&module); }
