// The plain calls of the Python modules in native code: argument checks, output
// allocation and the launches of one public call in one extension call.
//
// Issued from Python through ctypes, a call costs 9 to 50 us of interpreter
// time (shape tests, torch.empty, stream lookups, argument conversion) for 4
// to 30 us of kernels: the M = 1 weight product took 14.2 us for an 8.3 us
// kernel, a small MXFP4Linear forward 48 us for 30.  Every function here
// takes the arguments of its Python caller and handles the form that programs
// pass in a loop -- exact torch tensors on one GPU, the layouts the kernels
// read in place -- and returns None for anything else (other strides,
// alignments, types, empty shapes, wrong arguments, tensor subclasses,
// functorch wrappers, calls under a dispatch mode or a functorch transform):
// the caller then runs its general path, which converts,
// or raises as it always has.  The launches go through the same C ABI
// (include/lsmx.h), on torch's current stream, with the GIL released.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/lsmx.h"

namespace {

using at::Tensor;

PyObject *g_error = nullptr;      // _capi.check(rc): raises LsmxError
PyObject *g_workspace = nullptr;  // _capi.workspace(device, nbytes)
PyObject *g_epoch = nullptr;      // _capi.next_epoch()

// A dispatch mode or a functorch transform around the call: at::empty gives
// that mode's tensors, which may have no data pointer.
bool transformed() {
    return c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// A plain GPU tensor: exactly torch.Tensor (or Parameter), with storage, and no
// dispatch key that changes what its data means.
const Tensor *plain(PyObject *o) {
    if (!THPVariable_CheckExact(o) || transformed()) return nullptr;
    const Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
    constexpr c10::DispatchKeySet odd{c10::DispatchKey::Python, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                      c10::DispatchKey::ZeroTensor, c10::DispatchKey::FuncTorchBatched,
                                      c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize};
    return t.key_set().has_any(odd) ? nullptr : &t;
}

bool al(const Tensor &t, uintptr_t a) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % a == 0; }

// rows of a 2-D tensor with unit stride and 16-byte aligned starts
bool rows16(const Tensor &t) {
    return t.dim() == 2 && t.stride(1) == 1 && al(t, 16) && t.stride(0) >= t.size(1) &&
           (t.stride(0) * t.element_size()) % 16 == 0;
}

int dtype_of(at::ScalarType s) {
    return s == at::kFloat ? LSMX_F32 : s == at::kBFloat16 ? LSMX_BF16 : s == at::kHalf ? LSMX_F16 : -1;
}

// scalar type of a torch.dtype argument, or Undefined (None included: only
// weight()'s callers give it a meaning)
at::ScalarType out_type(PyObject *o) {
    if (!THPDtype_Check(o)) return at::ScalarType::Undefined;
    const at::ScalarType s = reinterpret_cast<THPDtype *>(o)->scalar_type;
    return dtype_of(s) >= 0 ? s : at::ScalarType::Undefined;
}

Tensor make(at::IntArrayRef shape, at::ScalarType s, const Tensor &like) {
    return at::empty(shape, at::TensorOptions().dtype(s).device(like.device()));
}
void *stream_of(const Tensor &t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// Holds the GIL released; takes it back when a C++ exception leaves the scope
// too, so that HANDLE_TH_ERRORS sets the Python error with it held.
struct NoGil {
    PyThreadState *s = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(s); }
};

// Runs launches with the GIL released; returns false with a Python error set
// (LsmxError through _capi.check) if one fails.
template <typename F>
bool launch(F &&f) {
    int rc;
    {
        NoGil released;
        rc = f();
    }
    if (rc == LSMX_OK) return true;
    PyObject *r = PyObject_CallFunction(g_error, "i", rc);
    Py_XDECREF(r);
    return false;
}

PyObject *wrap2(const Tensor &a, const Tensor &b) {
    PyObject *t = PyTuple_New(2);
    if (!t) return nullptr;
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
    return t;
}

#define NONE_IF(c) \
    if (c) Py_RETURN_NONE

// ---------------------------------------------------------------- quantizers
// what the row quantizer reads in place: fp32 / bf16 / fp16 rows, K % 32 == 0
bool quant_rows(const Tensor *x, int64_t kmult) {
    return x && rows16(*x) && dtype_of(x->scalar_type()) >= 0 && x->size(0) > 0 && x->size(1) > 0 &&
           x->size(1) % kmult == 0;
}

struct Quantized {
    Tensor codes, scale;
};
Quantized packed_out(const Tensor &x, bool km) {
    const int64_t R = x.size(0), K = x.size(1);
    return {make({R, K / 2}, at::kByte, x), km ? make({K / 128, R, 4}, at::kByte, x) : make({R, K / 32}, at::kByte, x)};
}
int quant_launch(const Tensor &x, const Quantized &q, bool km, void *s) {
    const int64_t R = x.size(0), K = x.size(1);
    return lsmx_quantize_mxfp4(x.data_ptr(), dtype_of(x.scalar_type()), R, K, R > 1 ? x.stride(0) : K, 32,
                               q.codes.data_ptr(), LSMX_CODES_PACKED, K / 2, q.scale.data_ptr(),
                               km ? LSMX_SCALE_E8M0_KMAJOR : LSMX_SCALE_E8M0, km ? R : K / 32, s);
}
// two tensors: one launch when they share a dtype
int quant2_launch(const Tensor &x, const Quantized &qx, const Tensor &w, const Quantized &qw, bool km, void *s) {
    if (x.scalar_type() != w.scalar_type()) {
        const int rc = quant_launch(x, qx, km, s);
        return rc == LSMX_OK ? quant_launch(w, qw, km, s) : rc;
    }
    lsmx_q_item it[2];
    const Tensor *ts[2] = {&x, &w};
    const Quantized *qs[2] = {&qx, &qw};
    for (int i = 0; i < 2; ++i) {
        const int64_t R = ts[i]->size(0), K = ts[i]->size(1);
        it[i] = lsmx_q_item{ts[i]->data_ptr(),       R,     K,
                            R > 1 ? ts[i]->stride(0) : K, qs[i]->codes.data_ptr(), K / 2,
                            qs[i]->scale.data_ptr(), km ? R : K / 32};
    }
    return lsmx_quantize_mxfp4_batch(it, 2, dtype_of(x.scalar_type()), km ? LSMX_SCALE_E8M0_KMAJOR : LSMX_SCALE_E8M0, s);
}

// quantize_pack(x, kmajor) -> (packed, e8m0)
PyObject *quantize_pack(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 2);
    const bool km = a[1] == Py_True;
    const Tensor *x = plain(a[0]);
    NONE_IF(!quant_rows(x, km ? 128 : 32));
    const Quantized q = packed_out(*x, km);
    void *s = stream_of(*x);
    if (!launch([&] { return quant_launch(*x, q, km, s); })) return nullptr;
    return wrap2(q.codes, q.scale);
    END_HANDLE_TH_ERRORS
}

// quantize_pack2([x, w], kmajor) -> [(packed, e8m0), (packed, e8m0)]
PyObject *quantize_pack2(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 2 || !PyList_CheckExact(a[0]) || PyList_GET_SIZE(a[0]) != 2);
    const bool km = a[1] == Py_True;
    const Tensor *x = plain(PyList_GET_ITEM(a[0], 0)), *w = plain(PyList_GET_ITEM(a[0], 1));
    NONE_IF(!quant_rows(x, km ? 128 : 32) || !quant_rows(w, km ? 128 : 32) || x->scalar_type() != w->scalar_type() ||
            x->device() != w->device());
    const Quantized qx = packed_out(*x, km), qw = packed_out(*w, km);
    void *s = stream_of(*x);
    if (!launch([&] { return quant2_launch(*x, qx, *w, qw, km, s); })) return nullptr;
    PyObject *l = PyList_New(2);
    if (!l) return nullptr;
    PyList_SET_ITEM(l, 0, wrap2(qx.codes, qx.scale));
    PyList_SET_ITEM(l, 1, wrap2(qw.codes, qw.scale));
    return l;
    END_HANDLE_TH_ERRORS
}

// quantize(x) -> (codes, fp32 scale): fp4.quantize_mxfp4 with 32-blocks
PyObject *quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 1);
    const Tensor *x = plain(a[0]);
    NONE_IF(!quant_rows(x, 32));
    const int64_t R = x->size(0), K = x->size(1);
    const Tensor codes = make({R, K}, at::kByte, *x), scale = make({R, K / 32}, at::kFloat, *x);
    void *s = stream_of(*x);
    if (!launch([&] {
            return lsmx_quantize_mxfp4(x->data_ptr(), dtype_of(x->scalar_type()), R, K, R > 1 ? x->stride(0) : K, 32,
                                       codes.data_ptr(), LSMX_CODES_UNPACKED, K, scale.data_ptr(), LSMX_SCALE_F32,
                                       K / 32, s);
        }))
        return nullptr;
    return wrap2(codes, scale);
    END_HANDLE_TH_ERRORS
}

// quantize_2d(x) -> (row_packed, row_scale, col_packed, col_scale), K-major
PyObject *quantize_2d(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 1);
    const Tensor *x = plain(a[0]);
    NONE_IF(!quant_rows(x, 128) || x->size(0) % 128 || x->scalar_type() == at::kFloat);
    const int64_t R = x->size(0), K = x->size(1);
    const Tensor rp = make({R, K / 2}, at::kByte, *x), rs = make({K / 128, R, 4}, at::kByte, *x);
    const Tensor cp = make({K, R / 2}, at::kByte, *x), cs = make({R / 128, K, 4}, at::kByte, *x);
    void *s = stream_of(*x);
    if (!launch([&] {
            return lsmx_quantize_mxfp4_2d(x->data_ptr(), dtype_of(x->scalar_type()), R, K, x->stride(0),
                                          rp.data_ptr<uint8_t>(), K / 2, rs.data_ptr<uint8_t>(), R,
                                          cp.data_ptr<uint8_t>(), R / 2, cs.data_ptr<uint8_t>(), K,
                                          LSMX_SCALE_E8M0_KMAJOR, s);
        }))
        return nullptr;
    PyObject *t = PyTuple_New(4);
    if (!t) return nullptr;
    const Tensor *o[4] = {&rp, &rs, &cp, &cs};
    for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(t, i, THPVariable_Wrap(*o[i]));
    return t;
    END_HANDLE_TH_ERRORS
}

// pack(codes) -> packed
PyObject *pack(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 1);
    const Tensor *c = plain(a[0]);
    NONE_IF(!c || c->scalar_type() != at::kByte || c->dim() != 2 || !c->is_contiguous() || c->size(1) % 2 ||
            c->numel() == 0 || !al(*c, 16));
    const Tensor out = make({c->size(0), c->size(1) / 2}, at::kByte, *c);
    void *s = stream_of(*c);
    if (!launch([&] { return lsmx_pack_fp4(c->data_ptr<uint8_t>(), out.data_ptr<uint8_t>(), out.numel(), s); }))
        return nullptr;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------ f4 x f4 GEMM
int gemm_km(const Tensor &a, const Tensor &as, const Tensor &b, const Tensor &bs, const Tensor &c, int64_t K, void *s) {
    const int64_t M = a.size(0), N = b.size(0);
    return lsmx_gemm_f4f4(a.data_ptr<uint8_t>(), M > 1 ? a.stride(0) : K / 2, as.data_ptr(), M, b.data_ptr<uint8_t>(),
                          N > 1 ? b.stride(0) : K / 2, bs.data_ptr(), N, LSMX_SCALE_E8M0_KMAJOR, c.data_ptr(),
                          dtype_of(c.scalar_type()), N, M, N, K, s);
}

// fp32 block scales of the two operands -> K-major E8M0 in one launch, with the
// flag that lsmx_gemm_mx_promote tests unless the caller knows them exact
struct ScaleConv {
    Tensor a, b, flag;
    uint64_t epoch = 0;
    lsmx_e8m0_item it[2];
};
bool scales_f32(const Tensor *s, int64_t r, int64_t c) {
    return s && s->scalar_type() == at::kFloat && s->dim() == 2 && s->size(0) == r && s->size(1) == c &&
           s->stride(1) == 1 && s->stride(0) >= c;
}
bool conv_prepare(ScaleConv &v, const Tensor &sa, int64_t M, const Tensor &sb, bool sb_t, int64_t N, int64_t K,
                  bool flagged) {
    v.a = make({K / 128, M, 4}, at::kByte, sa);
    v.b = make({K / 128, N, 4}, at::kByte, sa);
    const Tensor *ss[2] = {&sa, &sb};
    for (int i = 0; i < 2; ++i) {
        const Tensor &s = *ss[i];
        v.it[i] = lsmx_e8m0_item{s.data_ptr<float>(), s.size(0), s.size(1), s.size(0) > 1 ? s.stride(0) : s.size(1),
                                 i == 1 && sb_t ? LSMX_E8M0_IN_T : 0, (i ? v.b : v.a).data_ptr<uint8_t>(), i ? N : M};
    }
    if (flagged) {
        v.flag = make({1}, at::kLong, sa);
        PyObject *e = PyObject_CallNoArgs(g_epoch);
        if (!e) return false;
        v.epoch = PyLong_AsUnsignedLongLong(e);
        Py_DECREF(e);
        if (PyErr_Occurred()) return false;
    }
    return true;
}
uint64_t *flag_of(const ScaleConv &v) { return v.flag.defined() ? reinterpret_cast<uint64_t *>(v.flag.data_ptr()) : nullptr; }
int conv_launch(const ScaleConv &v, void *s) { return lsmx_scale_to_e8m0_batch(v.it, 2, flag_of(v), v.epoch, s); }

// gemm_packed(a_pk, bt_pk, a_scale, b_scale, out_dtype, exact)
PyObject *gemm_packed(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 6);
    const Tensor *ap = plain(a[0]), *bp = plain(a[1]), *as = plain(a[2]), *bs = plain(a[3]);
    const at::ScalarType ot = out_type(a[4]);
    NONE_IF(!ap || !bp || !as || !bs || ot == at::ScalarType::Undefined || ap->scalar_type() != at::kByte ||
            bp->scalar_type() != at::kByte || !rows16(*ap) || !rows16(*bp) || ap->size(1) != bp->size(1));
    const int64_t M = ap->size(0), N = bp->size(0), K = 2 * ap->size(1);
    NONE_IF(M == 0 || N == 0 || K == 0 || K % 128 || bp->device() != ap->device() || as->device() != ap->device() ||
            bs->device() != ap->device() || as->scalar_type() != bs->scalar_type());
    if (as->scalar_type() == at::kByte) {
        for (int i = 0; i < 2; ++i) {
            const Tensor &s = i ? *bs : *as;
            NONE_IF(s.dim() != 3 || s.size(0) != K / 128 || s.size(1) != (i ? N : M) || s.size(2) != 4 ||
                    !s.is_contiguous());
        }
        const Tensor c = make({M, N}, ot, *ap);
        void *s = stream_of(c);
        if (!launch([&] { return gemm_km(*ap, *as, *bp, *bs, c, K, s); })) return nullptr;
        return THPVariable_Wrap(c);
    }
    NONE_IF(!scales_f32(as, M, K / 32) || !scales_f32(bs, N, K / 32));
    const bool flagged = a[5] != Py_True;
    const Tensor c = make({M, N}, ot, *ap);
    void *s = stream_of(c);
    ScaleConv v;
    if (!conv_prepare(v, *as, M, *bs, false, N, K, flagged)) return nullptr;
    if (!launch([&] {
            int rc = conv_launch(v, s);
            if (rc == LSMX_OK) rc = gemm_km(*ap, v.a, *bp, v.b, c, K, s);
            if (rc == LSMX_OK && flagged)
                rc = lsmx_gemm_mx_promote(ap->data_ptr<uint8_t>(), M > 1 ? ap->stride(0) : K / 2, as->data_ptr<float>(),
                                          M > 1 ? as->stride(0) : K / 32, 1, bp->data_ptr<uint8_t>(),
                                          N > 1 ? bp->stride(0) : K / 2, bs->data_ptr<float>(),
                                          N > 1 ? bs->stride(0) : K / 32, 1, LSMX_CODES_PACKED, c.data_ptr(),
                                          dtype_of(ot), N, M, N, K, flag_of(v), v.epoch, s);
            return rc;
        }))
        return nullptr;
    return THPVariable_Wrap(c);
    END_HANDLE_TH_ERRORS
}

// linear(x, w, out_dtype): quantize both operands along K and multiply, the
// forward of MXFP4Linear
PyObject *linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 3);
    const Tensor *x = plain(a[0]), *w = plain(a[1]);
    const at::ScalarType ot = out_type(a[2]);
    NONE_IF(ot == at::ScalarType::Undefined || !quant_rows(x, 128) || !quant_rows(w, 128) || x->size(1) != w->size(1) ||
            x->device() != w->device());
    const int64_t K = x->size(1);
    const Quantized qx = packed_out(*x, true), qw = packed_out(*w, true);
    const Tensor c = make({x->size(0), w->size(0)}, ot, *x);
    void *s = stream_of(c);
    if (!launch([&] {
            const int rc = quant2_launch(*x, qx, *w, qw, true, s);
            return rc == LSMX_OK ? gemm_km(qx.codes, qx.scale, qw.codes, qw.scale, c, K, s) : rc;
        }))
        return nullptr;
    return THPVariable_Wrap(c);
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------- weight-only GEMMs
// weight(a0, a1 or None, w_pk, w_scale, out_dtype or None): a0 @ deq(W)^T (and
// a1 @ deq(W)^T); E8M0 weight scales
PyObject *weight(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 5);
    const Tensor *a0 = plain(a[0]), *w = plain(a[2]), *ws = plain(a[3]);
    const bool dual = a[1] != Py_None;
    const Tensor *a1 = dual ? plain(a[1]) : nullptr;
    NONE_IF(!a0 || !w || !ws || (dual && !a1) || !rows16(*a0) || !rows16(*w) || dtype_of(a0->scalar_type()) < 0 ||
            w->scalar_type() != at::kByte || ws->scalar_type() != at::kByte);
    const at::ScalarType at_ = a0->scalar_type(), ot = a[4] == Py_None ? at_ : out_type(a[4]);
    const int64_t M = a0->size(0), K = a0->size(1), N = w->size(0);
    NONE_IF(ot == at::ScalarType::Undefined || M == 0 || N == 0 || K == 0 || K % 128 || 2 * w->size(1) != K ||
            w->device() != a0->device() || ws->device() != a0->device());
    NONE_IF(ws->dim() != 2 || ws->size(0) != N || ws->size(1) != K / 32 || ws->stride(1) != 1 ||
            ws->stride(0) < K / 32 || (N > 1 && ws->stride(0) % 4) || !al(*ws, 4));
    NONE_IF(dual && (at_ != at::kBFloat16 || a1->scalar_type() != at_ || !rows16(*a1) || a1->size(0) != M ||
                     a1->size(1) != K || a1->stride(0) != a0->stride(0) || a1->device() != a0->device()));
    const int64_t lda = M > 1 ? a0->stride(0) : K, ldw = N > 1 ? w->stride(0) : K / 2, lds = N > 1 ? ws->stride(0) : K / 32;
    const Tensor c0 = make({M, N}, ot, *a0), c1 = dual ? make({M, N}, ot, *a0) : Tensor();
    void *s = stream_of(c0);
    if (at_ == at::kBFloat16) {
        const int64_t nws = lsmx_gemm_bf16f4_slices(M, N, K) > 1 ? lsmx_gemm_bf16f4_workspace(M, N, K, dual) : 0;
        void *wsp = nullptr;
        PyObject *keep = nullptr;
        if (nws > 0) {   // the split-K workspace of this device and stream
            PyObject *dev = PyObject_GetAttrString(a[0], "device");
            if (!dev) return nullptr;
            keep = PyObject_CallFunction(g_workspace, "OL", dev, (long long)nws);
            Py_DECREF(dev);
            if (!keep) return nullptr;
            wsp = THPVariable_Unpack(keep).data_ptr();
        }
        const bool ok = launch([&] {
            return lsmx_gemm_bf16f4_ws(a0->data_ptr(), dual ? a1->data_ptr() : nullptr, lda, w->data_ptr<uint8_t>(), ldw,
                                       ws->data_ptr(), lds, LSMX_SCALE_E8M0, c0.data_ptr(),
                                       dual ? c1.data_ptr() : nullptr, dtype_of(ot), N, M, N, K, wsp, nws, s);
        });
        Py_XDECREF(keep);
        if (!ok) return nullptr;
    } else if (!launch([&] {
                   return lsmx_gemm_wonly_f4(a0->data_ptr(), dtype_of(at_), lda, w->data_ptr<uint8_t>(), ldw,
                                             ws->data_ptr(), lds, LSMX_SCALE_E8M0, c0.data_ptr(), dtype_of(ot), N, M, N,
                                             K, s);
               })) {
        return nullptr;
    }
    return dual ? wrap2(c0, c1) : THPVariable_Wrap(c0);
    END_HANDLE_TH_ERRORS
}

// -------------------------------------------------------------- E4M3 GEMM
// gemm_fp8(a_fp8, b_fp8, a_scale, b_scale, out_dtype, exact): B [K, N] with N
// contiguous, fp32 scales
PyObject *gemm_fp8(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    NONE_IF(n != 6);
    const Tensor *x = plain(a[0]), *b = plain(a[1]), *as = plain(a[2]), *bs = plain(a[3]);
    const at::ScalarType ot = out_type(a[4]);
    auto bytes = [](const Tensor &t) { return t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kByte; };
    NONE_IF(!x || !b || !as || !bs || ot == at::ScalarType::Undefined || !bytes(*x) || !bytes(*b) || !rows16(*x) ||
            !rows16(*b) || x->size(1) != b->size(0));
    const int64_t M = x->size(0), K = x->size(1), N = b->size(1);
    NONE_IF(M == 0 || N == 0 || K == 0 || K % 128 || N % 16 || b->stride(0) >= 0x7FFFFFFF / 256 ||
            b->device() != x->device() || as->device() != x->device() || bs->device() != x->device() ||
            !scales_f32(as, M, K / 32) || !scales_f32(bs, K / 32, N));
    const bool flagged = a[5] != Py_True;
    const Tensor c = make({M, N}, ot, *x);
    void *s = stream_of(c);
    ScaleConv v;
    if (!conv_prepare(v, *as, M, *bs, true, N, K, flagged)) return nullptr;
    const uint8_t *xp = reinterpret_cast<const uint8_t *>(x->data_ptr()), *bp = reinterpret_cast<const uint8_t *>(b->data_ptr());
    const int64_t lda = M > 1 ? x->stride(0) : K, ldb = b->stride(0);
    if (!launch([&] {
            int rc = conv_launch(v, s);
            if (rc == LSMX_OK)
                rc = lsmx_gemm_f8f8_nb(xp, lda, v.a.data_ptr<uint8_t>(), M, bp, ldb, v.b.data_ptr<uint8_t>(), N,
                                       c.data_ptr(), dtype_of(ot), N, M, N, K, s);
            if (rc == LSMX_OK && flagged)
                rc = lsmx_gemm_mx_promote(xp, lda, as->data_ptr<float>(), M > 1 ? as->stride(0) : K / 32, 1, bp, ldb,
                                          bs->data_ptr<float>(), 1, K / 32 > 1 ? bs->stride(0) : N,
                                          LSMX_E4M3 | LSMX_B_NCONTIG, c.data_ptr(), dtype_of(ot), N, M, N, K,
                                          flag_of(v), v.epoch, s);
            return rc;
        }))
        return nullptr;
    return THPVariable_Wrap(c);
    END_HANDLE_TH_ERRORS
}

// init(check, workspace, next_epoch): the _capi functions the calls above use
PyObject *init(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "init(check, workspace, next_epoch)");
        return nullptr;
    }
    PyObject **g[3] = {&g_error, &g_workspace, &g_epoch};
    for (int i = 0; i < 3; ++i) {
        Py_INCREF(a[i]);
        Py_XDECREF(*g[i]);
        *g[i] = a[i];
    }
    Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(init),   FAST(quantize_pack), FAST(quantize_pack2), FAST(quantize), FAST(quantize_2d), FAST(pack),
                         FAST(gemm_packed), FAST(linear), FAST(weight), FAST(gemm_fp8), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast() { return PyModule_Create(&module); }
