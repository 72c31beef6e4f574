// Host side of the kernel-level entry points: tensors in, checks, output and workspace tensors, strides and the call
// of the C ABI, without the interpreter in between.  Forward + backward of B=2 H=2 L=16 D=32 in a loop, where the host
// time is what counts: 55 us through Python and ctypes, 14 us here.
//
// The functions serve well-formed calls on plain GPU tensors only and return None for everything else (wrong shapes
// or types, wrappers of functorch or of tensor subclasses, host tensors, empty problems): the caller in kernels.py
// then goes through its general form, which raises the errors.  They return the status of the C ABI when it is not 0.
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <climits>
#include <cmath>

#include "../../include/sjvp.h"

namespace {

using at::Tensor;

struct Abi {
    decltype(&sjvp_fwd) fwd = nullptr;
    decltype(&sjvp_fwd_rotary) fwd_rotary = nullptr;
    decltype(&sjvp_bwd_parts) bwd_parts = nullptr;
    decltype(&sjvp_bwd_rotary) bwd_rotary = nullptr;
    decltype(&sjvp_bwd_workspace_bytes) workspace_bytes = nullptr;
    decltype(&sjvp_cast) cast = nullptr;
    decltype(&sjvp_adaln_fwd) adaln_fwd = nullptr;
    decltype(&sjvp_adaln_bwd) adaln_bwd = nullptr;
    decltype(&sjvp_adaln_workspace_floats) adaln_workspace_floats = nullptr;
    decltype(&sjvp_gelu) gelu = nullptr;
    decltype(&sjvp_rope) rope = nullptr;
};
Abi abi;  // filled once by bind() when the library is loaded

struct Shape {
    int64_t B, H, Lq, Lk, D;
    at::ScalarType dtype;
    c10::Device device;
    int tag;  // element type of the C ABI
    int64_t stat_rows() const { return (Lq + 127) / 128 * 128; }
};

// A tensor that owns plain device memory: no functorch wrapper, no subclass, no zero or lazily conjugated tensor.
const Tensor* plain(PyObject* obj) {
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const Tensor& t = THPVariable_Unpack(obj);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
    const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
    constexpr c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::ZeroTensor,
                                           c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                           c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched,
                                           c10::DispatchKey::Functionalize});
    if (impl->has_symbolic_sizes_strides() || impl->key_set().has_any(special)) return nullptr;
    return &t;
}

// obj as a [B,H,L,D] operand of the call, or nullptr
const Tensor* operand(PyObject* obj, const Shape& s, int64_t L) {
    const Tensor* t = plain(obj);
    if (!t || t->dim() != 4 || t->scalar_type() != s.dtype || t->device() != s.device || t->stride(3) != 1 ||
        t->size(0) != s.B || t->size(1) != s.H || t->size(2) != L || t->size(3) != s.D)
        return nullptr;
    return t;
}

// obj as a row statistic: contiguous fp32 [B,H,Lr]
const Tensor* statistic(PyObject* obj, const Shape& s) {
    const Tensor* t = plain(obj);
    if (!t || t->dim() != 3 || t->scalar_type() != at::kFloat || t->device() != s.device || t->size(0) != s.B ||
        t->size(1) != s.H || t->size(2) != s.stat_rows() || !t->is_contiguous())
        return nullptr;
    return t;
}

bool shape_of(PyObject* q_obj, PyObject* k_obj, PyObject* arithmetic, Shape& s) {
    const Tensor* q = plain(q_obj);
    const Tensor* k = plain(k_obj);
    if (!q || !k || q->dim() != 4 || k->dim() != 4) return false;
    s.B = q->size(0), s.H = q->size(1), s.Lq = q->size(2), s.D = q->size(3), s.Lk = k->size(2);
    s.dtype = q->scalar_type();
    s.device = q->device();
    const bool fold = arithmetic != Py_None;
    if (fold && !(PyUnicode_Check(arithmetic) && PyUnicode_CompareWithASCIIString(arithmetic, "bf16") == 0)) return false;
    switch (s.dtype) {
        case at::kBFloat16: s.tag = SJVP_BF16; break;
        case at::kHalf: s.tag = SJVP_FP16; break;
        case at::kFloat: s.tag = fold ? SJVP_FP32_BF16 : SJVP_FP32; break;
        default: return false;
    }
    return s.D >= 16 && s.D <= 128 && s.B > 0 && s.H > 0 && s.Lq > 0 && s.Lk > 0 && s.B <= INT_MAX && s.H <= INT_MAX &&
           s.Lq <= INT_MAX && s.Lk <= INT_MAX;
}

// The softmax scale as the C ABI spells it (0: the default); negative for a value that the caller has to refuse.
float scale_arg(PyObject* obj) {
    if (obj == Py_None) return 0.0f;
    if (!PyFloat_CheckExact(obj)) return -1.0f;
    const double v = PyFloat_AS_DOUBLE(obj);
    return v > 0.0 && std::isfinite(v) ? static_cast<float>(v) : -1.0f;
}

struct Tables {
    const float *cos = nullptr, *sin = nullptr;
    int64_t stride = 0;
    int rows = 0;
};

bool tables(PyObject* cos_obj, PyObject* sin_obj, const Shape& s, Tables& out) {
    const Tensor* cos = plain(cos_obj);
    const Tensor* sin = plain(sin_obj);
    if (!cos || !sin || cos->dim() != 2 || sin->dim() != 2) return false;
    for (const Tensor* t : {cos, sin})
        if (t->scalar_type() != at::kFloat || t->device() != s.device || t->size(1) != 32 || t->stride(1) != 1 ||
            t->size(0) < std::max(s.Lq, s.Lk) || t->size(0) > INT_MAX)
            return false;
    if (cos->size(0) != sin->size(0) || cos->stride(0) != sin->stride(0)) return false;
    out = {cos->const_data_ptr<float>(), sin->const_data_ptr<float>(), cos->stride(0), static_cast<int>(cos->size(0))};
    return true;
}

void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

void put_strides(int64_t* out, const Tensor* t) {
    for (int d = 0; d < 3; ++d) out[d] = t ? t->stride(d) : 0;
}

PyObject* none() { Py_RETURN_NONE; }

// Uninitialised tensors for the results of a call, on the device of a call: straight from torch's allocator,
// without the dispatcher's round trips, of which a forward + backward of ten results and a workspace makes eleven (B=2 H=2 L=16
// D=32 in a loop 15.9 us of host time with them, 14.0 without).  Where a dispatch mode watches or memory has to be filled, they go the usual way.
struct Maker {
    c10::Device device;
    bool direct = !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
                  !(at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());

    Tensor operator()(at::IntArrayRef sizes, at::ScalarType dtype) const {
        if (!direct) return at::empty(sizes, at::TensorOptions().dtype(dtype).device(device));
        return Tensor(at::detail::empty_cuda(sizes, dtype, device, std::nullopt));
    }
    // like at::empty_like: the strides of a tensor without gaps and overlaps are kept
    Tensor like(const Tensor& t) const {
        if (!direct || !t.is_non_overlapping_and_dense()) return at::empty_like(t);
        return Tensor(at::detail::empty_strided_cuda(t.sizes(), t.strides(), t.scalar_type(), device));
    }
};

// forward(q, k, v, tq, tk, tv, o, to, lse, mu, li, with_li, scale, arithmetic, cos, sin) -> (o, to, lse, mu, li);
// an output that is None is allocated; with_li None: without tangents (tq, tk, tv, to, mu, li are None)
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 16 || !abi.fwd) return none();
    Shape s{.device = c10::Device(c10::kCPU)};
    if (!shape_of(a[0], a[1], a[13], s)) return none();
    const bool jvp = a[11] != Py_None;
    if (jvp && a[11] != Py_True && a[11] != Py_False) return none();
    const Tensor* in[6] = {};
    for (int i = 0; i < (jvp ? 6 : 3); ++i)
        if (!(in[i] = operand(a[i], s, i % 3 ? s.Lk : s.Lq))) return none();
    Tensor made[5];
    const Tensor* out[5] = {};  // o, to, lse, mu, li
    bool make[5] = {};
    for (int i = 0; i < 5; ++i) {
        const bool wanted = i == 0 || i == 2 || (jvp && (i != 4 || a[11] == Py_True || a[10] != Py_None));
        if (!wanted) continue;
        if (a[6 + i] == Py_None) make[i] = true;
        else if (!(out[i] = i < 2 ? operand(a[6 + i], s, s.Lq) : statistic(a[6 + i], s))) return none();
    }
    const float scale = scale_arg(a[12]);
    if (scale < 0.0f) return none();
    const bool rotary = a[14] != Py_None;
    Tables rope;
    if (rotary && !tables(a[14], a[15], s, rope)) return none();
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(s.device);
        const Maker make_tensor{s.device};
        for (int i = 0; i < 5; ++i) {
            if (!make[i]) continue;
            made[i] = i < 2 ? make_tensor({s.B, s.H, s.Lq, s.D}, s.dtype) : make_tensor({s.B, s.H, s.stat_rows()}, at::kFloat);
            out[i] = &made[i];
        }
        int64_t strides[SJVP_F_COUNT * 3];
        for (int i = 0; i < 6; ++i) put_strides(strides + 3 * i, in[i]);
        for (int i = 0; i < 2; ++i) put_strides(strides + 3 * (SJVP_F_O + i), out[i]);
        void* stream = c10::hip::getCurrentHIPStream(s.device.index()).stream();
        auto* lse = static_cast<float*>(ptr(out[2]));
        auto* mu = static_cast<float*>(ptr(out[3]));
        auto* li = static_cast<float*>(ptr(out[4]));
        const int B = s.B, H = s.H, Lq = s.Lq, Lk = s.Lk, D = s.D;
        rc = rotary ? abi.fwd_rotary(ptr(in[0]), ptr(in[1]), ptr(in[2]), ptr(in[3]), ptr(in[4]), ptr(in[5]), ptr(out[0]),
                                     ptr(out[1]), lse, mu, li, B, H, Lq, Lk, D, strides, scale, s.tag, rope.cos, rope.sin,
                                     rope.stride, rope.rows, stream)
                    : abi.fwd(ptr(in[0]), ptr(in[1]), ptr(in[2]), ptr(in[3]), ptr(in[4]), ptr(in[5]), ptr(out[0]),
                              ptr(out[1]), lse, mu, li, B, H, Lq, Lk, D, strides, scale, s.tag, stream);
    }
    if (rc != SJVP_OK) return PyLong_FromLong(rc);
    PyObject* res = PyTuple_New(5);
    if (!res) return nullptr;
    for (int i = 0; i < 5; ++i) {
        PyObject* item;
        if (make[i]) {
            item = THPVariable_Wrap(std::move(made[i]));
        } else {
            item = out[i] ? a[6 + i] : Py_None;
            Py_INCREF(item);
        }
        if (!item) {
            Py_DECREF(res);
            return nullptr;
        }
        PyTuple_SET_ITEM(res, i, item);
    }
    return res;
    END_HANDLE_TH_ERRORS
}

// backward(q, k, v, tq, tk, tv, o, to, lse, mu, dO, dTO, scale, grads, workspace, parts, arithmetic, cos, sin)
// -> (dq, dk, dv, dtq, dtk, dtv)
PyObject* backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 19 || !abi.bwd_parts) return none();
    Shape s{.device = c10::Device(c10::kCPU)};
    if (!shape_of(a[0], a[1], a[16], s)) return none();
    const bool has_do = a[10] != Py_None, has_g = a[11] != Py_None;
    if (!has_do && !has_g) return none();
    // q, k, v, tq, tk, tv, o, to, dO, dTO, dq, dk, dv, dtq, dtk, dtv as the stride table of the C ABI orders them
    const Tensor* t[SJVP_B_COUNT] = {};
    for (int i = 0; i < (has_g ? 6 : 3); ++i)
        if (!(t[i] = operand(a[i], s, i % 3 ? s.Lk : s.Lq))) return none();
    if (!(t[SJVP_B_O] = operand(a[6], s, s.Lq))) return none();
    if (has_g && !(t[SJVP_B_TO] = operand(a[7], s, s.Lq))) return none();
    if (has_do && !(t[SJVP_B_DO] = operand(a[10], s, s.Lq))) return none();
    if (has_g && !(t[SJVP_B_DTO] = operand(a[11], s, s.Lq))) return none();
    const Tensor* lse = statistic(a[8], s);
    const Tensor* mu = has_g ? statistic(a[9], s) : nullptr;
    if (!lse || (has_g && !mu)) return none();
    const int n_grads = has_g ? 6 : 3;
    const bool given = a[13] != Py_None;
    if (given) {
        if (!PyTuple_CheckExact(a[13]) || PyTuple_GET_SIZE(a[13]) != 6) return none();
        for (int i = 0; i < n_grads; ++i)
            if (!(t[SJVP_B_DQ + i] = operand(PyTuple_GET_ITEM(a[13], i), s, i % 3 ? s.Lk : s.Lq))) return none();
    }
    const float scale = scale_arg(a[12]);
    if (scale < 0.0f || !PyLong_CheckExact(a[15])) return none();
    const long parts = PyLong_AsLong(a[15]);
    if (parts < 0 || parts > INT_MAX) {
        PyErr_Clear();
        return none();
    }
    const bool rotary = a[17] != Py_None;
    Tables rope;
    if (rotary && (a[14] != Py_None || parts != SJVP_BWD_ALL || !tables(a[17], a[18], s, rope))) return none();
    const size_t bytes = rotary ? 0 : abi.workspace_bytes(s.B, s.H, s.Lq, s.Lk, s.D, s.tag);
    const Tensor* workspace = nullptr;
    if (a[14] != Py_None) {
        workspace = plain(a[14]);
        if (!workspace || workspace->scalar_type() != at::kByte || workspace->device() != s.device ||
            static_cast<size_t>(workspace->numel()) < bytes)
            return none();
    }
    Tensor made[6], scratch;
    bool dense = true;
    int rc = SJVP_OK;
    {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(s.device);
        const Maker make_tensor{s.device};
        if (!given)
            for (int i = 0; i < n_grads; ++i) {
                made[i] = make_tensor.like(*t[i]);
                t[SJVP_B_DQ + i] = &made[i];
                dense = dense && made[i].stride(3) == 1;  // not so for some inputs that overlap themselves
            }
        if (dense) {
            if (!rotary && !workspace) {
                scratch = make_tensor({static_cast<int64_t>(bytes)}, at::kByte);
                workspace = &scratch;
            }
            int64_t strides[SJVP_B_COUNT * 3];
            void* p[SJVP_B_COUNT];
            for (int i = 0; i < SJVP_B_COUNT; ++i) {
                put_strides(strides + 3 * i, t[i]);
                p[i] = ptr(t[i]);
            }
            void* stream = c10::hip::getCurrentHIPStream(s.device.index()).stream();
            auto* l = static_cast<const float*>(ptr(lse));
            auto* m = static_cast<const float*>(ptr(mu));
            const int B = s.B, H = s.H, Lq = s.Lq, Lk = s.Lk, D = s.D;
            rc = rotary ? abi.bwd_rotary(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], l, m, p[10], p[11],
                                         p[12], p[13], p[14], p[15], B, H, Lq, Lk, D, strides, scale, s.tag, rope.cos,
                                         rope.sin, rope.stride, rope.rows, stream)
                        : abi.bwd_parts(static_cast<int>(parts), p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8],
                                        p[9], l, m, p[10], p[11], p[12], p[13], p[14], p[15], ptr(workspace), bytes, B, H,
                                        Lq, Lk, D, strides, scale, s.tag, stream);
        }
    }
    if (!dense) return none();
    if (rc != SJVP_OK) return PyLong_FromLong(rc);
    PyObject* res = PyTuple_New(6);
    if (!res) return nullptr;
    for (int i = 0; i < 6; ++i) {
        PyObject* item = Py_None;
        if (i < n_grads && !given) {
            item = THPVariable_Wrap(std::move(made[i]));
        } else {
            if (i < n_grads) item = PyTuple_GET_ITEM(a[13], i);
            Py_INCREF(item);
        }
        if (!item) {
            Py_DECREF(res);
            return nullptr;
        }
        PyTuple_SET_ITEM(res, i, item);
    }
    return res;
    END_HANDLE_TH_ERRORS
}

// A copy as part of the graph of the tensor it was cast from: one node for each, so that a tensor that needs no gradient
// has none and one that does gets it as soon as it is there.
struct CastNode : torch::autograd::Function<CastNode> {
    static constexpr bool is_traceable = true;
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& from, Tensor* copy) {
        ctx->saved_data["type"] = static_cast<int64_t>(from.scalar_type());
        return std::move(*copy);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto type = static_cast<at::ScalarType>(ctx->saved_data["type"].toInt());
        return {grads[0].defined() ? grads[0].to(type) : Tensor(), Tensor()};
    }
};

// cast(list of tensors or None, dtype, recorded) -> list; a tensor that has the dtype is handed back itself, the others, dense
// and between fp32 and one 16-bit type, are copied in as few launches as it takes.  Autograd sees it only where `recorded`.
PyObject* cast(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || n > 3 || !abi.cast || !PyList_CheckExact(a[0]) || !THPDtype_Check(a[1])) return none();
    const bool recorded = n == 3 && a[2] == Py_True && at::GradMode::is_enabled();
    const at::ScalarType to = reinterpret_cast<THPDtype*>(a[1])->scalar_type;
    constexpr int kMost = 64;
    const Py_ssize_t count = PyList_GET_SIZE(a[0]);
    if (count > kMost) return none();
    auto tag = [](at::ScalarType t) { return t == at::kFloat ? SJVP_FP32 : t == at::kBFloat16 ? SJVP_BF16 : t == at::kHalf ? SJVP_FP16 : -1; };
    const Tensor* in[kMost] = {};
    at::ScalarType from = to;
    const Tensor* some = nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* obj = PyList_GET_ITEM(a[0], i);
        if (obj == Py_None) continue;
        const Tensor* t = plain(obj);
        if (!t) return none();
        if (t->scalar_type() == to) continue;
        if (!some) some = t, from = t->scalar_type();
        if (t->scalar_type() != from || t->device() != some->device() || !t->is_non_overlapping_and_dense()) return none();
        in[i] = t;
    }
    if (some && (tag(from) < 0 || tag(to) < 0 || (from == at::kFloat) == (to == at::kFloat))) return none();
    Tensor made[kMost];
    int rc = SJVP_OK;
    if (some) {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(some->device());
        void* stream = c10::hip::getCurrentHIPStream(some->device().index()).stream();
        const void* x[SJVP_CAST_MAX];
        void* y[SJVP_CAST_MAX];
        int64_t numel[SJVP_CAST_MAX];
        int k = 0;
        for (Py_ssize_t i = 0; i < count && rc == SJVP_OK; ++i) {
            if (in[i]) {
                made[i] = at::empty_like(*in[i], in[i]->options().dtype(to));
                x[k] = in[i]->const_data_ptr();
                y[k] = made[i].mutable_data_ptr();
                numel[k++] = in[i]->numel();
            }
            if (k == SJVP_CAST_MAX || (k && i + 1 == count)) {
                rc = abi.cast(k, x, y, numel, tag(from), tag(to), stream);
                k = 0;
            }
        }
    }
    if (rc != SJVP_OK) return PyLong_FromLong(rc);
    for (Py_ssize_t i = 0; i < count; ++i)
        if (recorded && in[i] && in[i]->requires_grad()) made[i] = CastNode::apply(*in[i], &made[i]);
    PyObject* res = PyList_New(count);
    if (!res) return nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* item;
        if (in[i]) {
            item = THPVariable_Wrap(std::move(made[i]));
        } else {
            item = PyList_GET_ITEM(a[0], i);
            Py_INCREF(item);
        }
        if (!item) {
            Py_DECREF(res);
            return nullptr;
        }
        PyList_SET_ITEM(res, i, item);
    }
    return res;
    END_HANDLE_TH_ERRORS
}

// rope(sequence of one to four [B,S,H,D] tensors, cos, sin, dtype of the results or None, inverse) -> tuple of contiguous
// [B,S,H,D] tensors; cos and sin None: no rotation
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5 || !abi.rope || !PyTuple_CheckExact(a[0]) || (a[3] != Py_None && !THPDtype_Check(a[3]))) return none();
    if (a[4] != Py_True && a[4] != Py_False) return none();
    constexpr int kMost = 4;
    const Py_ssize_t count = PyTuple_GET_SIZE(a[0]);
    if (count < 1 || count > kMost) return none();
    const Tensor* x[kMost];
    for (Py_ssize_t i = 0; i < count; ++i) {
        x[i] = plain(PyTuple_GET_ITEM(a[0], i));
        if (!x[i] || x[i]->dim() != 4 || x[i]->sizes() != x[0]->sizes() || x[i]->scalar_type() != x[0]->scalar_type() ||
            x[i]->device() != x[0]->device() || x[i]->stride(3) != 1)
            return none();
    }
    auto tag = [](at::ScalarType t) { return t == at::kFloat ? SJVP_FP32 : t == at::kBFloat16 ? SJVP_BF16 : t == at::kHalf ? SJVP_FP16 : -1; };
    const at::ScalarType from = x[0]->scalar_type(), to = a[3] == Py_None ? from : reinterpret_cast<THPDtype*>(a[3])->scalar_type;
    const int64_t B = x[0]->size(0), S = x[0]->size(1), H = x[0]->size(2), D = x[0]->size(3);
    if (tag(from) < 0 || tag(to) < 0 || B < 1 || S < 1 || H < 1 || D < 1 || B > INT_MAX || S > INT_MAX || H > INT_MAX || D > INT_MAX)
        return none();
    const Tensor *cos = nullptr, *sin = nullptr;
    if (a[1] != Py_None || a[2] != Py_None) {
        cos = plain(a[1]);
        sin = plain(a[2]);
        if (!cos || !sin || cos->dim() != 2 || cos->sizes() != sin->sizes() || cos->size(0) < S || 2 * cos->size(1) > D ||
            cos->stride(0) != sin->stride(0))
            return none();
        for (const Tensor* t : {cos, sin})
            if (t->scalar_type() != at::kFloat || t->device() != x[0]->device() || t->stride(1) != 1) return none();
    }
    Tensor made[kMost];
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(x[0]->device());
        const Maker make_tensor{x[0]->device()};
        const void* in[kMost];
        void* out[kMost];
        int64_t strides[6 * kMost];  // of [B,H,S,D], inputs and results in turn
        for (Py_ssize_t i = 0; i < count; ++i) {
            made[i] = make_tensor({B, S, H, D}, to);
            in[i] = x[i]->const_data_ptr();
            out[i] = made[i].mutable_data_ptr();
            int64_t* at = strides + 6 * i;
            for (const Tensor* t : {x[i], static_cast<const Tensor*>(&made[i])}) {
                *at++ = t->stride(0);
                *at++ = t->stride(2);
                *at++ = t->stride(1);
            }
        }
        rc = abi.rope(static_cast<int>(count), in, out, strides, cos ? cos->const_data_ptr<float>() : nullptr,
                      sin ? sin->const_data_ptr<float>() : nullptr, cos ? cos->stride(0) : 0, static_cast<int>(B),
                      static_cast<int>(H), static_cast<int>(S), static_cast<int>(D), cos ? static_cast<int>(2 * cos->size(1)) : 0,
                      tag(from), tag(to), a[4] == Py_True, c10::hip::getCurrentHIPStream(x[0]->device().index()).stream());
    }
    if (rc != SJVP_OK) return PyLong_FromLong(rc);
    PyObject* res = PyTuple_New(count);
    if (!res) return nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* item = THPVariable_Wrap(std::move(made[i]));
        if (!item) {
            Py_DECREF(res);
            return nullptr;
        }
        PyTuple_SET_ITEM(res, i, item);
    }
    return res;
    END_HANDLE_TH_ERRORS
}

// The pointer members of sjvp_adaln by the names of the tensors they take.
struct AdaField {
    const char* name;
    void** (*at)(sjvp_adaln&);
    int mod;  // place in mod_stride, or -1
};
#define SJVP_ADA(name, mod) {#name, [](sjvp_adaln& t) { return reinterpret_cast<void**>(const_cast<void*>(static_cast<const void*>(&t.name))); }, mod}
const AdaField ada_fields[] = {
    SJVP_ADA(x, -1), SJVP_ADA(tx, -1), SJVP_ADA(a, -1), SJVP_ADA(ta, -1), SJVP_ADA(gate, 0), SJVP_ADA(tgate, 1),
    SJVP_ADA(scale, 2), SJVP_ADA(tscale, 3), SJVP_ADA(shift, 4), SJVP_ADA(tshift, 5), SJVP_ADA(w, -1), SJVP_ADA(b, -1),
    SJVP_ADA(y, -1), SJVP_ADA(ty, -1), SJVP_ADA(h, -1), SJVP_ADA(th, -1), SJVP_ADA(dy, -1), SJVP_ADA(dty, -1),
    SJVP_ADA(dh, -1), SJVP_ADA(dth, -1), SJVP_ADA(dx, -1), SJVP_ADA(dtx, -1), SJVP_ADA(da, -1), SJVP_ADA(dta, -1),
    SJVP_ADA(dgate, -1), SJVP_ADA(dtgate, -1), SJVP_ADA(dscale, -1), SJVP_ADA(dtscale, -1), SJVP_ADA(dshift, -1),
    SJVP_ADA(dtshift, -1), SJVP_ADA(dw, -1), SJVP_ADA(db, -1)};
#undef SJVP_ADA
constexpr int kAdaFields = sizeof(ada_fields) / sizeof(ada_fields[0]);
PyObject* ada_names[kAdaFields];  // interned, made by bind()

// adaln(reverse, jvp, B, S, W, eps, {name: tensor or None}) -> status; the caller has laid the tensors out and keeps them
PyObject* adaln(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 7 || !abi.adaln_fwd || !PyDict_CheckExact(a[6])) return none();
    sjvp_adaln t{};
    t.B = static_cast<int>(PyLong_AsLong(a[2]));
    t.S = static_cast<int>(PyLong_AsLong(a[3]));
    t.W = static_cast<int>(PyLong_AsLong(a[4]));
    t.eps = static_cast<float>(PyFloat_AsDouble(a[5]));
    if (PyErr_Occurred()) return nullptr;
    const Tensor* x = nullptr;
    for (int i = 0; i < kAdaFields; ++i) {
        PyObject* obj = PyDict_GetItem(a[6], ada_names[i]);
        if (!obj || obj == Py_None) continue;
        const Tensor* z = plain(obj);
        if (!z || (x && z->device() != x->device())) return none();
        if (!x) x = z;
        *ada_fields[i].at(t) = z->data_ptr();
        if (ada_fields[i].mod >= 0) t.mod_stride[ada_fields[i].mod] = z->stride(0);
    }
    if (!x || !t.x) return none();
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(x->device());
        void* stream = c10::hip::getCurrentHIPStream(x->device().index()).stream();
        if (a[0] == Py_True) {
            const Tensor workspace = Maker{x->device()}({static_cast<int64_t>(abi.adaln_workspace_floats(&t))}, at::kFloat);
            t.workspace = workspace.data_ptr<float>();
            rc = abi.adaln_bwd(&t, a[1] == Py_True, stream);
        } else {
            rc = abi.adaln_fwd(&t, a[1] == Py_True, stream);
        }
    }
    return PyLong_FromLong(rc);
    END_HANDLE_TH_ERRORS
}

// gelu(u, tu, dy, dty, y, ty, reverse) -> status; the tensors may be None but for u
PyObject* gelu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 7 || !abi.gelu) return none();
    const Tensor* t[6] = {};
    for (int i = 0; i < 6; ++i)
        if (a[i] != Py_None && (!(t[i] = plain(a[i])) || !t[0] || t[i]->device() != t[0]->device())) return none();
    const long reverse = PyLong_AsLong(a[6]);
    if (PyErr_Occurred()) return nullptr;
    if (!t[0]) return none();
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        const c10::DeviceGuard guard(t[0]->device());
        rc = abi.gelu(ptr(t[0]), ptr(t[1]), ptr(t[2]), ptr(t[3]), ptr(t[4]), ptr(t[5]), t[0]->numel(), static_cast<int>(reverse),
                      c10::hip::getCurrentHIPStream(t[0]->device().index()).stream());
    }
    return PyLong_FromLong(rc);
    END_HANDLE_TH_ERRORS
}

// bind(addresses of the entry points, in the order of Abi)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    constexpr int kEntries = 11;
    if (n != kEntries) {
        PyErr_SetString(PyExc_TypeError, "bind() takes eleven addresses");
        return nullptr;
    }
    void* p[kEntries];
    for (int i = 0; i < kEntries; ++i) {
        p[i] = PyLong_AsVoidPtr(a[i]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind(): null address");
            return nullptr;
        }
    }
    for (int i = 0; i < kAdaFields; ++i)
        if (!ada_names[i] && !(ada_names[i] = PyUnicode_InternFromString(ada_fields[i].name))) return nullptr;
    abi = {reinterpret_cast<decltype(abi.fwd)>(p[0]),
           reinterpret_cast<decltype(abi.fwd_rotary)>(p[1]),
           reinterpret_cast<decltype(abi.bwd_parts)>(p[2]),
           reinterpret_cast<decltype(abi.bwd_rotary)>(p[3]),
           reinterpret_cast<decltype(abi.workspace_bytes)>(p[4]),
           reinterpret_cast<decltype(abi.cast)>(p[5]),
           reinterpret_cast<decltype(abi.adaln_fwd)>(p[6]),
           reinterpret_cast<decltype(abi.adaln_bwd)>(p[7]),
           reinterpret_cast<decltype(abi.adaln_workspace_floats)>(p[8]),
           reinterpret_cast<decltype(abi.gelu)>(p[9]),
           reinterpret_cast<decltype(abi.rope)>(p[10])};
    return none();
}

#ifndef SJVP_BUILD_ID
#define SJVP_BUILD_ID "SJVP_BUILD_ID=unknown"
#endif
const char build_id[] = SJVP_BUILD_ID;

PyMethodDef methods[] = {
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(forward)), METH_FASTCALL, nullptr},
    {"backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(backward)), METH_FASTCALL, nullptr},
    {"cast", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(cast)), METH_FASTCALL, nullptr},
    {"adaln", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(adaln)), METH_FASTCALL, nullptr},
    {"gelu", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gelu)), METH_FASTCALL, nullptr},
    {"rope", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rope)), METH_FASTCALL, nullptr},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sjvp_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sjvp_host() {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "build_id", build_id) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
