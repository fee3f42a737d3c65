// The host side of the public functions in C++: argument layout, allocation, autograd nodes and the calls into
// libfa_mi355.so, for the calls a program makes over and over.  It does what FlashAttentionFn and
// FlashAttentionQKVPackedFn of flash_attention.py do on the GPU, call by call the same, and declines (None)
// everything they are there for besides: whatever they reject, head dims that are no multiple of 8 and have to
// be padded, tensors off the GPU, tensor subclasses, tracing and transforms.
//
// Why: an autograd step through the Python classes and ctypes takes 160 - 250 us of host time (argument checks,
// two autograd.Function hops, ten allocations and their bookkeeping, filling the argument blocks field by field);
// problems whose kernels take less are bound by it.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/utils/pybind.h>

#include <cmath>
#include <optional>

#include "../../include/fa_mi355.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// (B, seq, H, D): unit head-dim stride, 16-byte aligned pointer and B, seq and H strides, a sequence stride the
// kernels' 32-bit offsets can hold
bool kernel_layout_ok(const Tensor& t) {
    if (t.stride(3) != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
    if (t.size(1) > 1 && !(t.stride(1) >= 0 && t.stride(1) < (1 << 23))) return false;
    for (int i = 0; i < 3; i++)
        if (t.size(i) != 1 && t.stride(i) % 8 != 0) return false;
    return true;
}
Tensor kernel_layout(const Tensor& t) { return kernel_layout_ok(t) ? t : t.contiguous(); }

int kernel_head_dim(int64_t d) { return d <= 16 ? 16 : d <= 32 ? 32 : d <= 64 ? 64 : d <= 128 ? 128 : 256; }

int bias_kind(const Tensor& b) {
    switch (b.scalar_type()) {
        case at::kBool: return FA_BIAS_BOOL;
        case at::kHalf: return FA_BIAS_F16;
        case at::kBFloat16: return FA_BIAS_BF16;
        case at::kFloat: return FA_BIAS_F32;
        default: return -1;
    }
}

int64_t padded_row(const Tensor& b) { return (b.size(3) * b.element_size() + 15) / 16 * 16; }  // bytes

// whether the C ABI, going by pointer and strides, fetches the rows of a 4-D bias in aligned 16-byte chunks
// (_bias_chunks_chosen in flash_attention.py)
bool bias_chunks_chosen(const Tensor& b) {
    const int64_t es = b.element_size(), n = b.size(3);
    if ((n > 1 && b.stride(3) != 1) || reinterpret_cast<uintptr_t>(b.data_ptr()) % 16 != 0) return false;
    for (int i = 0; i < 3; i++)
        if (b.size(i) > 1 && (b.stride(i) * es) % 16 != 0) return false;
    return n * es == padded_row(b) || b.stride(2) * es >= padded_row(b);
}

// ... and may: no chunk ends behind the storage (_bias_rows_ok)
bool bias_rows_ok(const Tensor& b) {
    if (b.size(2) == 1 || b.stride(2) == 0) return true;
    if (!bias_chunks_chosen(b)) return false;
    const int64_t es = b.element_size();
    if (b.size(3) * es == padded_row(b)) return true;
    int64_t last = b.storage_offset();
    for (int i = 0; i < 3; i++) last += (b.size(i) - 1) * b.stride(i);
    return last * es + padded_row(b) <= (int64_t)b.storage().nbytes();
}

// ... or 4 bytes at a time (_bias_dwords_ok), which pays where every (batch, head) pair has its own and no backward may follow
// (_bias_kernel_layout)
bool bias_dwords_ok(const Tensor& b, int D) {
    return b.scalar_type() == at::kFloat && D <= 64 && (b.size(3) == 1 || b.stride(3) == 1) && b.stride(2) >= 0 &&
           ((b.size(2) - 1) * b.stride(2) + b.size(3)) * 4 < (int64_t)1 << 31 && !bias_chunks_chosen(b);
}

// rows that start at multiples of 16 bytes, from 512 bytes on at whole cache lines (_empty_padded_rows in flash_attention.py)
Tensor empty_padded_rows(at::IntArrayRef shape, const at::TensorOptions& opt) {
    const int64_t es = (int64_t)opt.dtype().itemsize(), n = shape[3];
    const bool lines = n * es % 16 != 0 && n * es >= 512 && shape[2] * (n * es + 128) < (int64_t)1 << 31;
    const int64_t per = (lines ? 128 : 16) / es, n_pad = (n + per - 1) / per * per;
    if (n_pad == n) return at::empty(shape, opt);
    return at::empty({shape[0], shape[1], shape[2], n_pad}, opt).narrow(3, 0, n);
}

// what one call works on: q, k, v as given, the bias as a 4-D tensor whose rows the kernels can fetch
struct Call {
    Tensor q, k, v, bias, slopes;
    bool causal = false;
    double sm_scale = 1.;

    int64_t B() const { return q.size(0); }
    int64_t M() const { return q.size(1); }
    int64_t H() const { return q.size(2); }
    int64_t N() const { return k.size(1); }
    int d_qk() const { return (int)q.size(3); }
    int d_v() const { return (int)v.size(3); }
    fa_problem problem() const {
        const int kind = slopes.defined() ? FA_BIAS_ALIBI : bias.defined() ? bias_kind(bias) : FA_BIAS_NONE;
        return fa_problem{(int32_t)B(), (int32_t)H(), (int32_t)M(), (int32_t)N(), kernel_head_dim(std::max(d_qk(), d_v())),
                          q.scalar_type() == at::kHalf ? FA_F16 : FA_BF16, kind, causal ? 1 : 0, (float)sm_scale};
    }
};

void set_strides(int64_t (&dst)[4], const Tensor& t) {
    for (int i = 0; i < 4; i++) dst[i] = t.stride(i);
}
// strides of a bias (or its gradient) expanded to (B, H, M, N)
void set_bias_strides(int64_t (&dst)[4], const Tensor& b, const Call& c) {
    const int64_t want[4] = {c.B(), c.H(), c.M(), c.N()};
    for (int i = 0; i < 4; i++) dst[i] = b.size(i) == 1 && want[i] > 1 ? 0 : b.stride(i);
}
// NativeLibraryError, as _native.check raises it; from a node of the backward it reaches the caller as it is
void check(int status) {
    if (status == FA_OK) return;
    py::gil_scoped_acquire gil;
    const std::string text = "libfa_mi355: " + std::string(fa_strerror(status)) + " (status " + std::to_string(status) + ")";
    PyErr_SetString(py::module_::import("triton_flashattn_amd._native").attr("NativeLibraryError").ptr(), text.c_str());
    python_error error;
    error.persist();
    throw error;
}
void* current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor scratch(size_t bytes, const Tensor& like) {
    return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
}

std::pair<Tensor, Tensor> forward(const Call& c) {
    c10::DeviceGuard guard(c.q.device());
    const Tensor q = kernel_layout(c.q), k = kernel_layout(c.k), v = kernel_layout(c.v);
    Tensor o = at::empty({c.B(), c.M(), c.H(), c.d_v()}, q.options());
    Tensor lse = at::empty({c.B(), c.H(), c.M()}, q.options().dtype(at::kFloat));
    fa_fwd_args a{};
    a.p = c.problem();
    a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.o = o.data_ptr(); a.lse = lse.data_ptr<float>();
    set_strides(a.q_strides, q); set_strides(a.k_strides, k); set_strides(a.v_strides, v); set_strides(a.o_strides, o);
    if (c.slopes.defined()) {
        a.bias = c.slopes.data_ptr();
    } else if (c.bias.defined()) {
        a.bias = c.bias.data_ptr();
        set_bias_strides(a.bias_strides, c.bias, c);
    }
    Tensor workspace;  // (only touched by work enqueued on this stream: it may be dropped at once)
    if (const size_t bytes = fa_fwd_workspace_bytes(&a.p)) {
        workspace = scratch(bytes, q);
        a.workspace = workspace.data_ptr();
        a.workspace_bytes = bytes;
    }
    check(fa_fwd_dims(&a, c.d_qk(), c.d_v(), current_stream(q)));
    return {o, lse};
}

// dq undefined: not wanted; dk and dv both undefined: not wanted; dbias: undefined, of the bias's shape, or H slope
// gradients
void backward(const Call& c, const Tensor& dout, const Tensor& o, const Tensor& lse, const Tensor& dq, const Tensor& dk,
              const Tensor& dv, const Tensor& dbias) {
    c10::DeviceGuard guard(c.q.device());
    const Tensor q = kernel_layout(c.q), k = kernel_layout(c.k), v = kernel_layout(c.v), go = kernel_layout(dout);
    auto writable = [](const Tensor& t) { return !t.defined() || kernel_layout_ok(t) ? t : at::empty(t.sizes(), t.options()); };
    Tensor gq = writable(dq), gk = writable(dk), gv = writable(dv);
    int stages = FA_STAGE_PREP;
    if (gk.defined() || dbias.defined()) {
        stages |= FA_STAGE_MAIN;
        if (!gk.defined()) {
            gk = at::empty(k.sizes(), k.options());
            gv = at::empty(v.sizes(), v.options());
        }
    }
    if (gq.defined()) stages |= FA_STAGE_DQ;
    fa_bwd_args a{};
    a.p = c.problem();
    a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.o = o.data_ptr(); a.dout = go.data_ptr();
    a.lse = lse.data_ptr<float>();
    set_strides(a.q_strides, q); set_strides(a.k_strides, k); set_strides(a.v_strides, v); set_strides(a.o_strides, o);
    set_strides(a.do_strides, go);
    if (gq.defined()) {
        a.dq = gq.data_ptr();
        set_strides(a.dq_strides, gq);
    }
    if (gk.defined()) {
        a.dk = gk.data_ptr();
        a.dv = gv.data_ptr();
        set_strides(a.dk_strides, gk);
        set_strides(a.dv_strides, gv);
    }
    if (c.slopes.defined()) {
        a.bias = c.slopes.data_ptr();
        if (dbias.defined()) a.dbias = dbias.data_ptr();
    } else if (c.bias.defined()) {
        a.bias = c.bias.data_ptr();
        set_bias_strides(a.bias_strides, c.bias, c);
        if (dbias.defined()) {
            a.dbias = dbias.data_ptr();
            set_bias_strides(a.dbias_strides, dbias, c);
        }
    }
    const size_t bytes = fa_bwd_args_workspace_bytes(&a);
    const Tensor workspace = scratch(bytes, q);
    a.workspace = workspace.data_ptr();
    a.workspace_bytes = bytes;
    check(fa_bwd_stages_dims(&a, c.d_qk(), c.d_v(), current_stream(q), stages));
    if (dq.defined() && !gq.is_same(dq)) dq.copy_(gq);
    if (dk.defined() && !gk.is_same(dk)) dk.copy_(gk);
    if (dv.defined() && !gv.is_same(dv)) dv.copy_(gv);
}

Tensor bias_grad_like(const Call& c) {
    if (c.slopes.defined()) return at::empty_like(c.slopes);
    const int64_t full[4] = {c.B(), c.H(), c.M(), c.N()};
    if (c.bias.sizes() == at::IntArrayRef(full, 4)) return empty_padded_rows(c.bias.sizes(), c.bias.options());
    return at::empty(c.bias.sizes(), c.bias.options());
}

// the bias in the form the kernels read, next to the tensor that autograd knows
struct KernelBias {
    Tensor t;
};
using Maybe = std::optional<Tensor>;  // an absent argument has no edge in the graph
Maybe maybe(const Tensor& t) { return t.defined() ? Maybe(t) : std::nullopt; }

struct AttentionNode : torch::autograd::Function<AttentionNode> {
    // inputs: q, k, v, or one packed tensor with k and v undefined; bias or slopes or neither
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Maybe& k_, const Maybe& v_, const Maybe& bias,
                          const Maybe& slopes_, const KernelBias& bias4, bool causal, double sm_scale) {
        const Tensor k = k_.value_or(Tensor()), v = v_.value_or(Tensor()), slopes = slopes_.value_or(Tensor());
        auto [o, lse] = ::forward(make(q, k, v, bias4.t, slopes, causal, sm_scale));
        ctx->save_for_backward({q, k, v, o, lse, bias4.t, slopes});
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["sm_scale"] = sm_scale;
        if (bias) ctx->saved_data["bias_shape"] = bias->sizes().vec();
        return o;
    }
    static Call make(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& bias4, const Tensor& slopes, bool causal,
                     double sm_scale) {
        Call c;
        if (k.defined()) {
            c.q = q; c.k = k; c.v = v;
        } else {
            c.q = q.select(2, 0); c.k = q.select(2, 1); c.v = q.select(2, 2);
        }
        c.bias = bias4;
        if (slopes.defined()) c.slopes = slopes.contiguous();
        c.causal = causal;
        c.sm_scale = sm_scale;
        return c;
    }
    // A saved tensor is whatever the unpack hook of a program hands back: every extent the kernels use is taken from
    // q and k, so whatever else they read has to agree with them.
    static void check_saved(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& bias4,
                            const Tensor& slopes, const Tensor& dout) {
        const bool packed = !k.defined();
        const auto dev = dout.device();
        const auto dt = dout.scalar_type();
        for (const Tensor* t : {&q, &k, &v, &o, &lse, &bias4, &slopes})
            TORCH_CHECK_VALUE(!t->defined() || t->device() == dev, "flash_attention: all tensors must be on the same device");
        TORCH_CHECK_VALUE(dev.type() == c10::DeviceType::CUDA && (dt == at::kHalf || dt == at::kBFloat16) &&
                              (packed ? q.dim() == 5 && q.size(2) == 3 : q.dim() == 4 && k.dim() == 4 && v.dim() == 4),
                          "flash_attention: a saved tensor came back with another shape");
        const int64_t B = q.size(0), M = q.size(1), H = q.size(packed ? 3 : 2), d_qk = q.size(packed ? 4 : 3);
        const int64_t N = packed ? M : k.size(1), d_v = packed ? d_qk : v.size(3);
        auto expect = [&](const Tensor& t, const char* name, at::IntArrayRef shape, at::ScalarType type) {
            TORCH_CHECK_VALUE(t.sizes() == shape && t.scalar_type() == type, name, " has shape ", t.sizes(), " and type ",
                              t.scalar_type(), ", the kernels need ", shape, " and ", type);
        };
        expect(q, "q", packed ? at::IntArrayRef({B, M, 3, H, d_qk}) : at::IntArrayRef({B, M, H, d_qk}), dt);
        if (!packed) {
            expect(k, "k", {B, N, H, d_qk}, dt);
            expect(v, "v", {B, N, H, d_v}, dt);
        }
        expect(o, "o", {B, M, H, d_v}, dt);
        expect(dout, "do", {B, M, H, d_v}, dt);
        expect(lse, "lse", {B, H, M}, at::kFloat);
        TORCH_CHECK_VALUE(lse.is_contiguous(), "lse must be a dense float32 tensor of shape (B, H, M)");
        if (slopes.defined()) expect(slopes, "slopes", {H}, at::kFloat);
        if (bias4.defined()) {
            const int64_t want[4] = {B, H, M, N};
            bool fits = bias4.dim() == 4 && bias_kind(bias4) >= 0;
            for (int i = 0; fits && i < 4; i++) fits = bias4.size(i) == want[i] || bias4.size(i) == 1;
            TORCH_CHECK_VALUE(fits, "bias has shape ", bias4.sizes(), ", which does not broadcast to ", at::IntArrayRef(want, 4));
        }
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &lse = saved[4];
        check_saved(q, k, v, saved[3], lse, saved[5], saved[6], grads[0]);
        const Tensor o = kernel_layout(saved[3]);
        const Call c = make(q, k, v, saved[5], saved[6], ctx->saved_data["causal"].toBool(), ctx->saved_data["sm_scale"].toDouble());
        const bool packed = !k.defined();
        // (the edges that exist are numbered in the order of the arguments)
        int edge = 0;
        auto wanted = [&](bool present) { return present && ctx->needs_input_grad(edge++); };
        const bool need_q = wanted(true), need_k = wanted(!packed), need_v = wanted(!packed);
        const bool has_bias = ctx->saved_data.count("bias_shape") != 0;
        const bool need_bias = wanted(has_bias), need_slopes = wanted(c.slopes.defined());
        Tensor gq, gk, gv, dq, dk, dv, dbias;
        if (packed) {
            if (need_q) {
                gq = at::empty_like(q);
                dq = gq.select(2, 0); dk = gq.select(2, 1); dv = gq.select(2, 2);
            }
        } else {
            if (need_q) gq = dq = at::empty_like(q);
            if (need_k || need_v) {
                gk = dk = at::empty_like(k);
                gv = dv = at::empty_like(v);
            }
        }
        if (need_bias || need_slopes) dbias = bias_grad_like(c);
        if (dq.defined() || dk.defined() || dbias.defined()) ::backward(c, grads[0], o, lse, dq, dk, dv, dbias);
        Tensor gbias = need_bias ? dbias.view(ctx->saved_data["bias_shape"].toIntVector()) : Tensor();
        return {gq, need_k ? gk : Tensor(), need_v ? gv : Tensor(), gbias, need_slopes ? dbias : Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

bool has_tangent(const Tensor& t) {
    const auto* meta = torch::autograd::impl::get_autograd_meta(t);
    return meta && meta->fw_grad_ && !meta->fw_grad_->empty();
}
// a plain GPU tensor: not a subclass, no wrapper of a transform, no forward-mode tangent
bool plain(const Tensor& t, c10::Device dev) {
    using c10::DispatchKey;
    const auto keys = t.key_set();
    return t.device() == dev && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() &&
           !keys.has_any(c10::DispatchKeySet({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                              DispatchKey::Batched, DispatchKey::Functionalize})) &&
           !has_tangent(t);
}
std::optional<Tensor> unpack(PyObject* x) {
    if (x == Py_None) return Tensor();
    if (!THPVariable_CheckExact(x)) return std::nullopt;
    return THPVariable_Unpack(x);
}

// q, k, v (k and v None: q is a packed qkv), bias or None, slopes or None, causal, sm_scale or None -> out, or None where
// this is not a call for it
py::object attention(py::handle q_, py::handle k_, py::handle v_, py::handle bias_, py::handle slopes_, py::handle causal_, py::handle scale_) {
    auto uq = unpack(q_.ptr()), uk = unpack(k_.ptr()), uv = unpack(v_.ptr()), ub = unpack(bias_.ptr()), us = unpack(slopes_.ptr());
    if (!uq || !uk || !uv || !ub || !us || !uq->defined() || c10::impl::dispatch_mode_enabled()) return py::none();
    // a trace would not see the kernels; a transform is for the classes to refuse, whichever tensors it wraps
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return py::none();
    if (!PyBool_Check(causal_.ptr()) || !(scale_.is_none() || PyFloat_Check(scale_.ptr()))) return py::none();
    const Tensor q = *uq, k = *uk, v = *uv, bias = *ub, slopes = *us;
    const bool causal = causal_.ptr() == Py_True, packed = !k.defined();
    const c10::Device dev = q.device();
    if (dev.type() != c10::DeviceType::CUDA || k.defined() != v.defined() || (bias.defined() && slopes.defined())) return py::none();
    for (const Tensor* t : {&q, &k, &v, &bias, &slopes})
        if (t->defined() && !plain(*t, dev)) return py::none();
    const auto dt = q.scalar_type();
    if (dt != at::kHalf && dt != at::kBFloat16) return py::none();
    int64_t B, M, H, N, d_qk, d_v;
    if (packed) {
        if (q.dim() != 5 || q.size(2) != 3) return py::none();
        B = q.size(0); M = N = q.size(1); H = q.size(3); d_qk = d_v = q.size(4);
    } else {
        if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || k.scalar_type() != dt || v.scalar_type() != dt) return py::none();
        B = q.size(0); M = q.size(1); H = q.size(2); d_qk = q.size(3); N = k.size(1); d_v = v.size(3);
        if (k.size(0) != B || v.size(0) != B || k.size(2) != H || v.size(2) != H || v.size(1) != N || k.size(3) != d_qk) return py::none();
    }
    if (B < 1 || M < 1 || H < 1 || N < 1 || d_qk < 8 || d_v < 8 || (causal && M != N)) return py::none();
    // the library's own head dims, or whole 16-byte chunks below one of them up to 128
    const int D = kernel_head_dim(std::max(d_qk, d_v));
    const bool full = d_qk == D && d_v == D;
    if (!full && (D > 128 || d_qk % 8 != 0 || d_v % 8 != 0)) return py::none();
    Tensor bias4;
    if (bias.defined()) {
        if (bias.dim() > 4 || bias_kind(bias) < 0) return py::none();
        const int64_t want[4] = {B, H, M, N};
        int64_t shape[4] = {1, 1, 1, 1};
        for (int i = 0; i < bias.dim(); i++) shape[4 - bias.dim() + i] = bias.size(i);
        for (int i = 0; i < 4; i++)
            if (shape[i] != want[i] && shape[i] != 1) return py::none();
        if (bias.requires_grad()) {
            if (shape[3] != N) return py::none();
            const bool shared = (shape[0] != B || shape[1] != H) && shape[2] != 1;
            if (shared && !full) return py::none();  // that gradient's kernel takes full head dims only
        }
    }
    if (slopes.defined() && (slopes.dim() != 1 || slopes.size(0) != H || slopes.scalar_type() != at::kFloat)) return py::none();
    const double sm_scale = scale_.is_none() ? std::pow((double)d_qk, -0.5) : PyFloat_AsDouble(scale_.ptr());

    const bool grad = at::GradMode::is_enabled() &&
                      (q.requires_grad() || (k.defined() && (k.requires_grad() || v.requires_grad())) ||
                       (bias.defined() && bias.requires_grad()) || (slopes.defined() && slopes.requires_grad()));

    py::gil_scoped_release no_gil;
    Tensor out;
    {
        // (views and copies of the bias have no edges; but a view shares the version of the tensor it is taken from, so
        // that the backward notices when that has been written to in the meantime)
        at::AutoGradMode no_grad(false);
        if (bias.defined()) {
            bias4 = bias;
            if (bias.dim() < 4) {
                int64_t shape[4] = {1, 1, 1, 1};
                for (int i = 0; i < bias.dim(); i++) shape[4 - bias.dim() + i] = bias.size(i);
                bias4 = bias.reshape(at::IntArrayRef(shape, 4));
            }
            if (!bias_rows_ok(bias4) && (grad || bias4.size(0) * bias4.size(1) != B * H || !bias_dwords_ok(bias4, D))) {
                Tensor padded = empty_padded_rows(bias4.sizes(), bias4.options());
                padded.copy_(bias4);
                bias4 = padded;
            }
        }
    }
    if (grad) {
        out = AttentionNode::apply(q, maybe(k), maybe(v), maybe(bias), maybe(slopes), KernelBias{bias4}, causal, sm_scale);
    } else {
        at::AutoDispatchBelowADInplaceOrView below;
        out = forward(AttentionNode::make(q, k, v, bias4, slopes, causal, sm_scale)).first;
    }
    py::gil_scoped_acquire gil;
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(std::move(out)));
}

}  // namespace

PYBIND11_MODULE(_torch_host, m) {
    m.doc() = "C++ host path of triton_flashattn_amd";
    m.def("attention", &attention);
}
