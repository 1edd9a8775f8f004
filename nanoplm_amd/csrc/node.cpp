// The differentiable calls of nanoplm_amd as native autograd nodes (Python module nanoplm_amd._node): plain, gated and
// LayerNorm-fused conv, forward and backward through the C ABI of libnplm_dwconv.so.
//
// What bounds a small training step is the host. As torch.autograd.Function the backward runs Python on the engine's
// thread, which first has to get the interpreter lock from the thread that waits for it; as torch.library custom ops (the
// pre-norm door's eager route before) both directions go through Python dispatch as well. Here neither direction runs Python.
// Forward + backward of one call after another, T=2048, 7 taps, bf16, before and now: plain, C=768 65 to 126 us (by how the threads
// meet at the lock) and 34 to 67 (by how soon the waiting thread and the engine's wake each other); gated 124 to 129 and 38 to 68; pre-norm
// 217 to 223 and 79 to 83. A multiplication by a constant takes 24 to 47. Inference, T=776, C=64, 3 taps 15.2 and 7.0; padded door, 32 x 512
// rows 23.9 and 15.8.
//
// A call that is not of the usual form - arguments that the checks below do not settle, tensor subclasses, modes, transforms,
// tracing, forward-mode AD - is answered with None, and the Python route takes it with its own messages. So nothing
// is accepted or refused here that it would treat otherwise.
//
// Replaces no reference code (peymanvahidi/nanoplm 0.1.6 has no convolution); the backward is what autograd runs at
// src/nanoplm/pretraining/pure_pipeline.py:739-742.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <climits>
#include <stdexcept>
#include <string>

#include "../../include/nplm_dwconv.h"

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<at::Tensor>;

// The library has no fused kernel for the call: the Python route composes it.
struct Unsupported : std::runtime_error {
    Unsupported() : std::runtime_error("no fused kernel for this call") {}
};

int dtype_code(const at::Tensor& t) {
    if (t.scalar_type() == at::kFloat) return NPLM_DWCONV_F32;
    if (t.scalar_type() == at::kBFloat16) return NPLM_DWCONV_BF16;
    return -1;
}
// Whether t's values are what lies at its data pointer, one after the other: not so for wrappers (of a batch, of another tensor), for a
// tensor known to be zero, and for a view that negates its values when they are read.
bool dense(const at::Tensor& t, const at::Device& dev) {
    return t.layout() == at::kStrided && t.device() == dev && !at::isTensorSubclassLike(t) && !t.is_neg() && !t._is_zerotensor() &&
           t.is_contiguous();
}
// a parameter of one value a channel, in w's dtype on its device
bool vector_as(const at::Tensor& t, const at::Tensor& w, int32_t C) {
    return dense(t, w.device()) && t.dim() == 1 && t.size(0) == C && t.scalar_type() == w.scalar_type();
}

struct Sizes {
    int64_t T;
    int32_t C, K, S, act, wdt;
};
// Sizes of a call on x [T, width * C], if everything about its tensors is as the kernels take it.
bool sizes_of(const at::Tensor& x, int width, const at::Tensor& cu, const at::Tensor& w, const OptTensor& b, Sizes* s) {
    if (!x.is_cuda() || x.dim() != 2 || w.dim() != 2 || cu.dim() != 1) return false;
    const at::Device dev = x.device();
    if (!dense(x, dev) || !dense(w, dev) || !dense(cu, dev) || cu.scalar_type() != at::kInt || cu.numel() < 1) return false;
    s->act = dtype_code(x);
    s->wdt = dtype_code(w);
    if (s->act < 0 || s->wdt < 0) return false;
    const int64_t C = x.size(1) / width, K = w.size(1);
    if (x.size(1) % width || w.size(0) != C || K % 2 == 0 || C > INT_MAX || K > INT_MAX || cu.numel() > INT_MAX) return false;
    if (b && !vector_as(*b, w, (int32_t)C)) return false;
    s->T = x.size(0);
    s->C = (int32_t)C;
    s->K = (int32_t)K;
    s->S = (int32_t)(cu.numel() - 1);
    return true;
}

const void* ptr(const OptTensor& t) { return t ? t->const_data_ptr() : nullptr; }
const int32_t* ints(const at::Tensor& t) { return t.const_data_ptr<int32_t>(); }
bool aligned16(const at::Tensor& t) { return (uintptr_t)t.const_data_ptr() % 16 == 0; }
void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
void check(int rc, const char* what) {
    if (rc == -NPLM_DWCONV_EUNSUPPORTED) throw Unsupported();
    if (rc != 0) throw std::runtime_error(std::string(what) + " failed with code " + std::to_string(rc) + ": " + nplm_dwconv_strerror(rc));
}
uint32_t flags_of(bool residual, bool grads_bf16) {
    return (residual ? NPLM_DWCONV_RESIDUAL : 0u) | (grads_bf16 ? NPLM_DWCONV_GRADS_BF16 : 0u);
}
at::Tensor scratch(size_t bytes, const at::Tensor& like) {
    return at::empty({(int64_t)(bytes > 256 ? bytes : 256)}, like.options().dtype(at::kByte));
}
// dy as the kernels take it
at::Tensor incoming(const at::Tensor& dy, const at::Tensor& x) {
    return dy.scalar_type() == x.scalar_type() ? dy.contiguous() : dy.to(x.scalar_type()).contiguous();
}
at::Tensor as(const at::Tensor& t, bool wanted, at::ScalarType dt) {
    return !wanted ? at::Tensor() : t.scalar_type() == dt ? t : t.to(dt);
}

// The Python route of a backward whose call turns out to be of another form (its result as a list of tensors).
template <typename... Args>
variable_list python_backward(const char* module, const char* name, Args&&... args) {
    pybind11::gil_scoped_acquire gil;
    pybind11::object out = pybind11::module_::import(module).attr(name)(std::forward<Args>(args)...);
    variable_list r;
    for (pybind11::handle h : out) r.push_back(h.is_none() ? at::Tensor() : h.cast<at::Tensor>());
    return r;
}

// Calls (and backwards) that something else records, rewrites or looks into go the Python way.
bool observed() {
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0 ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || torch::jit::tracer::isTracing() ||
           torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr;
}

// The tensors of a backward are what saved-tensor hooks gave back, which need not be what was saved, and a gradient of whatever kind its
// caller has: whether they are as the kernels take them. If not, the Python route makes them so, takes them apart or refuses them.
bool usual_backward(const at::Tensor& x, int width, const at::Tensor& cu, const at::Tensor& w, const at::Tensor& dy, Sizes* s) {
    return !observed() && x.defined() && cu.defined() && w.defined() && sizes_of(x, width, cu, w, std::nullopt, s) && dense(dy, x.device()) &&
           dy.dim() == 2 && dy.size(0) == s->T && dy.size(1) == s->C;
}

}  // namespace

// The nodes, by the names that profiles and autograd's messages give them; their calls are recorded there as the registered ops are.
namespace nanoplm_amd {
struct VarlenDWConv1d : torch::autograd::Function<VarlenDWConv1d> {
    static at::Tensor run(const at::Tensor& x, const at::Tensor& cu, const at::Tensor& w, const OptTensor& b, bool residual) {
        RECORD_FUNCTION("nanoplm_amd::varlen_dwconv_fwd", {});
        Sizes s;
        sizes_of(x, 1, cu, w, b, &s);
        const c10::DeviceGuard on(x.device());
        at::Tensor y = at::empty({s.T, s.C}, x.options());
        check(nplm_dwconv_fwd_ex(x.const_data_ptr(), ints(cu), w.const_data_ptr(), ptr(b), y.mutable_data_ptr(), s.T, s.C, s.K, s.S, s.act,
                                 s.wdt, flags_of(residual, false), stream_of(x)), "nplm_dwconv_fwd");
        return y;
    }
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& cu, const at::Tensor& w, const OptTensor& b,
                              bool residual) {
        ctx->save_for_backward({x, cu, w});
        ctx->saved_data["bias"] = b.has_value();
        ctx->saved_data["residual"] = residual;
        return run(x, cu, w, b, residual);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        RECORD_FUNCTION("nanoplm_amd::varlen_dwconv_bwd", {});
        const variable_list saved = ctx->get_saved_variables();
        const at::Tensor &x = saved[0], &cu = saved[1], &w = saved[2];
        const bool has_bias = ctx->saved_data["bias"].toBool(), residual = ctx->saved_data["residual"].toBool();
        const bool need_dx = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(2), need_b = has_bias && ctx->needs_input_grad(3);
        Sizes s;
        const c10::DeviceGuard on(x.device());
        const at::Tensor dy = incoming(grads[0], x);
        const bool bf16 = w.scalar_type() == at::kBFloat16;
        const at::ScalarType gdt = w.scalar_type();          // (fp32 or bf16: what the reduction kernel writes)
        at::Tensor dx, dw, db, ws;
        if (!usual_backward(x, 1, cu, w, dy, &s)) {
            using namespace pybind11::literals;
            pybind11::gil_scoped_acquire gil;
            const variable_list r = python_backward("nanoplm_amd.dwconv", "varlen_dwconv_bwd", x, dy, cu, w, "need_dx"_a = need_dx,
                                                    "need_dw"_a = need_w || need_b, "residual"_a = residual, "grads_bf16"_a = bf16);
            return {r[0], at::Tensor(), need_w ? r[1] : at::Tensor(), need_b ? r[2] : at::Tensor(), at::Tensor()};
        }
        if (need_dx) dx = at::empty({s.T, s.C}, x.options());
        size_t bytes = 0;
        if (need_w || need_b) {
            dw = at::empty({s.C, s.K}, x.options().dtype(gdt));
            db = at::empty({s.C}, x.options().dtype(gdt));
            bytes = nplm_dwconv_bwd_workspace_bytes(s.T, s.C, s.K, s.act);
            ws = scratch(bytes, x);
        }
        auto at_of = [](const at::Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; };
        check(nplm_dwconv_bwd_ex(x.const_data_ptr(), dy.const_data_ptr(), ints(cu), w.const_data_ptr(), at_of(dx), (float*)at_of(dw),
                                 (float*)at_of(db), at_of(ws), ws.defined() ? (size_t)ws.numel() : 0, s.T, s.C, s.K, s.S, s.act, s.wdt,
                                 flags_of(residual, bf16), stream_of(x)), "nplm_dwconv_bwd");
        return {dx, at::Tensor(), need_w ? dw : at::Tensor(), need_b ? db : at::Tensor(), at::Tensor()};
    }
};

struct GatedVarlenDWConv1d : torch::autograd::Function<GatedVarlenDWConv1d> {
    static at::Tensor run(const at::Tensor& z, const at::Tensor& cu, const at::Tensor& w, const OptTensor& b, bool residual) {
        RECORD_FUNCTION("nanoplm_amd::gated_dwconv_fwd", {});
        Sizes s;
        sizes_of(z, 2, cu, w, b, &s);
        const c10::DeviceGuard on(z.device());
        at::Tensor y = at::empty({s.T, s.C}, z.options());
        check(nplm_dwconv_gated_fwd(z.const_data_ptr(), ints(cu), w.const_data_ptr(), ptr(b), y.mutable_data_ptr(), s.T, s.C, s.K, s.S,
                                    s.act, s.wdt, flags_of(residual, false), stream_of(z)), "nplm_dwconv_gated_fwd");
        return y;
    }
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& z, const at::Tensor& cu, const at::Tensor& w, const OptTensor& b,
                              bool residual) {
        ctx->save_for_backward({z, cu, w});
        ctx->saved_data["bias"] = b.has_value();
        ctx->saved_data["residual"] = residual;
        return run(z, cu, w, b, residual);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        RECORD_FUNCTION("nanoplm_amd::gated_dwconv_bwd", {});
        const variable_list saved = ctx->get_saved_variables();
        const at::Tensor &z = saved[0], &cu = saved[1], &w = saved[2];
        const bool has_bias = ctx->saved_data["bias"].toBool(), residual = ctx->saved_data["residual"].toBool();
        Sizes s;
        const c10::DeviceGuard on(z.device());
        const at::Tensor dy = incoming(grads[0], z);
        const bool bf16 = w.scalar_type() == at::kBFloat16;
        const at::ScalarType gdt = w.scalar_type();
        const bool usual = usual_backward(z, 2, cu, w, dy, &s);
        const size_t bytes = usual ? nplm_dwconv_gated_bwd_workspace_bytes(s.T, s.C, s.K, s.act) : 0;
        at::Tensor dz, dw, db;
        int rc = -NPLM_DWCONV_EUNSUPPORTED;
        if (bytes > 0) {
            dz = at::empty({s.T, 2 * (int64_t)s.C}, z.options());
            dw = at::empty({s.C, s.K}, z.options().dtype(gdt));
            db = at::empty({s.C}, z.options().dtype(gdt));
            const at::Tensor ws = scratch(bytes, z);
            rc = nplm_dwconv_gated_bwd(z.const_data_ptr(), dy.const_data_ptr(), ints(cu), w.const_data_ptr(), dz.mutable_data_ptr(),
                                       (float*)dw.mutable_data_ptr(), (float*)db.mutable_data_ptr(), ws.mutable_data_ptr(),
                                       (size_t)ws.numel(), s.T, s.C, s.K, s.S, s.act, s.wdt, flags_of(residual, bf16), stream_of(z));
        }
        if (rc == -NPLM_DWCONV_EUNSUPPORTED) {
            using namespace pybind11::literals;
            pybind11::gil_scoped_acquire gil;
            const variable_list r = python_backward("nanoplm_amd.gated", "gated_dwconv_bwd", z, dy, cu, w, "residual"_a = residual, "grads_bf16"_a = bf16);
            dz = r[0], dw = r[1], db = r[2];
        } else {
            check(rc, "nplm_dwconv_gated_bwd");
        }
        return {ctx->needs_input_grad(0) ? dz : at::Tensor(), at::Tensor(), as(dw, ctx->needs_input_grad(2), gdt),
                as(db, has_bias && ctx->needs_input_grad(3), gdt), at::Tensor()};
    }
};

struct LnVarlenDWConv1d : torch::autograd::Function<LnVarlenDWConv1d> {
    // stats [T, 2] come back for the backward
    static at::Tensor run(const at::Tensor& x, const at::Tensor& cu, const at::Tensor& g, const OptTensor& beta, const at::Tensor& w,
                          const OptTensor& b, double eps, bool residual, at::Tensor* stats) {
        RECORD_FUNCTION("nanoplm_amd::ln_dwconv_fwd", {});
        Sizes s;
        sizes_of(x, 1, cu, w, b, &s);
        const c10::DeviceGuard on(x.device());
        at::Tensor y = at::empty({s.T, s.C}, x.options());
        *stats = at::empty({s.T, 2}, x.options().dtype(at::kFloat));
        check(nplm_dwconv_ln_fwd(x.const_data_ptr(), ints(cu), g.const_data_ptr(), ptr(beta), (float)eps, w.const_data_ptr(), ptr(b),
                                 y.mutable_data_ptr(), stats->mutable_data_ptr<float>(), s.T, s.C, s.K, s.S, s.act, s.wdt,
                                 flags_of(residual, false), stream_of(x)), "nplm_dwconv_ln_fwd");
        return y;
    }
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& cu, const at::Tensor& g, const OptTensor& beta,
                              const at::Tensor& w, const OptTensor& b, double eps, bool residual) {
        at::Tensor stats;
        at::Tensor y = run(x, cu, g, beta, w, b, eps, residual, &stats);
        ctx->save_for_backward({x, cu, g, beta ? *beta : at::Tensor(), w, stats});
        ctx->saved_data["bias"] = b.has_value();
        ctx->saved_data["residual"] = residual;
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        RECORD_FUNCTION("nanoplm_amd::ln_dwconv_bwd", {});
        const variable_list saved = ctx->get_saved_variables();
        const at::Tensor &x = saved[0], &cu = saved[1], &g = saved[2], &beta = saved[3], &w = saved[4], &stats = saved[5];
        const bool has_bias = ctx->saved_data["bias"].toBool(), residual = ctx->saved_data["residual"].toBool();
        Sizes s;
        const c10::DeviceGuard on(x.device());
        const at::Tensor dy = incoming(grads[0], x);
        const bool bf16 = w.scalar_type() == at::kBFloat16;
        const at::ScalarType gdt = w.scalar_type();
        const bool usual = usual_backward(x, 1, cu, w, dy, &s) && vector_as(g, w, s.C) && (!beta.defined() || vector_as(beta, w, s.C)) &&
                           dense(stats, x.device()) && stats.scalar_type() == at::kFloat && stats.dim() == 2 && stats.size(0) == s.T &&
                           stats.size(1) == 2;
        const size_t bytes = usual ? nplm_dwconv_ln_bwd_workspace_bytes(s.T, s.C, s.K, s.act) : 0;
        at::Tensor dx, dw, db, dg, dbeta;
        int rc = -NPLM_DWCONV_EUNSUPPORTED;
        // (under create_graph the op records itself, and says so if it is differentiated once more)
        if (bytes > 0 && !at::GradMode::is_enabled()) {
            const at::TensorOptions go = x.options().dtype(gdt);
            dx = at::empty({s.T, s.C}, x.options());
            dw = at::empty({s.C, s.K}, go);
            db = at::empty({s.C}, go);
            dg = at::empty({s.C}, go);
            if (beta.defined()) dbeta = at::empty({s.C}, go);
            const at::Tensor ws = scratch(bytes, x);
            rc = nplm_dwconv_ln_bwd(x.const_data_ptr(), dy.const_data_ptr(), ints(cu), stats.const_data_ptr<float>(), g.const_data_ptr(),
                                    beta.defined() ? beta.const_data_ptr() : nullptr, w.const_data_ptr(), dx.mutable_data_ptr(),
                                    (float*)dw.mutable_data_ptr(), (float*)db.mutable_data_ptr(), (float*)dg.mutable_data_ptr(),
                                    beta.defined() ? (float*)dbeta.mutable_data_ptr() : nullptr, ws.mutable_data_ptr(), (size_t)ws.numel(),
                                    s.T, s.C, s.K, s.S, s.act, s.wdt, flags_of(residual, bf16), stream_of(x));
        }
        if (rc == -NPLM_DWCONV_EUNSUPPORTED) {
            const OptTensor ob = beta.defined() ? OptTensor(beta) : OptTensor();
            const variable_list r = python_backward("nanoplm_amd.lnconv", "ln_dwconv_bwd_op", x, dy, cu, stats, g, ob, w, residual, bf16);
            dx = r[0], dg = r[1], dbeta = r[2], dw = r[3], db = r[4];
        } else {
            check(rc, "nplm_dwconv_ln_bwd");
        }
        return {dx, at::Tensor(), dg, beta.defined() ? dbeta : at::Tensor(), dw, has_bias ? db : at::Tensor(), at::Tensor(), at::Tensor()};
    }
};
}  // namespace nanoplm_amd

namespace {

bool tensor_arg(PyObject* o, at::Tensor* t) {
    if (!THPVariable_CheckExact(o)) return false;
    *t = THPVariable_Unpack(o);
    return true;
}
bool tensor_arg(PyObject* o, OptTensor* t) {
    if (o == Py_None) return true;
    if (!THPVariable_CheckExact(o)) return false;
    *t = THPVariable_Unpack(o);
    return true;
}
bool wants_grad(const OptTensor& t) { return t && t->requires_grad(); }

// (x or z, cu_seqlens, weight, bias or None, residual) -> y, or None
template <typename Node, int WIDTH>
PyObject* conv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 5, "5 arguments");
    at::Tensor x, cu, w, y;
    OptTensor b;
    Sizes s;
    if (observed() || !tensor_arg(a[0], &x) || !tensor_arg(a[1], &cu) || !tensor_arg(a[2], &w) || !tensor_arg(a[3], &b)) Py_RETURN_NONE;
    const int residual = PyObject_IsTrue(a[4]);
    if (residual < 0) return nullptr;
    if (!sizes_of(x, WIDTH, cu, w, b, &s)) Py_RETURN_NONE;
    // (asked first: a forward of the composed route would start with an allocation and an exception here, 4 us)
    if (WIDTH == 2 && (s.T == 0 || !aligned16(x) || nplm_dwconv_gated_bwd_workspace_bytes(s.T, s.C, s.K, s.act) == 0)) Py_RETURN_NONE;
    try {
        pybind11::gil_scoped_release no_gil;
        const bool grad = at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad() || wants_grad(b));
        y = grad ? Node::apply(x, cu, w, b, residual != 0) : Node::run(x, cu, w, b, residual != 0);
    } catch (const Unsupported&) {
        Py_RETURN_NONE;
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// (x, cu_seqlens, ln_weight, ln_bias or None, weight, bias or None, eps, residual) -> y, or None
PyObject* prenorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 8, "8 arguments");
    at::Tensor x, cu, g, w, y, stats;
    OptTensor beta, b;
    Sizes s;
    if (observed() || !tensor_arg(a[0], &x) || !tensor_arg(a[1], &cu) || !tensor_arg(a[2], &g) || !tensor_arg(a[3], &beta) ||
        !tensor_arg(a[4], &w) || !tensor_arg(a[5], &b)) Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(a[6]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    const int residual = PyObject_IsTrue(a[7]);
    if (residual < 0) return nullptr;
    if (!sizes_of(x, 1, cu, w, b, &s) || s.T == 0 || !aligned16(x)) Py_RETURN_NONE;
    for (const at::Tensor& t : {g, beta ? *beta : g})        // (one dtype for all parameters)
        if (!vector_as(t, w, s.C)) Py_RETURN_NONE;
    if (nplm_dwconv_ln_bwd_workspace_bytes(s.T, s.C, s.K, s.act) == 0) Py_RETURN_NONE;
    try {
        pybind11::gil_scoped_release no_gil;
        const bool grad = at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad() || g.requires_grad() || wants_grad(beta) || wants_grad(b));
        y = grad ? nanoplm_amd::LnVarlenDWConv1d::apply(x, cu, g, beta, w, b, eps, residual != 0) : nanoplm_amd::LnVarlenDWConv1d::run(x, cu, g, beta, w, b, eps, residual != 0, &stats);
    } catch (const Unsupported&) {
        Py_RETURN_NONE;
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"dwconv", (PyCFunction)(void (*)(void))&conv<nanoplm_amd::VarlenDWConv1d, 1>, METH_FASTCALL, "y = conv(x), differentiable; None: take the Python route"},
    {"gated_dwconv", (PyCFunction)(void (*)(void))&conv<nanoplm_amd::GatedVarlenDWConv1d, 2>, METH_FASTCALL, "y = conv(u * silu(g)), differentiable; None: take the Python route"},
    {"ln_dwconv", (PyCFunction)(void (*)(void))&prenorm, METH_FASTCALL, "y = conv(layer_norm(x)), differentiable; None: take the Python route"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_node", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__node() {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
