// Shared host-side glue of the two PyTorch extension modules: argument checks,
// element-type mapping, the current HIP stream, scratch from the caching
// allocator, and status -> exception.  No kernels here; everything goes
// through the C ABI of libteletron_norm.so.
#pragma once

#include <torch/extension.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include "teletron_norm.h"

namespace ttn_glue {

inline int dtype_code(const at::Tensor &t, const char *name) {
    if (t.scalar_type() == at::kBFloat16) return TT_NORM_BF16;
    if (t.scalar_type() == at::kFloat) return TT_NORM_F32;
    if (t.scalar_type() == at::kHalf) return TT_NORM_F16;
    TORCH_CHECK(false, name, ": expected a bfloat16, float16 or float32 tensor, got ", t.scalar_type());
}

inline void check_dense_on(const at::Tensor &t, const at::Device &dev, const char *name) {
    TORCH_CHECK(t.defined(), name, " is undefined");
    TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor");
    TORCH_CHECK(t.device() == dev, name, " is on ", t.device(), ", expected ", dev);
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

inline void check_elems(const at::Tensor &t, int64_t n, at::ScalarType st, const char *name) {
    TORCH_CHECK(t.numel() == n, name, " has ", t.numel(), " elements, expected ", n);
    TORCH_CHECK(t.scalar_type() == st, name, " has dtype ", t.scalar_type(), ", expected ", st);
}

inline void *current_stream(const at::Tensor &t) {
    return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

inline at::Tensor scratch(size_t bytes, const at::Tensor &like) {
    return at::empty({(int64_t)(bytes ? bytes : 16)}, like.options().dtype(at::kByte));
}

inline void raise_on(int status, const char *what) {
    TORCH_CHECK(status == TT_NORM_OK, what, " failed: ", tt_norm_status_string(status), " -- ",
                tt_norm_last_error());
}

// ---- whole calls -----------------------------------------------------------------------------
// The autograd functions' forward and backward as one call each: checks, allocations and launch without a return to
// Python between them.  They take only operands that need no preparation -- `ready`: an ordinary GPU tensor, contiguous,
// 16-byte aligned, of the row tensor's dtype and device -- and return None for anything else, which the Python code then
// prepares, or refuses with its own error.
inline bool ready(const at::Tensor &t, const at::Tensor &like) {
    return t.defined() && t.is_cuda() && !t.key_set().has(c10::DispatchKey::Python) && t.scalar_type() == like.scalar_type() &&
           t.device() == like.device() && t.is_contiguous() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}

inline bool ready_rows(const at::Tensor &x, int64_t cols) {
    const auto st = x.scalar_type();
    if (st != at::kBFloat16 && st != at::kHalf && st != at::kFloat) return false;
    return ready(x, x) && cols > 0 && x.numel() % cols == 0 && tt_norm_supported(cols, dtype_code(x, "input"));
}

// ---- call sites ------------------------------------------------------------------------------
// The functions a block calls, as autograd nodes of the host runtime: graph recording, forward, and a backward that runs on
// the engine's thread without the interpreter, its lock or a Python frame.  A call of forward and backward at 256 tokens is
// host work only (its kernels take 15 us): 77 us a pass with the Python functions, 65 with the nodes, of which the engine's
// hand-over to its thread and back takes 36 (QK-norm 106 -> 78, strided RMSNorm 90 -> 67, RMSNorm 6001 x 5120 78 -> 60).
// The nodes take operands that are ready and ordinary tensors; under a transform, a dispatch mode, tracing or a tangent they
// return None, and the Python functions handle or refuse the call as they always have (having been asked costs such a call 0.7 us
// of 22-34).  What is kept goes through SavedVariable, so saved-tensor hooks and version checks apply.
inline bool ordinary_call(std::initializer_list<const at::Tensor *> operands) {
    using c10::DispatchKey;
    const c10::DispatchKeySet modes({DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
                                     DispatchKey::FuncTorchVmapMode, DispatchKey::VmapMode, DispatchKey::Functionalize,
                                     DispatchKey::Tracer, DispatchKey::Python, DispatchKey::PreDispatch});
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        c10::impl::tls_local_dispatch_key_set().included_.has_any(modes))
        return false;
    const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                       DispatchKey::Batched, DispatchKey::Functionalize, DispatchKey::Negative,
                                       DispatchKey::Conjugate, DispatchKey::ZeroTensor});
    for (const at::Tensor *t : operands)
        if (!t->defined() || t->key_set().has_any(wrapped) || t->_fw_grad(0).defined()) return false;
    return true;
}

// Under create_graph the engine runs a node's backward with grad mode on and takes gradients that carry no graph for
// constants: a second derivative would lose their part without a word.  They leave with a graph that refuses instead.
constexpr const char *kFirstOrderOnly =
    "the fused norms have no second derivative: a gradient of theirs taken with create_graph=True cannot be differentiated again";

struct FirstOrderOnly : torch::autograd::Function<FirstOrderOnly> {
    static at::Tensor forward(torch::autograd::AutogradContext *, const at::Tensor &grad, at::TensorList) {
        return grad.tensor_data();
    }
    static std::vector<at::Tensor> backward(torch::autograd::AutogradContext *, std::vector<at::Tensor>) {
        TORCH_CHECK(false, kFirstOrderOnly);
    }
};

// kept, incoming: what the gradients were computed from, so that asking for a derivative by any of it meets the refusal.
inline std::vector<at::Tensor> first_order(std::vector<at::Tensor> grads, const std::vector<at::Tensor> &kept,
                                           const std::vector<at::Tensor> &incoming) {
    if (!at::GradMode::is_enabled()) return grads;
    std::vector<at::Tensor> from = kept;
    for (const at::Tensor &g : incoming)
        if (g.defined()) from.push_back(g);
    for (at::Tensor &g : grads)
        if (g.defined()) g = FirstOrderOnly::apply(g.detach().requires_grad_(true), at::TensorList(from));
    return grads;
}

// A gradient as the kernels take it: the saved tensor's dtype, contiguous, 16-byte aligned.
inline at::Tensor prepared(const at::Tensor &g, const at::Tensor &like) {
    if (!g.defined() || ready(g, like)) return g;
    at::Tensor t = g.to(like.scalar_type()).contiguous();
    return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) ? t.clone() : t;
}

inline std::vector<at::Tensor> taken(c10::optional<std::vector<at::Tensor>> done, const char *what) {
    TORCH_CHECK(done.has_value(), what, ": a gradient the kernels cannot take (another device, or no ordinary tensor)");
    return std::move(*done);
}

inline at::Tensor row_statistics(const at::Tensor &x, int64_t rows) { return at::empty({rows}, x.options().dtype(at::kFloat)); }

}  // namespace ttn_glue
