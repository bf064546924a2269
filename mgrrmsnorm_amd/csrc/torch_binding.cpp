// The torch extension over the C ABI of libmegagemm_hip.so: host-only C++ (no device code
// here), taking the place of the reference's pytorch_binding/binding.cpp.
//
//   rmsnorm_forward / rmsnorm_backward   the reference's two module functions
//       (binding.cpp:136-139), same checks and messages (binding.cpp:9-11,17-24,62-65),
//       outputs allocated here (binding.cpp:29-30,89-90); the dtype ladders collapse into one
//       C call each.
//   rmsnorm_backward_f32                 the same backward with dW also kept in fp32
//   swiglu_forward / swiglu_backward     tensor-level form of the two Triton launches
//       (megagemm/swiglu.py:89-131)
//   rmsnorm / swiglu                     the two operators as autograd nodes written in C++,
//       doing what RMSNormFunction (megagemm/rmsnorm.py:18-48) and MegaGemmFunction
//       (megagemm/swiglu.py:86-131) do, without a round trip through Python in backward
//
// Everything runs on torch's current stream of the tensors' device and never synchronises.
#include <torch/extension.h>
// torch on ROCm presents its devices as "cuda": the guard and stream types that go with that
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <algorithm>
#include <tuple>
#include <vector>

#include "megagemm_hip.h"
#include "megagemm_hip_fused.h"
#include "megagemm_hip_mlp.h"

namespace {

using torch::Tensor;

void check_input(const Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return MG_F32;
        case at::kHalf: return MG_F16;
        case at::kBFloat16: return MG_BF16;
        default: TORCH_CHECK(false, "Unsupported dtype ", t, ". Use float32, float16, or bfloat16."); return -1;
    }
}

void check_pair(const Tensor& input, const Tensor& weight) {
    TORCH_CHECK(input.dim() == 2, "Input must be 2D");
    TORCH_CHECK(weight.dim() == 1 && weight.size(0) == input.size(1), "Weight size must match hidden size");
    TORCH_CHECK(weight.scalar_type() == input.scalar_type(), "weight dtype (", weight.scalar_type(),
                ") must equal input dtype (", input.scalar_type(),
                "); cast the module, e.g. model.half() or model.to(torch.bfloat16)");
    TORCH_CHECK(weight.device() == input.device(), "input and weight must be on the same device");
}

// A contiguous tensor like a contiguous `t`: what empty_like gives, without the extra dispatch.
Tensor empty_as(const Tensor& t) { return at::empty(t.sizes(), t.options()); }

// `t` as a matrix of rows of `cols` elements: itself when it already is one (a view costs a dispatch,
// and forward + backward of a layer would make four).
Tensor as_rows(const Tensor& t, int64_t cols) { return t.dim() == 2 && t.size(1) == cols ? t : t.view({-1, cols}); }
Tensor as_shape(const Tensor& t, at::IntArrayRef shape) { return t.sizes() == shape ? t : t.view(shape); }

void* current_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

std::vector<Tensor> rmsnorm_forward(const Tensor& input, const Tensor& weight, double epsilon) {
    check_input(input, "input");
    check_input(weight, "weight");
    check_pair(input, weight);
    const int64_t rows = input.size(0), cols = input.size(1);
    TORCH_CHECK(cols >= 1, "hidden size must be >= 1");
    const int code = dtype_code(input.scalar_type());
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    auto output = empty_as(input);
    auto inv_rms = at::empty({rows}, input.options().dtype(torch::kFloat32));
    const int rc = mg_rmsnorm_fwd(output.data_ptr(), inv_rms.data_ptr<float>(), input.data_ptr(), weight.data_ptr(),
                                  rows, cols, (float)epsilon, code, current_stream());
    TORCH_CHECK(rc == MG_OK, "RMSNorm forward failed (code ", rc, "): ", mg_last_error());
    return {output, inv_rms};
}

// (grad_input, grad_weight in fp32, grad_weight in the weight's dtype); the last two are
// undefined tensors when need_weight_grad is false, and the same tensor for fp32 weights.
std::tuple<Tensor, Tensor, Tensor> backward_impl(const Tensor& grad_output, const Tensor& input, const Tensor& weight,
                                                 const Tensor& inv_rms, bool need_weight_grad, bool want_f32) {
    check_input(grad_output, "grad_output");
    check_input(input, "input");
    check_input(weight, "weight");
    check_input(inv_rms, "inv_rms");
    check_pair(input, weight);
    const int64_t rows = input.size(0), cols = input.size(1);
    TORCH_CHECK(grad_output.sizes() == input.sizes() && grad_output.scalar_type() == input.scalar_type(),
                "grad_output must have the shape and dtype of input");
    TORCH_CHECK(inv_rms.scalar_type() == at::kFloat && inv_rms.dim() == 1 && inv_rms.size(0) == rows,
                "inv_rms must be a float32 vector with one entry per row");
    const int code = dtype_code(input.scalar_type());
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    const auto f32 = input.options().dtype(torch::kFloat32);
    auto grad_input = empty_as(input);
    void* stream = current_stream();
    Tensor dw_f32, dw_cast;
    if (need_weight_grad) {
        if (want_f32 || code == MG_F32) dw_f32 = at::empty({cols}, f32);
        dw_cast = code == MG_F32 ? dw_f32 : empty_as(weight);   // weight dtype, as binding.cpp:90
    }
    float* const to_f32 = dw_f32.defined() ? dw_f32.data_ptr<float>() : nullptr;
    void* const to_cast = need_weight_grad && code != MG_F32 ? dw_cast.data_ptr() : nullptr;
    if (mg_rmsnorm_bwd_small_fits(rows, cols, code)) {   // few rows: one launch, no workspace
        const int rc = mg_rmsnorm_bwd_small(grad_input.data_ptr(), to_f32, to_cast, grad_output.data_ptr(), input.data_ptr(),
                                            weight.data_ptr(), inv_rms.data_ptr<float>(), rows, cols, code, stream);
        TORCH_CHECK(rc == MG_OK, "RMSNorm backward failed (code ", rc, "): ", mg_last_error());
        return {grad_input, dw_f32, dw_cast};
    }
    int64_t num_partials = 0, ld = 0;
    TORCH_CHECK(mg_rmsnorm_bwd_workspace(rows, cols, code, &num_partials, &ld) == MG_OK,
                "RMSNorm backward (workspace query) failed: ", mg_last_error());
    auto partial = at::empty({num_partials, ld}, f32);
    int rc = mg_rmsnorm_bwd(grad_input.data_ptr(), partial.data_ptr<float>(), grad_output.data_ptr(),
                            input.data_ptr(), weight.data_ptr(), inv_rms.data_ptr<float>(), rows, cols, code,
                            num_partials, ld, stream);
    TORCH_CHECK(rc == MG_OK, "RMSNorm backward failed (code ", rc, "): ", mg_last_error());
    if (need_weight_grad) {
        rc = mg_rmsnorm_dw_reduce(to_f32, to_cast, code, partial.data_ptr<float>(), num_partials, ld, cols, stream);
        TORCH_CHECK(rc == MG_OK, "RMSNorm backward (dW reduction) failed (code ", rc, "): ", mg_last_error());
    }
    return {grad_input, dw_f32, dw_cast};
}

std::tuple<Tensor, Tensor, Tensor> rmsnorm_backward_f32(const Tensor& grad_output, const Tensor& input,
                                                        const Tensor& weight, const Tensor& inv_rms,
                                                        bool need_weight_grad) {
    return backward_impl(grad_output, input, weight, inv_rms, need_weight_grad, true);
}

std::vector<Tensor> rmsnorm_backward(const Tensor& grad_output, const Tensor& input, const Tensor& weight,
                                     const Tensor& inv_rms) {
    auto r = backward_impl(grad_output, input, weight, inv_rms, true, false);
    return {std::get<0>(r), std::get<2>(r)};
}

// `backward_follows`: gate_up will be read again
Tensor swiglu_forward_impl(const Tensor& gate_up, int64_t hidden_dim, bool backward_follows) {
    check_input(gate_up, "w12_out");
    TORCH_CHECK(gate_up.dim() == 2 && gate_up.size(1) == 2 * hidden_dim, "expected a [M, ", 2 * hidden_dim,
                "] matrix, got ", gate_up.sizes());
    const int code = dtype_code(gate_up.scalar_type());
    const int64_t M = gate_up.size(0);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(gate_up.device());
    auto out = at::empty({M, hidden_dim}, gate_up.options());
    const auto forward = backward_follows ? mg_swiglu_fwd : mg_swiglu_fwd_only;
    const int rc = forward(out.data_ptr(), gate_up.data_ptr(), M, hidden_dim, code, current_stream());
    TORCH_CHECK(rc == MG_OK, "SwiGLU forward failed (code ", rc, "): ", mg_last_error());
    return out;
}

Tensor swiglu_forward(const Tensor& gate_up, int64_t hidden_dim) { return swiglu_forward_impl(gate_up, hidden_dim, true); }

Tensor swiglu_backward(const Tensor& grad_out, const Tensor& gate_up, int64_t hidden_dim) {
    check_input(grad_out, "grad_output");
    check_input(gate_up, "w12_out");
    TORCH_CHECK(gate_up.dim() == 2 && gate_up.size(1) == 2 * hidden_dim, "expected a [M, ", 2 * hidden_dim,
                "] matrix, got ", gate_up.sizes());
    const int64_t M = gate_up.size(0);
    TORCH_CHECK(grad_out.dim() == 2 && grad_out.size(0) == M && grad_out.size(1) == hidden_dim &&
                    grad_out.scalar_type() == gate_up.scalar_type(),
                "grad_output must be [M, hidden_dim] with the dtype of the forward input");
    const int code = dtype_code(gate_up.scalar_type());
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(gate_up.device());
    auto grad_in = empty_as(gate_up);
    const int rc = mg_swiglu_bwd(grad_in.data_ptr(), grad_out.data_ptr(), gate_up.data_ptr(), M, hidden_dim, code,
                                 current_stream());
    TORCH_CHECK(rc == MG_OK, "SwiGLU backward failed (code ", rc, "): ", mg_last_error());
    return grad_in;
}

// ---- autograd nodes ----
// Neither backward can be differentiated again (the kernels record no graph); asking for a
// second derivative raises, like torch's once_differentiable.
void refuse_double_backward(const Tensor& grad, const char* what) {
    TORCH_CHECK(!(torch::GradMode::is_enabled() && grad.requires_grad()), what,
                ": trying to differentiate twice a function whose backward is not differentiable");
}

struct RMSNormNode : public torch::autograd::Function<RMSNormNode> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& input, const Tensor& weight,
                          double epsilon) {
        TORCH_CHECK(input.dim() >= 1, "RMSNorm needs at least one dimension");
        // a view even of what is a matrix already: it keeps the data it was made of when a caller gives
        // `input` other data (`x.data = ...`) before the backward pass
        auto x2d = input.contiguous().view({-1, input.size(-1)});
        auto w = weight.contiguous();
        auto out = rmsnorm_forward(x2d, w, epsilon);
        ctx->save_for_backward({x2d, w, out[1]});
        return as_shape(out[0], input.sizes());
    }

    static torch::autograd::tensor_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::tensor_list grads) {
        refuse_double_backward(grads[0], "RMSNorm");
        torch::NoGradGuard no_grad;
        const auto saved = ctx->get_saved_variables();
        const Tensor &x2d = saved[0], &w = saved[1], &inv_rms = saved[2];
        auto dy = as_shape(grads[0].contiguous(), x2d.sizes());
        if (dy.scalar_type() != x2d.scalar_type()) dy = dy.to(x2d.scalar_type());
        auto r = backward_impl(dy, x2d, w, inv_rms, ctx->needs_input_grad(1), false);
        return {as_shape(std::get<0>(r), grads[0].sizes()), std::get<2>(r), Tensor()};   // y has the shape of x
    }
};

struct SwigluNode : public torch::autograd::Function<SwigluNode> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& w12_out, int64_t hidden_dim) {
        TORCH_CHECK(w12_out.dim() >= 1 && w12_out.size(-1) == 2 * hidden_dim, "last dimension must be 2*hidden_dim = ",
                    2 * hidden_dim, ", got ", w12_out.dim() >= 1 ? w12_out.size(-1) : 0);
        auto fused = w12_out.contiguous();
        ctx->save_for_backward({fused});
        auto shape = fused.sizes().vec();
        shape.back() = hidden_dim;
        return as_shape(swiglu_forward(as_rows(fused, 2 * hidden_dim), hidden_dim), shape);
    }

    static torch::autograd::tensor_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::tensor_list grads) {
        refuse_double_backward(grads[0], "SwiGLU");
        torch::NoGradGuard no_grad;
        const auto saved = ctx->get_saved_variables();
        const Tensor& fused = saved[0];
        const int64_t hidden_dim = fused.size(-1) / 2;
        auto dh = as_rows(grads[0].contiguous(), hidden_dim);
        if (dh.scalar_type() != fused.scalar_type()) dh = dh.to(fused.scalar_type());
        auto grad = swiglu_backward(dh, as_rows(fused, 2 * hidden_dim), hidden_dim);
        return {as_shape(grad, fused.sizes()), Tensor()};
    }
};

// y = x * rsqrt(mean(x^2, -1) + epsilon) * weight over the last dimension, differentiable.
Tensor rmsnorm(const Tensor& input, const Tensor& weight, double epsilon) {
    if (torch::GradMode::is_enabled() && (input.requires_grad() || weight.requires_grad()))
        return RMSNormNode::apply(input, weight, epsilon);
    // nothing to differentiate: same kernel, no node, no saved tensors and no per-row scale
    // (the C ABI takes a null inv_rms); the output keeps the input's shape, so no views either
    TORCH_CHECK(input.dim() >= 1, "RMSNorm needs at least one dimension");
    TORCH_CHECK(input.is_cuda(), "input must be a CUDA tensor");
    TORCH_CHECK(weight.is_cuda(), "weight must be a CUDA tensor");
    const Tensor x = input.contiguous(), w = weight.contiguous();   // themselves when they already are
    const int64_t cols = x.size(-1);
    TORCH_CHECK(cols >= 1, "hidden size must be >= 1");
    TORCH_CHECK(w.dim() == 1 && w.size(0) == cols, "Weight size must match hidden size");
    TORCH_CHECK(w.scalar_type() == x.scalar_type(), "weight dtype (", w.scalar_type(), ") must equal input dtype (",
                x.scalar_type(), "); cast the module, e.g. model.half() or model.to(torch.bfloat16)");
    TORCH_CHECK(w.device() == x.device(), "input and weight must be on the same device");
    const int code = dtype_code(x.scalar_type());
    const int64_t rows = x.numel() / cols;
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    auto output = empty_as(x);
    const int rc = mg_rmsnorm_fwd(output.data_ptr(), nullptr, x.data_ptr(), w.data_ptr(), rows, cols, (float)epsilon,
                                  code, current_stream());
    TORCH_CHECK(rc == MG_OK, "RMSNorm forward failed (code ", rc, "): ", mg_last_error());
    return output;
}

// silu(gate) * up on a fused [..., 2*hidden_dim] tensor, differentiable.
Tensor swiglu(const Tensor& w12_out, int64_t hidden_dim) {
    if (torch::GradMode::is_enabled() && w12_out.requires_grad()) return SwigluNode::apply(w12_out, hidden_dim);
    TORCH_CHECK(w12_out.dim() >= 1 && w12_out.size(-1) == 2 * hidden_dim, "last dimension must be 2*hidden_dim = ",
                2 * hidden_dim, ", got ", w12_out.dim() >= 1 ? w12_out.size(-1) : 0);
    auto fused = w12_out.contiguous();
    auto shape = fused.sizes().vec();
    shape.back() = hidden_dim;
    return as_shape(swiglu_forward_impl(as_rows(fused, 2 * hidden_dim), hidden_dim, false), shape);
}

// Where the two kernels of mg_block_gate_up and mg_block_down take no more GPU time than the projections
// and the activation between them; eager calls, which three operators keep at 47 us on the host, then win
// by more.  Each further tile of 16 tokens has every workgroup read that much more of the activations, and so
// does each pass that a wide projection takes, while the library's products take about as long for 17
// tokens as for 64.  GPU time in a replayed graph, us, these / projections and activation; d_model x hidden,
// MiB of weights; weights read from memory, and the same three layers in turn (what fits the cache):
//   16 tokens, every size measured (1 MiB to 2.3 GiB): 2048 x 3584 16.6 / 29.1, 4096 x 6912 38.8 / 54.6, 8192 x 28672
//     253 / 267, 12288 x 32768 412 / 428; the one loss is 8192 x 1024 with cached weights (21.1 / 23.7, 21.9 / 20.3);
//   32 tokens: 2048 x 3584 (42) 22.5 / 26.8, 22.2 / 22.9; 1280 x 5120 (38) 24.0 / 27.2, 24.1 / 24.3; beyond, 1792 x 4864
//     (50) 26.5 / 28.7, 26.2 / 25.5, 3072 x 8192 (144) 48.1 / 41.3 and at 17 tokens already 41.0 / 39.8, 5120 x
//     13824 (405) 108 / 92; wider than four to one, 1024 x 8192 (48) 32.2 / 30.3;
//   64 tokens: 768 x 2048 (9) 18.9 / 23.3, 19.3 / 19.3; 1024 x 1360 (8) 15.5 / 24.1, 15.7 / 20.1; beyond, 1024 x 2304 (14)
//     fp16 21.9 / 22.5, 22.6 / 19.0, 1536 x 2560 (22) 25.6 / 27.0, 25.8 / 22.3; wider than three to one, 576 x 2304
//     (8) fp16 19.6 / 19.1, 19.9 / 16.4.
bool block_in_two_kernels(int64_t tokens, int64_t d_model, int64_t hidden) {
    if (tokens < 1 || tokens > MG_BLOCK_MAX_TOKENS) return false;
    if (tokens <= 16) return true;
    const int64_t wide = std::max(d_model, hidden), narrow = std::min(d_model, hidden), bytes = 2 * 3 * d_model * hidden;
    return tokens <= 32 ? bytes <= (42LL << 20) && wide <= 4 * narrow : bytes <= (9LL << 20) && wide <= 3 * narrow;
}

// Whether a block of this hidden width may take `x` to swiglu_block at all, from x alone: asked first, so that
// the calls it is not for go on without the questions about modes and projections (2 us of 48).
bool swiglu_block_fits(const Tensor& x, int64_t hidden) {
    const auto type = x.scalar_type();
    if ((type != at::kHalf && type != at::kBFloat16) || !x.is_cuda() || x.dim() < 1 || x.size(-1) < 1) return false;
    if (x.requires_grad() && torch::GradMode::is_enabled()) return false;
    return block_in_two_kernels(x.numel() / x.size(-1), x.size(-1), hidden);
}

// w3(silu(gate) * up) with [gate | up] = w12(x) where nothing is to be differentiated and the call is
// one of those mg_block_gate_up and mg_block_down take; an undefined tensor (None) where it is not, and
// the caller then goes through the projections and the activation one by one.
Tensor swiglu_block(const Tensor& x, const Tensor& w12, const Tensor& w3) {
    const Tensor none;
    const auto type = x.scalar_type();
    if (!x.is_cuda() || (type != at::kHalf && type != at::kBFloat16) || x.dim() < 1 || w12.dim() != 2 || w3.dim() != 2)
        return none;
    // Sparse coordinate tensors are for the products (weights of that kind are not contiguous, below).
    // Compressed ones raise where they are asked whether they are contiguous, and should: torch's
    // product of 16-bit ones ends the process on ROCm 7 instead of raising.
    if (x.is_sparse()) return none;
    const int64_t d_model = w3.size(0), hidden = w3.size(1);
    if (d_model < 1 || x.size(-1) != d_model || w12.size(0) != 2 * hidden || w12.size(1) != d_model) return none;
    const int64_t tokens = x.numel() / d_model;
    if (!block_in_two_kernels(tokens, d_model, hidden) || d_model % 8 != 0 || hidden % 8 != 0 || hidden < 8) return none;
    if (w12.scalar_type() != type || w3.scalar_type() != type || w12.device() != x.device() || w3.device() != x.device() ||
        !w12.is_contiguous() || !w3.is_contiguous())
        return none;
    if (torch::GradMode::is_enabled() && (x.requires_grad() || w12.requires_grad() || w3.requires_grad())) return none;
    const Tensor xc = x.contiguous();
    const auto off = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0; };
    if (off(xc) || off(w12) || off(w3)) return none;
    const int code = dtype_code(type);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    auto h = at::empty({tokens, hidden}, xc.options());
    auto out = empty_as(xc);
    void* stream = current_stream();
    int rc = mg_block_gate_up(h.data_ptr(), xc.data_ptr(), w12.data_ptr(), tokens, d_model, hidden, code, stream);
    if (rc == MG_OK) rc = mg_block_down(out.data_ptr(), h.data_ptr(), w3.data_ptr(), tokens, d_model, hidden, code, stream);
    TORCH_CHECK(rc == MG_OK, "SwiGLU block failed (code ", rc, "): ", mg_last_error());
    return out;
}

// ---- the whole block on this package's own products ----
// A dense tensor of a GPU that nothing else wants to see the operations of: no transform of torch.func, no
// tangent, no lazy conjugate or negative, no subclass.
bool plain_dense(const Tensor& t) {
    constexpr c10::DispatchKeySet others({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Python,
                                          c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                          c10::DispatchKey::ZeroTensor, c10::DispatchKey::NestedTensor, c10::DispatchKey::Batched});
    return t.layout() == at::kStrided && t.is_cuda() && !t.key_set().has_any(others) && !t._fw_grad(0).defined();
}

// Saved tensors that somebody packs (checkpointing, offloading) and torch.func's transforms are for the
// projections, whose tensors these have always been.
bool calls_transformed() {
    return at::SavedTensorDefaultHooks::get_hooks(false).has_value() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// Whether a backward pass is for the kernels: one gradient, of which the same holds as of the operands (a batch of them
// is no such tensor), and no dispatch mode that looks on.
bool plain_backward(const Tensor& grad) {
    return grad.defined() && plain_dense(grad) && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// What mg_mlp_fwd or mg_mlp_bwd needs besides its tensors; undefined where that is nothing.
Tensor mlp_workspace(const Tensor& x, int64_t tokens, int64_t d_model, int64_t hidden, int pass) {
    int64_t need = 0;
    TORCH_CHECK(mg_mlp_workspace(tokens, d_model, hidden, dtype_code(x.scalar_type()), pass, &need) == MG_OK,
                "SwiGLU block (workspace query) failed: ", mg_last_error());
    return need > 0 ? at::empty({need}, x.options().dtype(at::kByte)) : Tensor();
}
void* pointer_of(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor mlp_forward(const Tensor& x, const Tensor& w12, const Tensor& w3, Tensor* gate_up, Tensor* h) {
    const int64_t d_model = w3.size(0), hidden = w3.size(1), tokens = x.numel() / d_model;
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    if (gate_up != nullptr) *gate_up = at::empty({tokens, 2 * hidden}, x.options());
    auto lead = x.sizes().vec();
    lead.back() = hidden;
    *h = at::empty(lead, x.options());
    auto out = empty_as(x);
    const Tensor work = mlp_workspace(x, tokens, d_model, hidden, MG_MLP_FORWARD);
    const int rc = mg_mlp_fwd(out.data_ptr(), h->data_ptr(), gate_up != nullptr ? gate_up->data_ptr() : nullptr, x.data_ptr(),
                              w12.data_ptr(), w3.data_ptr(), pointer_of(work), work.defined() ? work.numel() : 0, tokens, d_model, hidden, dtype_code(x.scalar_type()), current_stream());
    TORCH_CHECK(rc == MG_OK, "SwiGLU block forward failed (code ", rc, "): ", mg_last_error());
    return out;
}

struct MlpNode : public torch::autograd::Function<MlpNode> {
    // [out], and h where w3 learns: a graph recorded over the gradient of w3 gets through it to x and w12.
    // What linear layers keep is kept: x (contiguous here) for the gradient of w12, w12 for that of x, w3, h for that of w3.
    static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w12, const Tensor& w3) {
        // Aliases: they keep the data they were made of when a caller gives an operand other data before the backward pass.
        const Tensor none;
        const bool for_x = x.requires_grad(), for_12 = w12.requires_grad(), for_3 = w3.requires_grad();
        Tensor gate_up, h;
        const Tensor out = mlp_forward(x, w12, w3, &gate_up, &h);
        ctx->save_for_backward({for_12 ? x.detach() : none, for_x ? w12.detach() : none, w3.detach(), gate_up, for_3 ? h : none});
        ctx->set_materialize_grads(false);
        if (!for_3) return {out};
        return {out, h};
    }

    static torch::autograd::tensor_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::tensor_list grads) {
        const auto saved = ctx->get_saved_variables();
        const bool want[] = {ctx->needs_input_grad(0), ctx->needs_input_grad(1), ctx->needs_input_grad(2)};
        torch::autograd::tensor_list out(3);
        const bool records = torch::GradMode::is_enabled();
        const auto node = records ? torch::autograd::get_current_node() : nullptr;
        const auto operand = [&](int i) { return records ? connected(saved[i], node->next_edge(i)) : saved[i]; };
        if (!records && (grads.size() == 1 || !grads[1].defined()) && plain_backward(grads[0])) {
            in_kernels(out, grads[0], want, saved);
        } else {
            in_operations(out, grads, want, operand(0), operand(1), operand(2), saved[3], saved[4]);
        }
        return out;
    }

    // An operand as it was kept, in the graph where the operand was.
    static Tensor connected(const Tensor& kept, const torch::autograd::Edge& edge) {
        if (!kept.defined() || !edge.is_valid()) return kept;
        const Tensor t = kept.detach();
        torch::autograd::impl::set_gradient_edge(t, edge);
        return t;
    }

    static void in_kernels(torch::autograd::tensor_list& out, const Tensor& grad, const bool* want, const torch::autograd::variable_list& saved) {
        const Tensor &x = saved[0], &w12 = saved[1], &w3 = saved[2], &gate_up = saved[3], &h = saved[4];
        const auto type = gate_up.scalar_type();
        const int64_t d_model = w3.size(0), hidden = w3.size(1), tokens = gate_up.size(0);
        const c10::hip::HIPGuardMasqueradingAsCUDA guard(gate_up.device());
        auto dy = grad.contiguous();
        if (dy.scalar_type() != type) dy = dy.to(type);
        if (reinterpret_cast<uintptr_t>(dy.data_ptr()) % 16 != 0) dy = dy.clone();
        Tensor d_gate_up;
        if (want[0] || want[1]) d_gate_up = empty_as(gate_up);
        if (want[0]) out[0] = empty_as(dy);
        if (want[1]) out[1] = at::empty({2 * hidden, d_model}, dy.options());
        if (want[2]) out[2] = at::empty({d_model, hidden}, dy.options());
        const Tensor work = mlp_workspace(gate_up, tokens, d_model, hidden, (want[0] ? MG_MLP_DX : 0) | (want[1] ? MG_MLP_DW12 : 0) | (want[2] ? MG_MLP_DW3 : 0));
        const int rc = mg_mlp_bwd(pointer_of(out[0]), pointer_of(out[1]), pointer_of(out[2]), pointer_of(d_gate_up), dy.data_ptr(), pointer_of(x),
                                  pointer_of(w12), w3.data_ptr(), gate_up.data_ptr(), pointer_of(h), pointer_of(work),
                                  work.defined() ? work.numel() : 0, tokens, d_model, hidden, dtype_code(type), current_stream());
        TORCH_CHECK(rc == MG_OK, "SwiGLU block backward failed (code ", rc, "): ", mg_last_error());
    }

    // What the projections' and the activation's backward passes do, as operations that record a graph where one is wanted,
    // take the gradients those take and refuse what those refuse.
    static void in_operations(torch::autograd::tensor_list& out, const torch::autograd::tensor_list& grads, const bool* want, const Tensor& x,
                              const Tensor& w12, const Tensor& w3, const Tensor& gate_up, const Tensor& h) {
        const int64_t d_model = w3.size(0), hidden = w3.size(1);
        const auto type = gate_up.scalar_type();
        const bool through_h = grads.size() == 2 && grads[1].defined();
        Tensor dy, dh = through_h ? grads[1].reshape({-1, hidden}) : Tensor();
        if (grads[0].defined()) {
            dy = grads[0].to(type).reshape({-1, d_model});
            if (want[2]) out[2] = at::mm(dy.t(), h.reshape({-1, hidden}));
            if (want[0] || want[1]) dh = dh.defined() ? dh + at::mm(dy, w3) : at::mm(dy, w3);
        }
        if (!dh.defined() || !(want[0] || want[1])) return;
        refuse_double_backward(dh, "SwiGLU");
        Tensor d_gate_up;
        {
            torch::NoGradGuard no_grad;
            d_gate_up = swiglu_backward(dh.to(type).contiguous(), gate_up, hidden);
        }
        if (want[0]) {
            auto shape = (through_h ? grads[1] : grads[0]).sizes().vec();
            shape.back() = d_model;
            out[0] = at::mm(d_gate_up, w12).reshape(shape);
        }
        if (want[1]) out[1] = at::mm(d_gate_up.t(), x.reshape({-1, d_model}));
    }
};

// Whether a block of this hidden width may take `x` to swiglu_mlp at all, from x alone.
bool swiglu_mlp_fits(const Tensor& x, int64_t hidden) {
    const auto type = x.scalar_type();
    if ((type != at::kHalf && type != at::kBFloat16) || !x.is_cuda() || x.dim() < 1 || x.size(-1) < 1) return false;
    return mg_mlp_preferred(x.numel() / x.size(-1), x.size(-1), hidden, dtype_code(type), torch::GradMode::is_enabled() ? MG_MLP_ALL : MG_MLP_FORWARD_ONLY) == 1;
}

// w3(silu(gate) * up) with [gate | up] = w12(x), differentiable, in this package's own products; an undefined tensor
// (None) where the call is not one of theirs, and the caller then goes through the projections and the activation.
Tensor swiglu_mlp(const Tensor& x, const Tensor& w12, const Tensor& w3) {
    const Tensor none;
    const auto type = x.scalar_type();
    if ((type != at::kHalf && type != at::kBFloat16) || x.dim() < 1 || w12.dim() != 2 || w3.dim() != 2) return none;
    if (!plain_dense(x) || !plain_dense(w12) || !plain_dense(w3) || calls_transformed()) return none;
    const int64_t d_model = w3.size(0), hidden = w3.size(1);
    if (d_model < 1 || x.size(-1) != d_model || w12.size(0) != 2 * hidden || w12.size(1) != d_model) return none;
    if (w12.scalar_type() != type || w3.scalar_type() != type || w12.device() != x.device() || w3.device() != x.device() ||
        !w12.is_contiguous() || !w3.is_contiguous())
        return none;
    const bool weights_learn = w12.requires_grad() || w3.requires_grad(), learns = torch::GradMode::is_enabled() && (x.requires_grad() || weights_learn);
    const int call = !learns ? MG_MLP_FORWARD_ONLY : weights_learn ? MG_MLP_ALL : MG_MLP_X_LEARNS;
    if (mg_mlp_preferred(x.numel() / d_model, d_model, hidden, dtype_code(type), call) != 1) return none;
    const auto off = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0; };
    if (off(w12) || off(w3) || (x.is_contiguous() && off(x))) return none;   // a copy of x is aligned
    if (learns) {
        if (!x.requires_grad() && !w12.requires_grad()) return none;   // only w3 learns: nothing of the activation has to be kept
        return MlpNode::apply(x.contiguous(), w12, w3)[0];
    }
    Tensor h;
    return mlp_forward(x.contiguous(), w12, w3, nullptr, &h);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "torch extension over libmegagemm_hip.so (C ABI version " + std::to_string(MG_ABI_VERSION) + ")";
    m.def("abi_version", [] { return mg_abi_version(); }, "ABI version of the loaded libmegagemm_hip.so");
    m.def("built_abi_version", [] { return MG_ABI_VERSION; },
          "MG_ABI_VERSION of the header this extension was compiled against");
    m.def("rmsnorm_forward", &rmsnorm_forward, "RMSNorm forward: [output, inv_rms]", py::arg("input"),
          py::arg("weight"), py::arg("epsilon"));
    m.def("rmsnorm_backward", &rmsnorm_backward, "RMSNorm backward: [grad_input, grad_weight]",
          py::arg("grad_output"), py::arg("input"), py::arg("weight"), py::arg("inv_rms"));
    m.def("rmsnorm_backward_f32", &rmsnorm_backward_f32,
          "RMSNorm backward: (grad_input, grad_weight fp32, grad_weight in the weight's dtype)", py::arg("grad_output"),
          py::arg("input"), py::arg("weight"), py::arg("inv_rms"), py::arg("need_weight_grad") = true);
    m.def("swiglu_forward", &swiglu_forward, "silu(gate) * up on [M, 2H] -> [M, H]", py::arg("gate_up"),
          py::arg("hidden_dim"));
    m.def("swiglu_backward", &swiglu_backward, "[d_gate | d_up] from grad_out [M, H] and gate_up [M, 2H]",
          py::arg("grad_out"), py::arg("gate_up"), py::arg("hidden_dim"));
    m.def("rmsnorm", &rmsnorm, "differentiable RMSNorm over the last dimension", py::arg("input"), py::arg("weight"),
          py::arg("epsilon") = 1e-5);
    m.def("swiglu_block", &swiglu_block, "the whole SwiGLU block for a few rows, not differentiable; None where it does not apply",
          py::arg("x"), py::arg("w12"), py::arg("w3"));
    m.def("swiglu_block_fits", &swiglu_block_fits, "whether the size and type of x are for swiglu_block", py::arg("x"),
          py::arg("hidden_dim"));
    m.def("swiglu_mlp", &swiglu_mlp, "the whole SwiGLU block, differentiable, on the package's own products; None where it does not apply",
          py::arg("x"), py::arg("w12"), py::arg("w3"));
    m.def("swiglu_mlp_fits", &swiglu_mlp_fits, "whether the size and type of x are for swiglu_mlp", py::arg("x"), py::arg("hidden_dim"));
    m.def("swiglu", &swiglu, "differentiable silu(gate) * up over the last dimension", py::arg("w12_out"),
          py::arg("hidden_dim"));
}
