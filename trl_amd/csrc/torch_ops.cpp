// PyTorch operators of the logits-level steps over the C ABI (include/trlk.h): log-probs and entropies, the GRPO and DPO
// losses and what they log.  A step of a small run consists of a dozen launches of a few microseconds, so what a call
// costs on the host counts: an operator registered from Python spends 10 to 15 us per call in Python layers (argument
// conversion, the autograd and aliasing wrappers, ctypes, one Python tensor object per temporary), one registered here 3
// to 5.  Their shapes for tracers are registered in ops.py.
//
// Each operator checks its shapes, allocates its outputs and hands raw device pointers, sizes, strides and the
// current stream of the tensors' device to the library.  GPU tensors only: other devices have no kernel registered.
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/library.h>
#include <torch/python.h>

#include <cstdlib>
#include <map>
#include <mutex>
#include <string>

#include "trlk.h"

namespace {
using at::Tensor;
using std::optional;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A status of the library as the exception class that the Python package raises for it.
void check(int status) {
    if (status == 0) return;
    const std::string what = (status < 0 ? "trlk status " : "trlk launch failed with hipError_t ") + std::to_string(status) +
                             ": " + trlk_last_error();
    pybind11::gil_scoped_acquire gil;
    const auto lib = pybind11::module_::import("trl_amd._lib");
    const auto cls = lib.attr(status < 0 ? "TrlkArgumentError" : "TrlkError");
    PyErr_SetString(cls.ptr(), what.c_str());
    throw pybind11::error_already_set();
}

int dtype_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return TRLK_F32;
        case at::kBFloat16: return TRLK_BF16;
        case at::kHalf: return TRLK_F16;
        default:
            TORCH_CHECK_TYPE(false, "trl_amd kernels take float32, bfloat16 or float16 logits, got ", t.scalar_type());
    }
}

trlk_stream_t stream_of(const Tensor& t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}
Tensor f32(const Tensor& like, at::IntArrayRef sizes) { return at::empty(sizes, like.options().dtype(at::kFloat)); }
// fp32 and contiguous
Tensor f32c(const Tensor& t) { return t.contiguous().to(at::kFloat); }
optional<Tensor> f32c(const optional<Tensor>& t) { return t ? optional<Tensor>(f32c(*t)) : std::nullopt; }
// The data of an operand.  A call is dispatched here if ANY of its tensors is on a GPU: one in ordinary host memory among them
// is an error and must not reach a kernel (pinned memory can be read).
const void* operand(const Tensor& t) {
    TORCH_CHECK(t.is_cuda() || t.numel() == 0 || t.is_pinned(),
                "Expected all tensors to be on the same device, but found one of shape ", t.sizes(), " on ", t.device());
    return t.const_data_ptr();
}
const float* fptr(const Tensor& t) { return static_cast<const float*>(operand(t)); }
const float* fptr(const optional<Tensor>& t) { return t ? fptr(*t) : nullptr; }
float* out(const Tensor& t) { return static_cast<float*>(t.mutable_data_ptr()); }
const int64_t* iptr(const Tensor& t) { return static_cast<const int64_t*>(operand(t)); }

// The int32 word per device that the kernels OR error bits into.  It lives until the process ends.
struct ErrorFlags {
    std::mutex mutex;
    std::map<int64_t, Tensor> of_device;
};
ErrorFlags& error_flags() {
    static auto* flags = new ErrorFlags;  // (never destroyed: the runtime may be gone by then)
    return *flags;
}
Tensor error_flag(int64_t index) {
    ErrorFlags& flags = error_flags();
    std::lock_guard<std::mutex> lock(flags.mutex);
    auto it = flags.of_device.find(index);
    if (it == flags.of_device.end()) {
        const c10::InferenceMode off(false);  // (a word made in inference mode could not be cleared outside of it)
        it = flags.of_device.emplace(index, at::zeros({1}, at::TensorOptions().dtype(at::kInt).device(at::kCUDA, index))).first;
    }
    return it->second;
}
std::vector<Tensor> all_error_flags() {
    ErrorFlags& flags = error_flags();
    std::lock_guard<std::mutex> lock(flags.mutex);
    std::vector<Tensor> all;
    for (const auto& f : flags.of_device) all.push_back(f.second);
    return all;
}
int32_t* error_word(const Tensor& t) { return static_cast<int32_t*>(error_flag(t.device().index()).mutable_data_ptr()); }

// With TRL_AMD_SYNC_CHECKS=1 the error words are looked at behind each launch that reads token ids (a synchronisation).
const bool kSyncChecks = [] {
    const char* value = std::getenv("TRL_AMD_SYNC_CHECKS");
    return value != nullptr && std::string(value) == "1";
}();
void check_ids() {
    if (!kSyncChecks) return;
    pybind11::gil_scoped_acquire gil;
    pybind11::module_::import("trl_amd.ops").attr("check_device_errors")();
}

void check_logits3d(const Tensor& logits) {
    TORCH_CHECK_VALUE(logits.dim() == 3, "expected [n_seq, rows, vocab] logits, got shape ", logits.sizes());
    TORCH_CHECK_VALUE(logits.size(2) <= 1 || logits.stride(2) == 1, "the vocabulary axis of the logits must be contiguous");
    (void)operand(logits);
}
// the rows from keep_start on of every sequence
const char* window(const Tensor& logits, int64_t keep_start) {
    return static_cast<const char*>(logits.const_data_ptr()) + keep_start * logits.stride(1) * logits.element_size();
}
void check_window(const Tensor& logits, int64_t keep_start, int64_t keep_len) {
    TORCH_CHECK_VALUE(keep_start >= 0 && keep_len >= 0 && keep_start + keep_len <= logits.size(1), "rows ", keep_start, " to ",
                      keep_start + keep_len, " of ", logits.size(1));
}

// ---- log-probs and entropies ----------------------------------------------------------------------------------------
typedef std::tuple<Tensor, Tensor, Tensor> Tensor3;
typedef std::tuple<Tensor, Tensor, Tensor, Tensor> Tensor4;

Tensor4 run_logp_entropy(const Tensor& logits, const Tensor& index_, double temperature, int64_t keep_start, int64_t keep_len,
                         const optional<Tensor>& row_mask, bool with_stats, bool sum_p2) {
    check_logits3d(logits);
    const int64_t n_seq = logits.size(0), vocab = logits.size(2), rows = n_seq * keep_len, k = index_.size(-1);
    const c10::DeviceGuard guard(logits.device());
    Tensor logp = f32(logits, {rows, k}), ent = f32(logits, {rows}), lse = f32(logits, {rows}), stats;
    if (with_stats) stats = f32(logits, {rows, 4});
    if (rows == 0) return {logp, ent, lse, stats};
    check_window(logits, keep_start, keep_len);
    const Tensor index = index_.contiguous();
    check(trlk_logp_entropy_fwd(window(logits, keep_start), dtype_code(logits), n_seq, keep_len, vocab, logits.stride(0),
                                logits.stride(1), iptr(index), k, float(temperature),
                                row_mask ? static_cast<const uint8_t*>(operand(*row_mask)) : nullptr, out(logp), out(ent),
                                out(lse), with_stats ? out(stats) : nullptr, sum_p2 ? 1 : 0, error_word(logits),
                                stream_of(logits)));
    check_ids();
    return {logp, ent, lse, stats};
}
Tensor3 logp_entropy_fwd(const Tensor& logits, const Tensor& index, double temperature, int64_t keep_start, int64_t keep_len,
                         const optional<Tensor>& row_mask) {
    auto [logp, ent, lse, stats] = run_logp_entropy(logits, index, temperature, keep_start, keep_len, row_mask, false, true);
    return {logp, ent, lse};
}
Tensor4 logp_entropy_stats_fwd(const Tensor& logits, const Tensor& index, double temperature, int64_t keep_start,
                               int64_t keep_len, const optional<Tensor>& row_mask, bool sum_p2) {
    return run_logp_entropy(logits, index, temperature, keep_start, keep_len, row_mask, true, sum_p2);
}

Tensor logp_entropy_bwd(const Tensor& logits, const Tensor& index_, double temperature, int64_t keep_start, int64_t keep_len,
                        const Tensor& lse, const optional<Tensor>& entropy, const optional<Tensor>& g_logp_,
                        const optional<Tensor>& g_entropy_) {
    check_logits3d(logits);
    const int64_t n_seq = logits.size(0), length = logits.size(1), vocab = logits.size(2);
    const c10::DeviceGuard guard(logits.device());
    const Tensor dlogits = at::empty({n_seq, length, vocab}, logits.options());
    if (dlogits.numel() == 0) return dlogits;
    check_window(logits, keep_start, keep_len);
    const int64_t k = g_logp_ ? index_.size(-1) : 0;
    const Tensor index = index_.contiguous();
    const optional<Tensor> g_logp = f32c(g_logp_), g_entropy = f32c(g_entropy_);
    check(trlk_logp_entropy_bwd(window(logits, keep_start), dtype_code(logits), n_seq, keep_len, vocab, logits.stride(0),
                                logits.stride(1), iptr(index), k, float(temperature), fptr(lse),
                                g_entropy ? fptr(entropy) : nullptr, fptr(g_logp), fptr(g_entropy), dlogits.mutable_data_ptr(),
                                length, keep_start, dlogits.stride(0), dlogits.stride(1), stream_of(logits)));
    return dlogits;
}

// (the row window may be symbolic while a program is traced, so everything above the device kernels takes c10::SymInt)
typedef Tensor3 LogpEntropySig(const Tensor&, const Tensor&, double, c10::SymInt, c10::SymInt, const optional<Tensor>&);
typedef Tensor4 LogpEntropyStatsSig(const Tensor&, const Tensor&, double, c10::SymInt, c10::SymInt, const optional<Tensor>&, bool);
typedef Tensor LogpEntropyBwdSig(const Tensor&, const Tensor&, double, c10::SymInt, c10::SymInt, const Tensor&,
                                 const optional<Tensor>&, const optional<Tensor>&, const optional<Tensor>&);
template <typename Signature>
c10::TypedOperatorHandle<Signature> handle(const char* name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Signature>();
}
bool needs_grad(std::initializer_list<const Tensor*> tensors) {
    if (!c10::GradMode::is_enabled()) return false;
    for (const Tensor* t : tensors)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}
bool needs_grad(const optional<Tensor>& t) { return t && needs_grad({&*t}); }

// The gradient of the log-prob operators: the backward kernel recomputes the softmax from the saved per-row logsumexp.
class LogpEntropy : public torch::autograd::Function<LogpEntropy> {
  public:
    static variable_list forward(AutogradContext* ctx, const Tensor& logits, const Tensor& index, double temperature,
                                 c10::SymInt keep_start, c10::SymInt keep_len, const optional<Tensor>& row_mask, bool with_stats,
                                 bool sum_p2) {
        variable_list result;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            if (with_stats) {
                static const auto op = handle<LogpEntropyStatsSig>("trl_amd::logp_entropy_stats_fwd");
                auto [logp, ent, lse, stats] = op.call(logits, index, temperature, keep_start, keep_len, row_mask, sum_p2);
                result = {logp, ent, lse, stats};
            } else {
                static const auto op = handle<LogpEntropySig>("trl_amd::logp_entropy_fwd");
                auto [logp, ent, lse] = op.call(logits, index, temperature, keep_start, keep_len, row_mask);
                result = {logp, ent, lse};
            }
        }
        ctx->save_for_backward({logits, index, result[2], result[1]});
        ctx->saved_data["temperature"] = temperature;
        ctx->saved_data["keep_start"] = keep_start;
        ctx->saved_data["keep_len"] = keep_len;
        ctx->set_materialize_grads(false);
        return result;
    }
    // (the lse output only exists to be saved for this backward; a gradient arriving there is ignored)
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        variable_list result(8);
        Tensor g_logp = grads[0];
        const Tensor& g_ent = grads[1];
        if (!g_logp.defined() && !g_ent.defined()) return result;
        const auto saved = ctx->get_saved_variables();
        const Tensor &logits = saved[0], &index = saved[1];
        if (!g_logp.defined() && index.sym_size(-1) > 0)
            g_logp = at::zeros_symint(index.sym_sizes(), logits.options().dtype(at::kFloat));
        static const auto op = handle<LogpEntropyBwdSig>("trl_amd::logp_entropy_bwd");
        result[0] = op.call(logits, index, ctx->saved_data["temperature"].toDouble(), ctx->saved_data["keep_start"].toSymInt(),
                            ctx->saved_data["keep_len"].toSymInt(), saved[2], saved[3],
                            g_logp.defined() ? optional<Tensor>(g_logp) : std::nullopt,
                            g_ent.defined() ? optional<Tensor>(g_ent) : std::nullopt);
        return result;
    }
};
Tensor3 logp_entropy_fwd_autograd(const Tensor& logits, const Tensor& index, double temperature, c10::SymInt keep_start,
                                  c10::SymInt keep_len, const optional<Tensor>& row_mask) {
    if (needs_grad({&logits})) {
        const auto r = LogpEntropy::apply(logits, index, temperature, keep_start, keep_len, row_mask, false, true);
        return {r[0], r[1], r[2]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = handle<LogpEntropySig>("trl_amd::logp_entropy_fwd");
    return op.call(logits, index, temperature, keep_start, keep_len, row_mask);
}
Tensor4 logp_entropy_stats_fwd_autograd(const Tensor& logits, const Tensor& index, double temperature, c10::SymInt keep_start,
                                        c10::SymInt keep_len, const optional<Tensor>& row_mask, bool sum_p2) {
    if (needs_grad({&logits})) {
        const auto r = LogpEntropy::apply(logits, index, temperature, keep_start, keep_len, row_mask, true, sum_p2);
        return {r[0], r[1], r[2], r[3]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = handle<LogpEntropyStatsSig>("trl_amd::logp_entropy_stats_fwd");
    return op.call(logits, index, temperature, keep_start, keep_len, row_mask, sum_p2);
}

// ---- GRPO -----------------------------------------------------------------------------------------------------------
void check_token_shape(const char* op, const char* name, const optional<Tensor>& t, int64_t B, int64_t T) {
    TORCH_CHECK_VALUE(!t || (t->dim() == 2 && t->size(0) == B && t->size(1) == T), op, ": ", name, " has shape ",
                      t ? t->sizes() : at::IntArrayRef(), ", expected (", B, ", ", T, ")");
}
// strides of the advantages along (sequence, token): one per sequence, or one per token
std::pair<int64_t, int64_t> advantage_strides(const char* op, const Tensor& adv, int64_t B, int64_t T) {
    if (adv.dim() == 1 || (adv.dim() == 2 && adv.size(1) == 1)) {
        TORCH_CHECK_VALUE(adv.numel() == B, op, ": advantages must have one entry per sequence");
        return {1, 0};
    }
    TORCH_CHECK_VALUE(adv.dim() == 2 && adv.size(0) == B && adv.size(1) == T, op, ": advantages of shape ", adv.sizes(),
                      " do not match [B]=", B, " or [B,T]");
    return {T, 1};
}

Tensor4 grpo_loss(const Tensor& logp_, const optional<Tensor>& old_, const optional<Tensor>& ref_, const optional<Tensor>& ent_,
                  const Tensor& advantages_, const Tensor& mask_, const optional<Tensor>& weight_,
                  const optional<Tensor>& entropy_mask_, const optional<Tensor>& normalizer_, int64_t loss_type,
                  double epsilon_low, double epsilon_high, double delta, double beta, bool bias_correction_kl,
                  double grad_accum_steps, double dr_grpo_denominator, double num_processes, double entropy_coef,
                  int64_t policy_term, bool sequence_level, const optional<Tensor>& seq_coef_, double sapo_pos, double sapo_neg) {
    TORCH_CHECK_VALUE(logp_.dim() == 2, "grpo_loss: per-token log-probs must be [B, T]");
    const int64_t B = logp_.size(0), T = logp_.size(1);
    const c10::DeviceGuard guard(logp_.device());
    const Tensor logp = f32c(logp_), mask = f32c(mask_), advantages = f32c(advantages_);
    const optional<Tensor> old = f32c(old_), ref = f32c(ref_), ent = f32c(ent_), weight = f32c(weight_),
                           entropy_mask = f32c(entropy_mask_);
    const auto [sb, st] = advantage_strides("grpo_loss", advantages, B, T);
    check_token_shape("grpo_loss", "old_logp", old, B, T);
    check_token_shape("grpo_loss", "ref_logp", ref, B, T);
    check_token_shape("grpo_loss", "entropy", ent, B, T);
    check_token_shape("grpo_loss", "mask", mask, B, T);
    check_token_shape("grpo_loss", "token_weight", weight, B, T);
    check_token_shape("grpo_loss", "entropy_mask", entropy_mask, B, T);
    const optional<Tensor> normalizer = normalizer_ ? f32c(optional<Tensor>(normalizer_->reshape({1}))) : std::nullopt;
    TORCH_CHECK_VALUE(!seq_coef_ || seq_coef_->numel() == B, "grpo_loss: seq_coef must have one entry per sequence");
    const optional<Tensor> seq_coef = seq_coef_ ? f32c(optional<Tensor>(seq_coef_->reshape({B}))) : std::nullopt;
    const Tensor loss = f32(logp, {}), metrics = f32(logp, {TRLK_GRPO_NUM_METRICS}), dlogp = f32(logp, {B, T}),
                 dent = entropy_coef != 0.0 ? f32(logp, {B, T}) : f32(logp, {0});
    const size_t ws_bytes = trlk_grpo_workspace_bytes(B);
    const Tensor ws = at::empty({int64_t(ws_bytes)}, logp.options().dtype(at::kByte));
    check(trlk_grpo_loss(fptr(logp), fptr(old), fptr(ref), fptr(ent), fptr(advantages), sb, st, fptr(mask), fptr(weight),
                         fptr(entropy_mask), fptr(seq_coef), B, T, int(loss_type), int(policy_term), sequence_level ? 1 : 0,
                         float(epsilon_low), float(epsilon_high), float(delta), float(beta), bias_correction_kl ? 1 : 0,
                         float(grad_accum_steps), float(dr_grpo_denominator), fptr(normalizer), float(num_processes),
                         float(entropy_coef), float(sapo_pos), float(sapo_neg), out(loss), out(metrics), out(dlogp),
                         entropy_coef != 0.0 ? out(dent) : nullptr, ws.mutable_data_ptr(), ws_bytes, stream_of(logp)));
    return {loss, metrics, dlogp, dent};
}

class GrpoLoss : public torch::autograd::Function<GrpoLoss> {
  public:
    static variable_list forward(AutogradContext* ctx, const Tensor& logp, const optional<Tensor>& old, const optional<Tensor>& ref,
                                 const optional<Tensor>& ent, const Tensor& advantages, const Tensor& mask,
                                 const optional<Tensor>& weight, const optional<Tensor>& entropy_mask,
                                 const optional<Tensor>& normalizer, int64_t loss_type, double epsilon_low, double epsilon_high,
                                 double delta, double beta, bool bias_correction_kl, double grad_accum_steps,
                                 double dr_grpo_denominator, double num_processes, double entropy_coef, int64_t policy_term,
                                 bool sequence_level, const optional<Tensor>& seq_coef, double sapo_pos, double sapo_neg) {
        variable_list result;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            static const auto op = handle<decltype(grpo_loss)>("trl_amd::grpo_loss");
            auto [loss, metrics, dlogp, dent] =
                op.call(logp, old, ref, ent, advantages, mask, weight, entropy_mask, normalizer, loss_type, epsilon_low,
                        epsilon_high, delta, beta, bias_correction_kl, grad_accum_steps, dr_grpo_denominator, num_processes,
                        entropy_coef, policy_term, sequence_level, seq_coef, sapo_pos, sapo_neg);
            result = {loss, metrics, dlogp, dent};
        }
        ctx->save_for_backward({result[2], result[3]});
        ctx->saved_data["dtype"] = logp.scalar_type();
        ctx->saved_data["entropy"] = entropy_coef != 0.0 && ent.has_value();
        ctx->set_materialize_grads(false);
        return result;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        variable_list result(24);
        if (!grads[0].defined()) return result;
        const auto saved = ctx->get_saved_variables();
        result[0] = (grads[0] * saved[0]).to(ctx->saved_data["dtype"].toScalarType());
        if (ctx->saved_data["entropy"].toBool()) result[3] = grads[0] * saved[1];
        return result;
    }
};
Tensor4 grpo_loss_autograd(const Tensor& logp, const optional<Tensor>& old, const optional<Tensor>& ref, const optional<Tensor>& ent,
                           const Tensor& advantages, const Tensor& mask, const optional<Tensor>& weight,
                           const optional<Tensor>& entropy_mask, const optional<Tensor>& normalizer, int64_t loss_type,
                           double epsilon_low, double epsilon_high, double delta, double beta, bool bias_correction_kl,
                           double grad_accum_steps, double dr_grpo_denominator, double num_processes, double entropy_coef,
                           int64_t policy_term, bool sequence_level, const optional<Tensor>& seq_coef, double sapo_pos,
                           double sapo_neg) {
    const bool grad = needs_grad({&logp, &advantages, &mask}) || needs_grad(old) || needs_grad(ref) || needs_grad(ent) ||
                      needs_grad(weight) || needs_grad(entropy_mask) || needs_grad(normalizer) || needs_grad(seq_coef);
    if (grad) {
        const auto r = GrpoLoss::apply(logp, old, ref, ent, advantages, mask, weight, entropy_mask, normalizer, loss_type,
                                       epsilon_low, epsilon_high, delta, beta, bias_correction_kl, grad_accum_steps,
                                       dr_grpo_denominator, num_processes, entropy_coef, policy_term, sequence_level, seq_coef,
                                       sapo_pos, sapo_neg);
        return {r[0], r[1], r[2], r[3]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = handle<decltype(grpo_loss)>("trl_amd::grpo_loss");
    return op.call(logp, old, ref, ent, advantages, mask, weight, entropy_mask, normalizer, loss_type, epsilon_low, epsilon_high,
                   delta, beta, bias_correction_kl, grad_accum_steps, dr_grpo_denominator, num_processes, entropy_coef,
                   policy_term, sequence_level, seq_coef, sapo_pos, sapo_neg);
}

Tensor4 grpo_fused(const Tensor& logits, const Tensor& index_, double temperature, int64_t keep_start, int64_t keep_len,
                   const Tensor& mask_, const Tensor& advantages_, const Tensor& row_scale_, const optional<Tensor>& old_,
                   const optional<Tensor>& ref_, const optional<Tensor>& weight_, const optional<Tensor>& seq_coef_,
                   int64_t policy_term, double epsilon_low, double epsilon_high, double delta, double beta,
                   bool bias_correction_kl, double sapo_pos, double sapo_neg, bool compute_masked_rows,
                   const optional<Tensor>& entropy_weight_) {
    check_logits3d(logits);
    const int64_t n_seq = logits.size(0), length = logits.size(1), vocab = logits.size(2);
    for (const Tensor* t : {&index_, &mask_})
        TORCH_CHECK_VALUE(t->dim() == 2 && t->size(0) == n_seq && t->size(1) == keep_len, "grpo_fused: index and mask must be [",
                          n_seq, ", ", keep_len, "]");
    const c10::DeviceGuard guard(logits.device());
    const Tensor index = index_.contiguous().to(at::kLong), mask = f32c(mask_), advantages = f32c(advantages_);
    const optional<Tensor> old = f32c(old_), ref = f32c(ref_), weight = f32c(weight_), entropy_weight = f32c(entropy_weight_);
    check_token_shape("grpo_fused", "old_logp", old, n_seq, keep_len);
    check_token_shape("grpo_fused", "ref_logp", ref, n_seq, keep_len);
    check_token_shape("grpo_fused", "token_weight", weight, n_seq, keep_len);
    check_token_shape("grpo_fused", "entropy_weight", entropy_weight, n_seq, keep_len);
    const auto [sb, st] = advantage_strides("grpo_fused", advantages, n_seq, keep_len);
    const Tensor row_scale = f32c(row_scale_.reshape({n_seq}));
    const optional<Tensor> seq_coef = seq_coef_ ? f32c(optional<Tensor>(seq_coef_->reshape({n_seq}))) : std::nullopt;
    const Tensor logp = f32(logits, {n_seq, keep_len}), ent = f32(logits, {n_seq, keep_len}),
                 lse = f32(logits, {n_seq, keep_len}), dlogits = at::empty({n_seq, length, vocab}, logits.options());
    if (dlogits.numel() == 0) return {logp, ent, lse, dlogits};
    check_window(logits, keep_start, keep_len);
    check(trlk_grpo_fused_fwd_bwd(
        window(logits, keep_start), dtype_code(logits), n_seq, keep_len, vocab, logits.stride(0), logits.stride(1), iptr(index),
        float(temperature), fptr(old), fptr(ref), fptr(advantages), sb, st, fptr(mask), fptr(weight), fptr(seq_coef),
        fptr(row_scale), fptr(entropy_weight), int(policy_term), float(epsilon_low), float(epsilon_high), float(delta),
        float(beta), bias_correction_kl ? 1 : 0, float(sapo_pos), float(sapo_neg), out(logp), out(ent), out(lse),
        dlogits.mutable_data_ptr(), length, keep_start, dlogits.stride(0), dlogits.stride(1), compute_masked_rows ? 1 : 0,
        error_word(logits), stream_of(logits)));
    check_ids();
    return {logp, ent, lse, dlogits};
}

void scale_unless_one_(const Tensor& data, const Tensor& scale_) {
    TORCH_CHECK_VALUE(data.is_contiguous() && (data.scalar_type() == at::kBFloat16 || data.scalar_type() == at::kHalf ||
                                               data.scalar_type() == at::kFloat),
                      "scale_unless_one_: contiguous bf16 / fp16 / fp32 data expected");
    const c10::DeviceGuard guard(data.device());
    const Tensor scale = scale_.reshape({1}).to(data.options().dtype(at::kFloat));
    (void)operand(data);
    check(trlk_scale_unless_one(data.mutable_data_ptr(), dtype_code(data), data.numel(), fptr(scale), stream_of(data)));
}

// The loss of a pass that has written its gradient already.  Backward hands `dlogits` on as d loss / d logits, times what is left
// of the upstream gradient behind the factor `upstream` that the pass has applied: 1 as a rule, and then nothing is touched.
// A node of C++ and not of Python: the host takes longer than the device over a step of a small batch, and the device is idle
// from the metrics' copy to the next step's first launch, where this backward lies.  GRPO step, Python node -> this one, in us:
// bf16 [4, 256, 32000] 178-181 -> 137-154, [16, 509, 50257] 401-405 -> 365-380, [32, 1024, 151936] 2872 -> 2850.
class GradientInHand : public torch::autograd::Function<GradientInHand> {
  public:
    static Tensor forward(AutogradContext* ctx, const Tensor& loss, const Tensor& logits, const Tensor& dlogits,
                          const optional<Tensor>& upstream) {
        ctx->save_for_backward({dlogits, upstream ? *upstream : Tensor()});
        ctx->saved_data["consumed"] = false;
        ctx->set_materialize_grads(false);
        return loss.variable_data();  // (a tensor of its own on the same number, not a view: it may be changed in place)
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto saved = ctx->get_saved_variables();
        variable_list result(4);
        if (!grads[0].defined()) return result;
        // the gradient buffer is scaled in place and handed on: a second pass would scale it again
        TORCH_CHECK(!ctx->saved_data["consumed"].toBool(),
                    "grpo_loss_from_logits: its backward can run only once (the gradient written by the forward pass is handed to "
                    "the graph in place); call the function again instead of retain_graph=True");
        ctx->saved_data["consumed"] = true;
        {
            // in place: the buffer belongs to this node and is handed on once (the kernel returns at once for a scale of 1)
            const at::NoGradGuard no_grad;
            static const auto op = handle<decltype(scale_unless_one_)>("trl_amd::scale_unless_one_");
            op.call(saved[0], saved[1].defined() ? grads[0].to(at::kFloat) / saved[1] : grads[0]);
        }
        result[1] = saved[0];
        if (c10::GradMode::is_enabled() && grads[0].requires_grad()) {  // its own gradient is refused, not dropped
            const auto refuse = std::make_shared<torch::autograd::DelayedError>(
                "trying to differentiate twice: the gradient of grpo_loss_from_logits has no gradient of its own", 1);
            result[1] = (*refuse)({saved[0].detach().requires_grad_(true)})[0];
        }
        return result;
    }
};
Tensor gradient_in_hand(const Tensor& loss, const Tensor& logits, const Tensor& dlogits, const optional<Tensor>& upstream) {
    return GradientInHand::apply(loss, logits, dlogits, upstream);
}

Tensor grpo_log_values(const Tensor& metrics) {
    const c10::DeviceGuard guard(metrics.device());
    const Tensor values = f32(metrics, {TRLK_GRPO_LOG_VALUES});
    check(trlk_grpo_log_values(fptr(metrics), error_word(metrics), out(values), stream_of(metrics)));
    return values;
}

std::tuple<Tensor, Tensor> grpo_row_scale(const Tensor& mask, int64_t loss_type, double numerator, const optional<Tensor>& n_items,
                                          const optional<Tensor>& upstream, bool with_mask) {
    const int64_t B = mask.size(0), T = mask.size(1);
    for (const auto* t : {&n_items, &upstream})
        TORCH_CHECK_VALUE(!*t || (*t)->device() == mask.device(), "grpo_row_scale: the mask and the scalars must be on one GPU");
    int type = 0;
    switch (mask.scalar_type()) {
        case at::kBool:
        case at::kByte: type = 0; break;
        case at::kInt: type = 1; break;
        case at::kLong: type = 2; break;
        case at::kFloat: type = 3; break;
        default: TORCH_CHECK_TYPE(false, "grpo_row_scale: masks are bool, uint8, int32, int64 or float32");
    }
    const c10::DeviceGuard guard(mask.device());
    const Tensor mask_f = with_mask ? f32(mask, {B, T}) : f32(mask, {0}), scale = f32(mask, {B});
    check(trlk_grpo_row_scale(operand(mask), type, B, T, mask.stride(0), mask.stride(1), int(loss_type), float(numerator),
                              fptr(n_items), fptr(upstream), with_mask ? out(mask_f) : nullptr, out(scale), stream_of(mask)));
    return {mask_f, scale};
}

// ---- DPO ------------------------------------------------------------------------------------------------------------
Tensor4 dpo_loss(const Tensor& logp_, const Tensor& mask_, const Tensor& ref_chosen_, const Tensor& ref_rejected_, double beta) {
    TORCH_CHECK_VALUE(logp_.dim() == 2, "dpo_loss: per-token log-probs must be [B, T]");
    const int64_t B = logp_.size(0), T = logp_.size(1);
    TORCH_CHECK_VALUE(B % 2 == 0 && B >= 2, "dpo_loss: the batch must be [chosen; rejected], i.e. an even number of sequences");
    const c10::DeviceGuard guard(logp_.device());
    const Tensor logp = f32c(logp_), mask = f32c(mask_), ref_chosen = f32c(ref_chosen_), ref_rejected = f32c(ref_rejected_);
    TORCH_CHECK_VALUE(mask.dim() == 2 && mask.size(0) == B && mask.size(1) == T && ref_chosen.numel() == B / 2 &&
                          ref_rejected.numel() == B / 2,
                      "dpo_loss: mask must be [B, T] and the reference log-probs [B/2] each");
    const Tensor loss = f32(logp, {}), seq = f32(logp, {B}), metrics = f32(logp, {TRLK_DPO_NUM_METRICS}), dlogp = f32(logp, {B, T});
    check(trlk_dpo_loss(fptr(logp), fptr(mask), fptr(ref_chosen), fptr(ref_rejected), B, T, float(beta), out(seq), out(loss),
                        out(metrics), out(dlogp), stream_of(logp)));
    return {loss, seq, metrics, dlogp};
}
class DpoLoss : public torch::autograd::Function<DpoLoss> {
  public:
    static variable_list forward(AutogradContext* ctx, const Tensor& logp, const Tensor& mask, const Tensor& ref_chosen,
                                 const Tensor& ref_rejected, double beta) {
        variable_list result;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            static const auto op = handle<decltype(dpo_loss)>("trl_amd::dpo_loss");
            auto [loss, seq, metrics, dlogp] = op.call(logp, mask, ref_chosen, ref_rejected, beta);
            result = {loss, seq, metrics, dlogp};
        }
        ctx->save_for_backward({result[3], mask});
        ctx->saved_data["dtype"] = logp.scalar_type();
        ctx->set_materialize_grads(false);
        return result;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        variable_list result(5);
        const auto saved = ctx->get_saved_variables();
        Tensor g;
        if (grads[0].defined()) g = grads[0] * saved[0];
        if (grads[1].defined()) {
            const Tensor extra = grads[1].unsqueeze(1) * saved[1].ne(0).to(at::kFloat);
            g = g.defined() ? g + extra : extra;
        }
        if (g.defined()) result[0] = g.to(ctx->saved_data["dtype"].toScalarType());
        return result;
    }
};
Tensor4 dpo_loss_autograd(const Tensor& logp, const Tensor& mask, const Tensor& ref_chosen, const Tensor& ref_rejected, double beta) {
    if (needs_grad({&logp, &mask, &ref_chosen, &ref_rejected})) {
        const auto r = DpoLoss::apply(logp, mask, ref_chosen, ref_rejected, beta);
        return {r[0], r[1], r[2], r[3]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = handle<decltype(dpo_loss)>("trl_amd::dpo_loss");
    return op.call(logp, mask, ref_chosen, ref_rejected, beta);
}

Tensor dpo_log_values(const Tensor& entropy_, const Tensor& row_stats_, const Tensor& mask_, const Tensor& seq_logps_,
                      const Tensor& ref_chosen_, const Tensor& ref_rejected_, double beta) {
    const int64_t B = mask_.size(0), T = mask_.size(1), P = B / 2;
    TORCH_CHECK_VALUE(B % 2 == 0 && entropy_.numel() == B * T && row_stats_.numel() == 4 * B * T && seq_logps_.numel() == B,
                      "dpo_log_values: the shapes do not match");
    (void)operand(mask_);
    const c10::DeviceGuard guard(mask_.device());
    const Tensor entropy = f32c(entropy_), row_stats = f32c(row_stats_), mask = f32c(mask_), seq_logps = f32c(seq_logps_);
    const Tensor ref_chosen = f32c(ref_chosen_.expand({P})), ref_rejected = f32c(ref_rejected_.expand({P}));
    const Tensor values = f32(mask, {8 + 2 * B});
    if (B == 0) return values.zero_();
    const Tensor ws = f32(mask, {4 * B});
    check(trlk_dpo_log_values(fptr(entropy), fptr(row_stats), fptr(mask), B, T, fptr(seq_logps), fptr(ref_chosen),
                              fptr(ref_rejected), float(beta), error_word(mask), out(values), out(ws), stream_of(mask)));
    return values;
}
}  // namespace

TORCH_LIBRARY_FRAGMENT(trl_amd, m) {
    m.def("error_flag(int device_index) -> Tensor", error_flag);
    m.def("error_flags() -> Tensor[]", all_error_flags);
    m.def("logp_entropy_fwd(Tensor logits, Tensor index, float temperature, SymInt keep_start, SymInt keep_len, Tensor? row_mask) "
          "-> (Tensor, Tensor, Tensor)");
    m.def("logp_entropy_stats_fwd(Tensor logits, Tensor index, float temperature, SymInt keep_start, SymInt keep_len, "
          "Tensor? row_mask, bool sum_p2=True) -> (Tensor, Tensor, Tensor, Tensor)");
    m.def("logp_entropy_bwd(Tensor logits, Tensor index, float temperature, SymInt keep_start, SymInt keep_len, Tensor lse, "
          "Tensor? entropy, Tensor? g_logp, Tensor? g_entropy) -> Tensor");
    m.def("grpo_loss(Tensor logp, Tensor? old_logp, Tensor? ref_logp, Tensor? entropy, Tensor advantages, Tensor mask, "
          "Tensor? token_weight, Tensor? entropy_mask, Tensor? dapo_normalizer, int loss_type, float epsilon_low, "
          "float epsilon_high, float delta, float beta, bool use_bias_correction_kl, float grad_accum_steps, "
          "float dr_grpo_denominator, float num_processes, float entropy_coef, int policy_term=0, bool sequence_level=False, "
          "Tensor? seq_coef=None, float sapo_temperature_pos=1.0, float sapo_temperature_neg=1.05) "
          "-> (Tensor, Tensor, Tensor, Tensor)");
    m.def("grpo_fused(Tensor logits, Tensor index, float temperature, SymInt keep_start, SymInt keep_len, Tensor mask, "
          "Tensor advantages, Tensor row_scale, Tensor? old_logp, Tensor? ref_logp, Tensor? token_weight, Tensor? seq_coef, "
          "int policy_term, float epsilon_low, float epsilon_high, float delta, float beta, bool use_bias_correction_kl, "
          "float sapo_temperature_pos, float sapo_temperature_neg, bool compute_masked_rows=False, Tensor? entropy_weight=None) "
          "-> (Tensor, Tensor, Tensor, Tensor)");
    m.def("scale_unless_one_(Tensor(a!) data, Tensor scale) -> ()");
    m.def("gradient_in_hand(Tensor(a) loss, Tensor logits, Tensor dlogits, Tensor? upstream) -> Tensor(a)", gradient_in_hand);
    m.def("grpo_log_values(Tensor metrics) -> Tensor");
    m.def("grpo_row_scale(Tensor mask, int loss_type, float numerator, Tensor? n_items, Tensor? upstream, bool with_mask) "
          "-> (Tensor, Tensor)");
    m.def("dpo_loss(Tensor token_logp, Tensor mask, Tensor ref_chosen, Tensor ref_rejected, float beta) "
          "-> (Tensor, Tensor, Tensor, Tensor)");
    m.def("dpo_log_values(Tensor entropy, Tensor row_stats, Tensor mask, Tensor seq_logps, Tensor ref_chosen, "
          "Tensor ref_rejected, float beta) -> Tensor");
}
TORCH_LIBRARY_IMPL(trl_amd, CUDA, m) {
    m.impl("logp_entropy_fwd", logp_entropy_fwd);
    m.impl("logp_entropy_stats_fwd", logp_entropy_stats_fwd);
    m.impl("logp_entropy_bwd", logp_entropy_bwd);
    m.impl("grpo_loss", grpo_loss);
    m.impl("grpo_fused", grpo_fused);
    m.impl("scale_unless_one_", scale_unless_one_);
    m.impl("grpo_log_values", grpo_log_values);
    m.impl("grpo_row_scale", grpo_row_scale);
    m.impl("dpo_loss", dpo_loss);
    m.impl("dpo_log_values", dpo_log_values);
}
TORCH_LIBRARY_IMPL(trl_amd, Autograd, m) {
    m.impl("logp_entropy_fwd", logp_entropy_fwd_autograd);
    m.impl("logp_entropy_stats_fwd", logp_entropy_stats_fwd_autograd);
    m.impl("grpo_loss", grpo_loss_autograd);
    m.impl("dpo_loss", dpo_loss_autograd);
    for (const char* name : {"logp_entropy_bwd", "grpo_row_scale", "dpo_log_values"})
        m.impl(name, torch::autograd::autogradNotImplementedFallback());
    // (these hand out a gradient or scale one in place: their results belong to no graph, whatever the logits require)
    for (const char* name : {"grpo_fused", "scale_unless_one_"}) m.impl(name, torch::CppFunction::makeFallthrough());
}
