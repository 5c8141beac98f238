// Autograd nodes of the fused step and of the packed attention, in C++: what a call spends on the host is then a few
// allocations and the launches themselves.  The same nodes written in Python cost 40 us of a forward and, because
// the autograd engine runs them on its own thread under the interpreter lock, 100 us of a backward - more than the
// kernels of a small batch take.  Nothing is computed here: every number comes out of libfgrpo, whose entry points
// are handed over by address (one copy of the library per process, the one the Python layer loaded).
// Shapes, types and devices are checked before any pointer is taken; errors are RuntimeErrors.
#include <torch/extension.h>

#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <optional>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/fgrpo.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

#define FGRPO_ENTRY(name) decltype(&::name) name = nullptr
struct Api {
  FGRPO_ENTRY(fgrpo_last_error);
  FGRPO_ENTRY(fgrpo_logprob_fwd_workspace);
  FGRPO_ENTRY(fgrpo_logprob_fwd);
  FGRPO_ENTRY(fgrpo_lmhead_bwd_workspace);
  FGRPO_ENTRY(fgrpo_lmhead_bwd);
  FGRPO_ENTRY(fgrpo_keep_supported);
  FGRPO_ENTRY(fgrpo_logits_keep_bytes);
  FGRPO_ENTRY(fgrpo_logprob_fwd_keep);
  FGRPO_ENTRY(fgrpo_lmhead_bwd_kept_workspace);
  FGRPO_ENTRY(fgrpo_lmhead_bwd_kept);
  FGRPO_ENTRY(fgrpo_loss_fwd_workspace);
  FGRPO_ENTRY(fgrpo_loss_fwd);
  FGRPO_ENTRY(fgrpo_loss_prepare);
  FGRPO_ENTRY(fgrpo_grpo_step_chunked_supported);
  FGRPO_ENTRY(fgrpo_grpo_step_chunked_workspace);
  FGRPO_ENTRY(fgrpo_grpo_step_chunked);
  FGRPO_ENTRY(fgrpo_scale_gradients);
  FGRPO_ENTRY(fgrpo_shift_labels);
  FGRPO_ENTRY(fgrpo_varlen_attn_workspace_len);
  FGRPO_ENTRY(fgrpo_varlen_attn_fwd_len);
  FGRPO_ENTRY(fgrpo_varlen_attn_bwd_len);
} api;

void init(const std::unordered_map<std::string, uint64_t>& at) {
  auto set = [&](const char* name, auto& slot) {
    const auto it = at.find(name);
    TORCH_CHECK(it != at.end() && it->second != 0, "fgrpo: entry point ", name, " missing");
    slot = reinterpret_cast<std::remove_reference_t<decltype(slot)>>(it->second);
  };
#define FGRPO_SET(name) set(#name, api.name)
  FGRPO_SET(fgrpo_last_error);
  FGRPO_SET(fgrpo_logprob_fwd_workspace);
  FGRPO_SET(fgrpo_logprob_fwd);
  FGRPO_SET(fgrpo_lmhead_bwd_workspace);
  FGRPO_SET(fgrpo_lmhead_bwd);
  FGRPO_SET(fgrpo_keep_supported);
  FGRPO_SET(fgrpo_logits_keep_bytes);
  FGRPO_SET(fgrpo_logprob_fwd_keep);
  FGRPO_SET(fgrpo_lmhead_bwd_kept_workspace);
  FGRPO_SET(fgrpo_lmhead_bwd_kept);
  FGRPO_SET(fgrpo_loss_fwd_workspace);
  FGRPO_SET(fgrpo_loss_fwd);
  FGRPO_SET(fgrpo_loss_prepare);
  FGRPO_SET(fgrpo_grpo_step_chunked_supported);
  FGRPO_SET(fgrpo_grpo_step_chunked_workspace);
  FGRPO_SET(fgrpo_grpo_step_chunked);
  FGRPO_SET(fgrpo_scale_gradients);
  FGRPO_SET(fgrpo_shift_labels);
  FGRPO_SET(fgrpo_varlen_attn_workspace_len);
  FGRPO_SET(fgrpo_varlen_attn_fwd_len);
  FGRPO_SET(fgrpo_varlen_attn_bwd_len);
}

void check(int rc, const char* what) { TORCH_CHECK(rc == 0, "fgrpo ", what, " failed (", rc, "): ", api.fgrpo_last_error()); }

// The tensors' device made current for the scope, as the launches go to that device's current stream.
struct OnDevice {
  c10::DeviceIndex prev, dev;
  explicit OnDevice(const Tensor& t) : dev(t.device().index()) {
    prev = c10::hip::current_device();
    if (prev != dev) c10::hip::set_device(dev);
  }
  ~OnDevice() {
    if (prev != dev) c10::hip::set_device(prev);
  }
  void* stream() const { return c10::hip::getCurrentHIPStream(dev).stream(); }
};

template <class... T>
void require_one_gpu(const Tensor& first, const T&... rest) {
  auto one = [&](const Tensor& t) {
    if (!t.defined()) return;
    TORCH_CHECK(t.is_cuda(), "fgrpo: tensors must live on the GPU (the HIP path has no CPU fallback)");
    TORCH_CHECK(t.device() == first.device(), "fgrpo: all tensors must be on the same device");
  };
  one(first);
  (one(rest), ...);
}

Tensor opt(const std::optional<Tensor>& t) { return t.has_value() ? *t : Tensor(); }
const void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }
bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// Contiguous and 16-byte aligned (a sliced view can start anywhere)
Tensor in_place(const Tensor& t) {
  Tensor c = t.detach().contiguous();
  return aligned16(c) ? c : c.clone();
}
Tensor per_token(const Tensor& t, int64_t n, const char* name) {
  if (!t.defined()) return t;
  Tensor f = t.detach().reshape({-1});
  TORCH_CHECK(f.numel() == n, "fgrpo: ", name, " has ", f.numel(), " elements, expected ", n);
  return f.scalar_type() == at::kFloat && f.is_contiguous() ? f : f.to(at::kFloat).contiguous();
}
Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)(bytes < 256 ? 256 : bytes)}, like.options().dtype(at::kByte).requires_grad(false));
}
int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return FGRPO_BF16;
  TORCH_CHECK(t.scalar_type() == at::kFloat, "fgrpo: unsupported dtype ", t.scalar_type(), " (bf16 and fp32 only)");
  return FGRPO_F32;
}
float clamp_f(double x) { return (float)(x > 3.0e38 ? 3.0e38 : x < -3.0e38 ? -3.0e38 : x); }

// ---------------------------------------------------------------------------------------------- the fused step
enum GradMode { kNone = 0, kRecompute = 1, kWhole = 2, kChunked = 3 };

struct StepArgs {
  Tensor labels, old_lp, adv, ref_lp, cu;      // shifted labels; per-token inputs; segment boundaries (sample mean)
  double inv_temp, clip_low, clip_high, clip_c, kl_beta, denom;
  bool by_sample;
  int64_t panel_hint;
  int mode, chunk_tokens;
  bool need_h, need_w, need_b;
};

struct Grads {
  Tensor dh, dw, db;
};

// Gradients of the projection by the recomputing pair or on the kept numerators, given g = d loss / d lp.
Grads lmhead_backward(const Tensor& h, const Tensor& w, const Tensor& b, const Tensor& y, const Tensor& lse, const Tensor& g,
                      const Tensor& gout, double inv_temp, int64_t hint, const Tensor& kept, bool nh, bool nw, bool nb) {
  const int T = (int)h.size(0), H = (int)h.size(1), V = (int)w.size(0), code = dtype_code(w);
  Grads r;
  if (nh) r.dh = at::empty_like(h, at::MemoryFormat::Contiguous);
  if (nw) r.dw = at::empty_like(w, at::MemoryFormat::Contiguous);
  if (nb && b.defined()) r.db = at::empty({V}, w.options().requires_grad(false));
  if (!r.dh.defined() && !r.dw.defined() && !r.db.defined()) return r;
  Tensor scale;
  if (gout.defined()) scale = gout.detach().reshape({-1}).to(at::kFloat).contiguous();
  OnDevice d(h);
  if (kept.defined()) {
    Tensor ws = workspace(api.fgrpo_lmhead_bwd_kept_workspace(T, H, V, code), h);
    check(api.fgrpo_lmhead_bwd_kept(ptr(h), ptr(w), ptr(b), y.data_ptr<int64_t>(), fptr(lse), fptr(g), fptr(scale),
                                    (float)inv_temp, T, H, V, code, kept.data_ptr(), (size_t)kept.numel(),
                                    const_cast<void*>(ptr(r.dh)), const_cast<void*>(ptr(r.dw)), const_cast<void*>(ptr(r.db)),
                                    ws.data_ptr(), (size_t)ws.numel(), d.stream()),
          "lmhead_bwd_kept");
  } else {
    Tensor ws = workspace(api.fgrpo_lmhead_bwd_workspace(T, H, V, code, hint), h);
    check(api.fgrpo_lmhead_bwd(ptr(h), ptr(w), ptr(b), y.data_ptr<int64_t>(), fptr(lse), fptr(g), fptr(scale),
                               (float)inv_temp, T, H, V, code, const_cast<void*>(ptr(r.dh)),
                               const_cast<void*>(ptr(r.dw)), const_cast<void*>(ptr(r.db)), hint, ws.data_ptr(),
                               (size_t)ws.numel(), d.stream()),
          "lmhead_bwd");
  }
  return r;
}

struct StepOut {
  Tensor loss, lp, ent, lse, g, lr, c1, l1, l2, kept;
  Grads grads;
};

StepOut step_forward(const Tensor& h, const Tensor& w, const Tensor& b, const StepArgs& a) {
  const int T = (int)h.size(0), H = (int)h.size(1), V = (int)w.size(0), code = dtype_code(w);
  const auto f32 = h.options().dtype(at::kFloat).requires_grad(false);
  OnDevice d(h);
  void* st = d.stream();
  StepOut o;
  for (Tensor* t : {&o.lp, &o.ent, &o.lse, &o.g, &o.lr, &o.c1, &o.l1, &o.l2}) *t = at::empty({T}, f32);
  Tensor scal = at::empty({4}, f32);
  o.loss = at::empty({}, f32);
  const float it = (float)a.inv_temp;
  const int nseq = a.cu.defined() ? (int)a.cu.numel() - 1 : 0;
  const int agg = a.by_sample ? FGRPO_AGG_SAMPLE_MEAN : FGRPO_AGG_TOKEN_MEAN;
  const int64_t* y = a.labels.data_ptr<int64_t>();
  const int32_t* cu = a.cu.defined() ? a.cu.data_ptr<int32_t>() : nullptr;
  if (a.mode == kChunked) {
    // normalisers first (per-token weights and segment counts only for the sample mean), then the whole step
    Tensor pre = at::empty({4}, f32.dtype(at::kDouble)), tokw, segc;
    if (a.by_sample) {
      tokw = at::empty({T}, f32);
      segc = at::empty({nseq > 0 ? nseq : 1}, f32.dtype(at::kInt));
    }
    check(api.fgrpo_loss_prepare(y, a.by_sample ? cu : nullptr, a.by_sample ? nseq : 0, T, agg, a.denom, fptr(tokw),
                                 segc.defined() ? segc.data_ptr<int32_t>() : nullptr, pre.data_ptr<double>(), st),
          "loss_prepare");
    if (a.need_h) o.grads.dh = at::empty_like(h, at::MemoryFormat::Contiguous);
    if (a.need_w) o.grads.dw = at::empty_like(w, at::MemoryFormat::Contiguous);
    if (a.need_b && b.defined()) o.grads.db = at::empty({V}, w.options().requires_grad(false));
    Tensor ws = workspace(api.fgrpo_grpo_step_chunked_workspace(T, H, V, code, a.chunk_tokens), h);
    check(api.fgrpo_grpo_step_chunked(ptr(h), ptr(w), ptr(b), y, fptr(a.old_lp), fptr(a.ref_lp), fptr(a.adv), fptr(tokw),
                                      pre.data_ptr<double>(), it, T, H, V, code, clamp_f(a.clip_low), clamp_f(a.clip_high),
                                      clamp_f(a.clip_c), clamp_f(a.kl_beta), a.chunk_tokens, fptr(o.lp), fptr(o.ent),
                                      fptr(o.lse), fptr(o.loss), fptr(o.g), fptr(o.lr), fptr(o.c1), fptr(o.l1), fptr(o.l2),
                                      fptr(scal), const_cast<void*>(ptr(o.grads.dh)), const_cast<void*>(ptr(o.grads.dw)),
                                      const_cast<void*>(ptr(o.grads.db)), ws.data_ptr(), (size_t)ws.numel(), st),
          "grpo_step_chunked");
    return o;
  }
  {
    Tensor ws = workspace(api.fgrpo_logprob_fwd_workspace(T, H, V, code), h);
    if (a.mode == kWhole) {
      o.kept = workspace(api.fgrpo_logits_keep_bytes(T, V), h);
      check(api.fgrpo_logprob_fwd_keep(ptr(h), ptr(w), ptr(b), y, it, T, H, V, code, fptr(o.lp), fptr(o.ent), fptr(o.lse),
                                       o.kept.data_ptr(), (size_t)o.kept.numel(), ws.data_ptr(), (size_t)ws.numel(), st),
            "logprob_fwd_keep");
    } else {
      check(api.fgrpo_logprob_fwd(ptr(h), ptr(w), ptr(b), y, it, T, H, V, code, fptr(o.lp), fptr(o.ent), fptr(o.lse),
                                  ws.data_ptr(), (size_t)ws.numel(), st),
            "logprob_fwd");
    }
  }
  Tensor ws = workspace(api.fgrpo_loss_fwd_workspace(T, nseq), h);
  check(api.fgrpo_loss_fwd(fptr(o.lp), fptr(a.old_lp), fptr(a.ref_lp), fptr(a.adv), y, cu, nseq, T, clamp_f(a.clip_low),
                           clamp_f(a.clip_high), clamp_f(a.clip_c), clamp_f(a.kl_beta), agg, a.denom, fptr(o.loss),
                           fptr(o.g), fptr(o.lr), fptr(o.c1), fptr(o.l1), fptr(o.l2), fptr(scal), ws.data_ptr(),
                           (size_t)ws.numel(), st),
        "loss_fwd");
  return o;
}

// (loss, entropy, log_ratio, clip1, unclipped, clipped, lp); only the loss carries a gradient.  The three per-token inputs
// get none, and are read in the form StepArgs holds them in; they are inputs of the node so that autograd sees them: a
// forward-mode tangent on one is refused, not dropped, and one that requires a gradient makes the loss require one.
struct FusedStep : torch::autograd::Function<FusedStep> {
  static variable_list forward(AutogradContext* ctx, const Tensor& hidden, const Tensor& weight,
                               const std::optional<Tensor>& bias_, const std::optional<Tensor>& /*old_lp*/,
                               const Tensor& /*adv*/, const std::optional<Tensor>& /*ref_lp*/, const StepArgs& a) {
    const Tensor bias = opt(bias_);
    const Tensor h = in_place(hidden), w = in_place(weight);
    const Tensor b = bias.defined() ? bias.detach().to(w.scalar_type()).contiguous() : Tensor();
    StepOut o = step_forward(h, w, b, a);
    // the chunked step leaves the gradients of the loss itself; the first backward scales them, a second recomputes
    ctx->saved_data["dh"] = o.grads.dh;
    ctx->saved_data["dw"] = o.grads.dw;
    ctx->saved_data["db"] = o.grads.db;
    ctx->saved_data["kept"] = o.kept;
    ctx->saved_data["fresh"] = a.mode == kChunked;
    ctx->saved_data["inv_temp"] = a.inv_temp;
    ctx->saved_data["hint"] = a.panel_hint;
    ctx->saved_data["nh"] = a.need_h;
    ctx->saved_data["nw"] = a.need_w;
    ctx->saved_data["nb"] = a.need_b;
    ctx->save_for_backward({hidden, weight, bias.defined() ? bias : Tensor(), a.labels, o.lse, o.g});
    ctx->mark_non_differentiable({o.ent, o.lr, o.c1, o.l1, o.l2, o.lp});
    ctx->set_materialize_grads(false);
    return {o.loss, o.ent, o.lr, o.c1, o.l1, o.l2, o.lp};
  }
  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const Tensor gout = gs[0];
    if (!gout.defined()) return variable_list(7);
    auto& sd = ctx->saved_data;
    if (sd["fresh"].toBool()) {
      sd["fresh"] = false;
      Grads r{sd["dh"].toTensor(), sd["dw"].toTensor(), sd["db"].toTensor()};
      sd["dh"] = Tensor(), sd["dw"] = Tensor(), sd["db"] = Tensor();
      const Tensor scale = gout.detach().reshape({-1}).to(at::kFloat).contiguous();
      OnDevice d(scale);
      auto count = [](const Tensor& t) { return t.defined() ? (long long)t.numel() : 0LL; };
      auto data = [](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
      check(api.fgrpo_scale_gradients(data(r.dh), count(r.dh), data(r.dw), count(r.dw), data(r.db), count(r.db), FGRPO_BF16,
                                      fptr(scale), d.stream()),
            "scale_gradients");
      return {r.dh, r.dw, r.db, Tensor(), Tensor(), Tensor(), Tensor()};
    }
    const auto saved = ctx->get_saved_variables();
    const Tensor kept = sd["kept"].toTensor();
    sd["kept"] = Tensor();                       // released by the first backward
    const Tensor h = in_place(saved[0]), w = in_place(saved[1]);
    const Tensor b = saved[2].defined() ? saved[2].detach().to(w.scalar_type()).contiguous() : Tensor();
    Grads r = lmhead_backward(h, w, b, saved[3], saved[4], saved[5], gout, sd["inv_temp"].toDouble(), sd["hint"].toInt(),
                              kept, sd["nh"].toBool(), sd["nw"].toBool(), sd["nb"].toBool());
    return {r.dh, r.dw, r.db, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// labels [..., L] -> next-token targets, -100 in the last column: one launch on plain contiguous int64 memory; anything else
// (wrapped by a function transform, seen by a dispatch mode, strided, rows past 32 bits) by torch's own operations
Tensor shift_labels(const Tensor& labels) {
  const bool wrapped = labels.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched,
      c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Python}));
  if (wrapped || c10::impl::TorchDispatchModeTLS::any_modes_set() || !labels.is_cuda() || labels.scalar_type() != at::kLong ||
      labels.dim() == 0 || !labels.is_contiguous() || labels.size(-1) >= (1LL << 31))
    return at::constant_pad_nd(labels, {0, 1}, -100).slice(-1, 1).contiguous();
  Tensor out = at::empty_like(labels);
  if (labels.numel() == 0) return out;
  OnDevice d(labels);
  const int64_t L = labels.size(-1);
  check(api.fgrpo_shift_labels(labels.data_ptr<int64_t>(), labels.numel() / L, (int)L, out.data_ptr<int64_t>(), d.stream()), "shift_labels");
  return out;
}

// mode: 0 "auto", 1 "recompute", 2 "whole", 3 "chunked" (what the gradients come from, where one is wanted)
variable_list fused_step(const Tensor& hidden, const Tensor& weight, const std::optional<Tensor>& bias_, const Tensor& labels,
                         const std::optional<Tensor>& old_lp, const Tensor& adv, const std::optional<Tensor>& ref_lp,
                         const std::optional<Tensor>& cu, double inv_temp, double clip_low, double clip_high, double clip_c,
                         double kl_beta, bool by_sample, double denom, int64_t panel_hint, int mode, int64_t chunk_tokens,
                         int64_t keep_whole_max_bytes) {
  const Tensor bias = opt(bias_);
  require_one_gpu(hidden, weight, bias, labels, adv);
  TORCH_CHECK(hidden.dim() == 2 && weight.dim() == 2 && hidden.size(1) == weight.size(1), "fgrpo: hidden ", hidden.sizes(),
              " / weight ", weight.sizes(), " mismatch");
  TORCH_CHECK(hidden.scalar_type() == weight.scalar_type(), "fgrpo: hidden and weight must share a dtype");
  const int64_t T = hidden.size(0), H = hidden.size(1), V = weight.size(0);
  TORCH_CHECK(T > 0 && T < (1LL << 31) && H < (1LL << 31) && V < (1LL << 31), "fgrpo: T=", T, " H=", H, " V=", V);
  TORCH_CHECK(!bias.defined() || bias.numel() == V, "fgrpo: bias must have V elements");
  TORCH_CHECK(!by_sample || cu.has_value(), "fgrpo: loss_agg_mode='sample_mean' needs cu_seqlens");
  const int code = dtype_code(weight);
  StepArgs a;
  a.labels = labels.reshape({-1}).to(at::kLong).contiguous();
  TORCH_CHECK(a.labels.numel() == T, "fgrpo: labels must have one entry per token");
  a.old_lp = per_token(opt(old_lp), T, "old_logprobs");
  a.adv = per_token(adv, T, "advantages");
  a.ref_lp = per_token(opt(ref_lp), T, "ref_logprobs");
  if (cu.has_value()) a.cu = cu->to(hidden.device(), at::kInt).contiguous();
  require_one_gpu(hidden, a.old_lp, a.ref_lp, a.cu);
  a.inv_temp = inv_temp, a.clip_low = clip_low, a.clip_high = clip_high, a.clip_c = clip_c, a.kl_beta = kl_beta;
  a.denom = denom, a.by_sample = by_sample, a.panel_hint = panel_hint, a.chunk_tokens = (int)chunk_tokens;
  const bool on = at::GradMode::is_enabled();
  a.need_h = on && hidden.requires_grad();
  a.need_w = on && weight.requires_grad();
  a.need_b = on && bias.defined() && bias.requires_grad();
  const bool wanted = a.need_h || a.need_w || a.need_b;
  a.mode = kNone;
  if (wanted) {
    a.mode = kRecompute;
    const bool chunked_ok = (mode == 0 || mode == 3) && code == FGRPO_BF16 &&
                            api.fgrpo_grpo_step_chunked_supported((int)T, (int)H, (int)V, code, (int)chunk_tokens);
    TORCH_CHECK(mode != 3 || chunked_ok, "fgrpo: keep_logits='chunked' but T=", T, " H=", H, " V=", V, " ", weight.scalar_type(),
                " is not supported");
    if (chunked_ok) {
      a.mode = kChunked;
    } else if (mode == 0 || mode == 2) {
      const bool keep_ok = code == FGRPO_BF16 && api.fgrpo_keep_supported((int)T, (int)H, (int)V, code);
      TORCH_CHECK(mode != 2 || keep_ok, "fgrpo: keep_logits=True but T=", T, " H=", H, " V=", V, " ", weight.scalar_type(),
                  " is not supported");
      if (mode == 2 || (keep_ok && (int64_t)api.fgrpo_logits_keep_bytes((int)T, (int)V) <= keep_whole_max_bytes)) a.mode = kWhole;
    }
  }
  return FusedStep::apply(hidden, weight, bias_, old_lp, adv, ref_lp, a);
}

// ---------------------------------------------------------------------------------------------- packed attention
// [T, H, D] bf16 view the kernels can read in place; anything else is copied once
Tensor attn_operand(const Tensor& t, const char* name) {
  TORCH_CHECK(t.dim() == 3, "fgrpo: ", name, " must be [tokens, heads, head_dim], got ", t.sizes());
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, "fgrpo: ", name, " must be bf16, got ", t.scalar_type());
  const bool ok = t.stride(2) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(0) > 0 && t.stride(1) > 0 && aligned16(t);
  return ok ? t.detach() : in_place(t);
}
int64_t bounds_numel(int64_t T) { return 2 * T + 2 * ((T + 127) / 128) + (T + 63) / 64 + (T + 31) / 32; }

// scratch of a call on a batch with few tiles; none elsewhere
Tensor attn_workspace(const Tensor& q, const Tensor& cu, int max_len, int Hkv, bool causal, bool backward) {
  const size_t n = api.fgrpo_varlen_attn_workspace_len((int)q.size(0), (int)cu.numel() - 1, max_len, (int)q.size(1), Hkv, (int)q.size(2), causal, backward);
  return n > 0 ? workspace(n, q) : Tensor();
}

struct AttnArgs {
  Tensor cu, bounds;
  bool bounds_valid, causal;
  double scale;
  int max_len;                 // the longest segment, 0: not known
};

struct VarlenAttention : torch::autograd::Function<VarlenAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_, AttnArgs a) {
    const Tensor q = attn_operand(q_, "q"), k = attn_operand(k_, "k"), v = attn_operand(v_, "v");
    const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2), Hkv = (int)k.size(1);
    const auto o = q.options().requires_grad(false);
    Tensor out = at::empty({T, Hq, D}, o), lse = at::empty({Hq, T}, o.dtype(at::kFloat));
    if (!a.bounds_valid) a.bounds = at::empty({bounds_numel(T)}, o.dtype(at::kInt));
    OnDevice d(q);
    const Tensor ws = attn_workspace(q, a.cu, a.max_len, Hkv, a.causal, false);
    if (T > 0)
      check(api.fgrpo_varlen_attn_fwd_len(ptr(q), ptr(k), ptr(v), q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0),
                                      v.stride(1), a.cu.data_ptr<int32_t>(), (int)a.cu.numel() - 1, a.max_len, T, Hq, Hkv, D,
                                      (float)a.scale, a.causal, out.data_ptr(), fptr(lse), a.bounds.data_ptr<int32_t>(),
                                      a.bounds_valid, ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? (size_t)ws.numel() : 0, d.stream()),
            "varlen_attn_fwd");
    if (ctx) {
      ctx->save_for_backward({q_, k_, v_, out, lse, a.cu, a.bounds});
      ctx->saved_data["scale"] = a.scale;
      ctx->saved_data["causal"] = a.causal;
      ctx->saved_data["max_len"] = (int64_t)a.max_len;
    }
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const auto s = ctx->get_saved_variables();
    const Tensor q = attn_operand(s[0], "q"), k = attn_operand(s[1], "k"), v = attn_operand(s[2], "v");
    const Tensor out = s[3], lse = s[4], cu = s[5], bounds = s[6];
    const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2), Hkv = (int)k.size(1);
    TORCH_CHECK(gs[0].sizes() == out.sizes(), "fgrpo: dout must be ", out.sizes(), ", got ", gs[0].sizes());
    const Tensor dout = in_place(gs[0].to(at::kBFloat16));
    require_one_gpu(q, dout);
    const auto o = q.options().requires_grad(false);
    Tensor dq = at::empty({T, Hq, D}, o), dk = at::empty({T, Hkv, D}, o), dv = at::empty({T, Hkv, D}, o);
    Tensor delta = at::empty({Hq, T}, o.dtype(at::kFloat));
    const int max_len = (int)ctx->saved_data["max_len"].toInt();
    OnDevice d(q);
    const Tensor ws = attn_workspace(q, cu, max_len, Hkv, ctx->saved_data["causal"].toBool(), true);
    if (T > 0)
      check(api.fgrpo_varlen_attn_bwd_len(ptr(dout), ptr(q), ptr(k), ptr(v), ptr(out), fptr(lse), q.stride(0), q.stride(1),
                                      k.stride(0), k.stride(1), v.stride(0), v.stride(1), cu.data_ptr<int32_t>(),
                                      (int)cu.numel() - 1, max_len, T, Hq, Hkv, D, (float)ctx->saved_data["scale"].toDouble(),
                                      ctx->saved_data["causal"].toBool(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                      fptr(delta), bounds.data_ptr<int32_t>(), 1, ws.defined() ? ws.data_ptr() : nullptr,
                                      ws.defined() ? (size_t)ws.numel() : 0, d.stream()),
            "varlen_attn_bwd");
    return {dq, dk, dv, Tensor()};
  }
};

Tensor varlen_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu, const std::optional<double>& scale,
                        bool causal, const std::optional<Tensor>& bounds, int64_t max_len) {
  require_one_gpu(q, k, v, cu);
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(2) == q.size(2),
              "fgrpo: q ", q.sizes(), ", k ", k.sizes(), ", v ", v.sizes(), " do not fit together");
  const int64_t T = q.size(0);
  TORCH_CHECK(T < (1LL << 31), "fgrpo: packed batch longer than 2^31 tokens");
  AttnArgs a;
  a.cu = cu.to(at::kInt).contiguous();
  a.causal = causal;
  a.scale = scale.has_value() ? *scale : 1.0 / std::sqrt((double)q.size(2));
  a.max_len = (int)std::min<int64_t>(std::max<int64_t>(max_len, 0), T);
  a.bounds_valid = bounds.has_value();
  if (a.bounds_valid) {
    a.bounds = *bounds;
    TORCH_CHECK(a.bounds.scalar_type() == at::kInt && a.bounds.numel() == bounds_numel(T) && a.bounds.device() == q.device() &&
                    a.bounds.is_contiguous(),
                "fgrpo: bounds does not come from an attention call of this shape");
  }
  // a forward-mode tangent goes to the node as well, which refuses it (also where gradients are off)
  auto dual = [](const Tensor& t) { return t._fw_grad(0).defined(); };
  const bool wanted = (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) ||
                      dual(q) || dual(k) || dual(v);
  return wanted ? VarlenAttention::apply(q, k, v, a) : VarlenAttention::forward(nullptr, q, k, v, a);
}

// The numbers of a Python list or tuple into a host array of its length, int64 or float32: what packing a batch spends
// most of its time on (4 ns an entry; numpy.fromiter 20).  Only plain ints into int64 and plain floats into float32, in their
// ranges, are taken: false, with the array partly written, for anything else, and numpy's rules decide.
struct HostArray {
  Py_buffer b;
  bool ints = false, floats = false;
  Py_ssize_t n = 0;
  explicit HostArray(const py::object& array) {
    if (PyObject_GetBuffer(array.ptr(), &b, PyBUF_WRITABLE | PyBUF_FORMAT | PyBUF_C_CONTIGUOUS) != 0) throw py::error_already_set();
    if (b.ndim != 1 || !b.format) return;
    const std::string format = b.format;
    n = b.shape ? b.shape[0] : 0;
    ints = b.itemsize == 8 && (format == "l" || format == "q");
    floats = b.itemsize == 4 && format == "f";
  }
  ~HostArray() { PyBuffer_Release(&b); }
  HostArray(const HostArray&) = delete;
  // `seq` into the array from entry `at` on
  bool read(PyObject* seq, Py_ssize_t at, Py_ssize_t count) const {
    if ((!ints && !floats) || (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq))) return false;
    if (PySequence_Fast_GET_SIZE(seq) != count || at < 0 || count > n - at) return false;
    PyObject* const* const src = PySequence_Fast_ITEMS(seq);      // nothing below runs Python code, so the list stays as it is
    if (ints) {
      int64_t* const out = (int64_t*)b.buf + at;
      for (Py_ssize_t i = 0; i < count; ++i) {
        int overflow = 0;
        if (!PyLong_CheckExact(src[i])) return false;
        out[i] = PyLong_AsLongLongAndOverflow(src[i], &overflow);
        if (overflow) return false;
      }
      return true;
    }
    float* const out = (float*)b.buf + at;
    for (Py_ssize_t i = 0; i < count; ++i) {
      if (!PyFloat_CheckExact(src[i])) return false;
      const double x = PyFloat_AS_DOUBLE(src[i]);
      out[i] = (float)x;
      if (std::isinf(out[i]) && !std::isinf(x)) return false;
    }
    return true;
  }
};
// Several of them, one behind the other, `lens` entries each; returns the places of those that were not taken.  One call a
// field: a batch of 16 samples made 80, two thirds of whose time was the way here.
std::vector<int64_t> fill_lists(py::object array, const py::list& lists, const std::vector<int64_t>& lens) {
  const HostArray dst(array);
  std::vector<int64_t> left;
  Py_ssize_t at = 0;
  for (size_t i = 0; i < lens.size(); ++i) {
    if (lens[i] < 0 || i >= lists.size() || !dst.read(lists[i].ptr(), at, (Py_ssize_t)lens[i])) left.push_back((int64_t)i);
    if (lens[i] > 0) at += (Py_ssize_t)lens[i];
  }
  return left;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "autograd nodes over libfgrpo";
  m.def("init", &init);
  m.def("fill_lists", &fill_lists);
  // without the interpreter lock: a call may wait, for memory or for room in a full launch queue, and other threads run
  m.def("shift_labels", &shift_labels, py::call_guard<py::gil_scoped_release>());
  m.def("fused_step", &fused_step, py::call_guard<py::gil_scoped_release>());
  m.def("varlen_attention", &varlen_attention, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("cu"), py::arg("scale"), py::arg("causal"),
        py::arg("bounds"), py::arg("max_len") = 0, py::call_guard<py::gil_scoped_release>());
}
