// The differentiable operators of a block as C++ autograd nodes: check, allocate, launch -- and the
// same in the backward, on the autograd engine's thread, without the interpreter.  A Python node
// costs 10-15 us per direction, more than most of these kernels run for at ordinary sizes.
#include "host.hpp"

#include <ATen/autocast_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/autograd/custom_function.h>

#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace mega_host {
namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
using Optional = std::optional<Tensor>;

int kernel_code(const Tensor& t) {
  const int code = code_of(t.scalar_type());
  if (code < 0) fail("unsupported dtype " + std::string(c10::toString(t.scalar_type())) + " (float32, bfloat16, float16 are supported)");
  return code;
}
void need_gpu(std::initializer_list<const Tensor*> ts) {
  const Tensor* first = nullptr;
  for (const Tensor* t : ts) {
    if (t == nullptr || !t->defined()) continue;
    require(t->is_cuda(), "megalodon_amd ops need GPU (HIP) tensors; there is no CPU fallback");
    if (first == nullptr) first = t;
    require(t->device() == first->device(), "all tensors must be on the same device");
  }
}
const Tensor* maybe(const Optional& t) { return t.has_value() ? &*t : nullptr; }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
Tensor some(const Optional& t) { return t.has_value() ? t->contiguous() : Tensor(); }
Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }
Tensor floats(at::IntArrayRef shape, const Tensor& like) { return at::empty(shape, like.options().dtype(at::kFloat)); }
// whether the call has to go through its autograd node: a gradient is wanted, or an operand carries a
// forward-mode tangent, which the node refuses (whatever the gradient mode) and a bare launch would drop
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  const bool on = at::GradMode::is_enabled();
  for (const Tensor* t : ts)
    if (t != nullptr && t->defined() && ((on && t->requires_grad()) || has_tangent(*t))) return true;
  return false;
}

// ---- x.transpose(-2, -1).contiguous() ------------------------------------------------
Tensor transpose_raw(const Tensor& x) {
  need_gpu({&x});
  require(x.dim() >= 2, "transpose_last2: x needs at least two dimensions");
  const int code = kernel_code(x);
  c10::DeviceGuard guard(x.device());
  const Tensor xc = x.contiguous();
  const int64_t R = xc.size(-2), C = xc.size(-1);
  auto shape = xc.sizes().vec();
  std::swap(shape[shape.size() - 1], shape[shape.size() - 2]);
  Tensor out = at::empty(shape, xc.options());
  check(mega_transpose(xc.data_ptr(), code, R * C > 0 ? xc.numel() / (R * C) : 0, R, C, out.data_ptr(), stream_of(x)), "mega_transpose");
  return out;
}
struct TransposeFn : Function<TransposeFn> {
  static Tensor forward(AutogradContext*, const Tensor& x) {
    at::AutoDispatchBelowADInplaceOrView below;
    return transpose_raw(x);
  }
  static variable_list backward(AutogradContext*, variable_list g) { return {transpose_raw(g[0])}; }
};
Tensor transpose_last2(const Tensor& x) { return wants_grad({&x}) ? TransposeFn::apply(x) : transpose_raw(x); }

// ---- silu(a) b ------------------------------------------------------------------------
Tensor silu_mul_raw(const Tensor& a, const Tensor& b) {
  need_gpu({&a, &b});
  require(a.sizes() == b.sizes() && a.scalar_type() == b.scalar_type(), "silu_mul: a and b must have the same shape and dtype");
  const int code = kernel_code(a);
  c10::DeviceGuard guard(a.device());
  const Tensor ac = a.contiguous(), bc = b.contiguous();
  Tensor out = at::empty_like(ac);
  check(mega_silu_mul_fwd(ac.data_ptr(), bc.data_ptr(), code, ac.numel(), out.data_ptr(), stream_of(a)), "mega_silu_mul_fwd");
  return out;
}
struct SiluMulFn : Function<SiluMulFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b) {
    at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({a, b});
    return silu_mul_raw(a, b);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    at::AutoDispatchBelowADInplaceOrView below;
    const auto saved = ctx->get_saved_variables();
    const Tensor a = saved[0].contiguous(), b = saved[1].contiguous(), go = g[0].contiguous();
    c10::DeviceGuard guard(a.device());
    Tensor da = at::empty_like(a), db = at::empty_like(b);
    check(mega_silu_mul_bwd(go.data_ptr(), a.data_ptr(), b.data_ptr(), kernel_code(a), a.numel(), da.data_ptr(), db.data_ptr(), stream_of(a)), "mega_silu_mul_bwd");
    return {da, db};
  }
};
Tensor silu_mul(const Tensor& a, const Tensor& b) { return wants_grad({&a, &b}) ? SiluMulFn::apply(a, b) : silu_mul_raw(a, b); }

// ---- LayerNorm / RMSNorm over the last axis, stored weight gamma - 1 ------------------------
std::tuple<Tensor, Tensor, Tensor> layer_norm_raw(const Tensor& x, const Optional& weight, const Optional& bias, double eps, bool rms) {
  need_gpu({&x});
  const int64_t D = x.size(-1);
  for (const Optional* t : {&weight, &bias})
    if (t->has_value())
      require((*t)->dim() == 1 && (*t)->size(0) == D && (*t)->scalar_type() == x.scalar_type() && (*t)->device() == x.device(),
              "layer_norm: weight and bias must have the last axis' length, x's dtype and x's device");
  const int code = kernel_code(x);
  c10::DeviceGuard guard(x.device());
  const Tensor xc = x.contiguous(), w = some(weight), b = rms ? Tensor() : some(bias);
  const int64_t rows = D > 0 ? xc.numel() / D : 0;
  Tensor y = at::empty_like(xc), mean = rms ? Tensor() : floats({rows}, x), rstd = floats({rows}, x);
  check(mega_layer_norm_fwd(xc.data_ptr(), ptr(w), ptr(b), code, rows, D, eps, rms, y.data_ptr(), fptr(mean), fptr(rstd), stream_of(x)), "mega_layer_norm_fwd");
  return {y, mean, rstd};
}
struct LayerNormFn : Function<LayerNormFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Optional& weight, const Optional& bias, double eps, bool rms) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [y, mean, rstd] = layer_norm_raw(x, weight, bias, eps, rms);
    ctx->save_for_backward({x, weight.value_or(Tensor()), mean, rstd});
    ctx->saved_data["rms"] = rms;
    ctx->saved_data["bias"] = bias.has_value();
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    at::AutoDispatchBelowADInplaceOrView below;
    const auto saved = ctx->get_saved_variables();
    const bool rms = ctx->saved_data["rms"].toBool(), has_bias = ctx->saved_data["bias"].toBool();
    const Tensor x = saved[0].contiguous(), weight = saved[1].defined() ? saved[1].contiguous() : Tensor(), go = g[0].contiguous();
    require(go.scalar_type() == x.scalar_type(), "layer_norm_bwd: y_grad and x must have the same shape and dtype");
    const Tensor mean = saved[2].defined() ? saved[2].contiguous() : Tensor(), rstd = saved[3].contiguous();
    c10::DeviceGuard guard(x.device());
    const int64_t D = x.size(-1), rows = D > 0 ? x.numel() / D : 0;
    Tensor dx = at::empty_like(x), dw, db, ws;
    if (weight.defined()) {
      dw = at::empty_like(weight);
      ws = bytes(mega_layer_norm_workspace_bytes(rows, D), x);
    }
    if (has_bias && !rms && weight.defined()) db = at::empty_like(weight);
    if (rows == 0) {
      if (dw.defined()) dw.zero_();
      if (db.defined()) db.zero_();
    } else {
      check(mega_layer_norm_bwd(go.data_ptr(), x.data_ptr(), ptr(weight), fptr(mean), fptr(rstd), kernel_code(x), rows, D, rms, dx.data_ptr(), ptr(dw), ptr(db), ptr(ws), stream_of(x)), "mega_layer_norm_bwd");
    }
    return {dx, dw, db, Tensor(), Tensor()};
  }
};
Tensor layer_norm_plus_one(const Tensor& x, const Optional& weight, const Optional& bias, double eps, bool rms) {
  if (wants_grad({&x, maybe(weight), maybe(bias)})) return LayerNormFn::apply(x, weight, bias, eps, rms);
  return std::get<0>(layer_norm_raw(x, weight, bias, eps, rms));
}

// ---- z -> (q, k): per-head RMSNorm, two affine maps, rotary -----------------------------------
Tensor real_freqs(const Optional& freqs, int64_t head_dim, const Tensor& z) {
  if (!freqs.has_value()) return Tensor();
  require(freqs->dim() == 2 && freqs->size(1) == head_dim / 2 && freqs->is_complex(), "qk_norm_rotary: freqs_cis must be complex (positions, head_dim / 2)");
  return stored(freqs->to(z.device(), at::kComplexFloat)).contiguous();
}
std::tuple<Tensor, Tensor, Tensor> qk_raw(const Tensor& z, const Tensor& gamma, const Tensor& beta, const Tensor& fr, int64_t head_dim, double eps) {
  need_gpu({&z, &gamma, &beta});
  require(z.dim() == 3 && gamma.dim() == 2 && gamma.size(0) == 2 && gamma.size(1) == z.size(2) && beta.sizes() == gamma.sizes(), "qk_norm_rotary: z must be (B, L, S), gamma and beta (2, S)");
  require(gamma.scalar_type() == z.scalar_type() && beta.scalar_type() == z.scalar_type(), "qk_norm_rotary: gamma and beta must have z's dtype");
  const int code = kernel_code(z);
  const Tensor zc = z.contiguous(), gc = gamma.contiguous(), bc = beta.contiguous();
  const int64_t B = z.size(0), L = z.size(1), S = z.size(2);
  Tensor q = at::empty_like(zc), k = at::empty_like(zc), rstd = floats({B * L, S / head_dim}, z);
  check(mega_qk_norm_rotary_fwd(zc.data_ptr(), gc.data_ptr(), bc.data_ptr(), fptr(fr), code, B * L, L, fr.defined() ? fr.size(0) : 1, S, head_dim, eps, q.data_ptr(), k.data_ptr(), fptr(rstd), stream_of(z)), "mega_qk_norm_rotary_fwd");
  return {q, k, rstd};
}
struct QkFn : Function<QkFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& z, const Tensor& gamma, const Tensor& beta, const Optional& freqs, int64_t head_dim, double eps) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor fr = freqs.value_or(Tensor());
    auto [q, k, rstd] = qk_raw(z, gamma, beta, fr, head_dim, eps);
    ctx->save_for_backward({z, gamma, rstd, fr});
    ctx->saved_data["head_dim"] = head_dim;
    return {q, k};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    at::AutoDispatchBelowADInplaceOrView below;
    const auto saved = ctx->get_saved_variables();
    const Tensor z = saved[0].contiguous(), gamma = saved[1].contiguous(), dq = g[0].contiguous(), dk = g[1].contiguous();
    const Tensor fr = saved[3].defined() ? saved[3].contiguous() : Tensor(), rstd = saved[2].contiguous();
    c10::DeviceGuard guard(z.device());
    const int64_t B = z.size(0), L = z.size(1), S = z.size(2);
    Tensor dz = at::empty_like(z), dgamma = at::empty_like(gamma), dbeta = at::empty_like(gamma), ws = bytes(mega_qk_norm_rotary_workspace_bytes(S), z);
    check(mega_qk_norm_rotary_bwd(dq.data_ptr(), dk.data_ptr(), z.data_ptr(), gamma.data_ptr(), fptr(rstd), fptr(fr), kernel_code(z), B * L, L, fr.defined() ? fr.size(0) : 1, S, ctx->saved_data["head_dim"].toInt(), dz.data_ptr(), dgamma.data_ptr(), dbeta.data_ptr(), ws.data_ptr(), stream_of(z)), "mega_qk_norm_rotary_bwd");
    return {dz, dgamma, dbeta, Tensor(), Tensor(), Tensor()};
  }
};
std::tuple<Tensor, Tensor> qk_norm_rotary(const Tensor& z, const Tensor& gamma, const Tensor& beta, const Optional& freqs, int64_t head_dim, double eps) {
  c10::OptionalDeviceGuard guard;
  if (z.is_cuda()) guard.reset_device(z.device());
  const Tensor fr = real_freqs(freqs, head_dim, z);
  if (wants_grad({&z, &gamma, &beta}) || (fr.defined() && has_tangent(fr))) {
    auto qk = QkFn::apply(z, gamma, beta, fr.defined() ? Optional(fr) : Optional(), head_dim, eps);
    return {qk[0], qk[1]};
  }
  auto [q, k, rstd] = qk_raw(z, gamma, beta, fr, head_dim, eps);
  return {q, k};
}

// ---- TimestepNorm, the layer's call -------------------------------------------------------------
// The last workspace of every (device, stream, direction) is kept for its status word
// (timestep_norm_status); the launches themselves take a fresh one each, so calls of
// different threads never share one.
// (never destroyed: at the process's end the allocator may be gone first)
std::mutex last_mutex;
auto& last_workspace = *new std::map<std::tuple<int, void*, bool>, Tensor>();
Tensor tsn_workspace(const Tensor& x, int64_t groups, bool backward) {
  Tensor ws = bytes(mega_group_timestep_norm_workspace_bytes(x.size(0), x.size(1), x.size(2), groups, backward), x);
  std::lock_guard<std::mutex> lock(last_mutex);
  last_workspace[{x.device().index(), stream_of(x), backward}] = ws;
  return ws;
}
std::vector<Tensor> tsn_last_workspaces(int device, uintptr_t stream) {
  std::lock_guard<std::mutex> lock(last_mutex);
  std::vector<Tensor> out;
  for (const bool backward : {false, true}) {
    auto it = last_workspace.find({device, reinterpret_cast<void*>(stream), backward});
    if (it != last_workspace.end()) out.push_back(it->second);
  }
  return out;
}
struct TsnOut {
  Tensor y, count, mean, var, cummean, cumrstd;
};
TsnOut tsn_raw(const Tensor& x, const Tensor& count0, const Tensor& mean0, const Tensor& var0, bool shared, const Tensor& weight, const Tensor& bias, const Optional& mask, int64_t groups, double eps) {
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2);
  TsnOut o;
  o.y = at::empty_like(x);
  o.count = at::empty({B}, x.options().dtype(at::kLong));
  o.mean = at::empty({B, groups}, x.options());
  o.var = at::empty({B, groups}, x.options());
  o.cummean = floats({B, groups, L}, x);
  o.cumrstd = floats({B, groups, L}, x);
  const Tensor m = some(mask), ws = tsn_workspace(x, groups, false);
  check(mega_timestep_norm_layer_fwd(x.data_ptr(), kernel_code(x), count0.data_ptr<int64_t>(), mean0.data_ptr(), var0.data_ptr(), shared, weight.data_ptr(), bias.data_ptr(), static_cast<const uint8_t*>(ptr(m)), B, L, D, groups, eps, o.y.data_ptr(), o.count.data_ptr<int64_t>(), o.mean.data_ptr(), o.var.data_ptr(), fptr(o.cummean), fptr(o.cumrstd), ws.data_ptr(), stream_of(x)), "mega_timestep_norm_layer_fwd");
  return o;
}
struct TsnFn : Function<TsnFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& count0, const Tensor& mean0, const Tensor& var0, bool shared, const Tensor& weight, const Tensor& bias, const Optional& mask, int64_t groups, double eps) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor xc = x.contiguous();
    TsnOut o = tsn_raw(xc, count0, mean0, var0, shared, weight, bias, mask, groups, eps);
    ctx->save_for_backward({xc, mean0, o.count, o.cummean, o.cumrstd, weight, mask.value_or(Tensor())});
    ctx->saved_data["groups"] = groups;
    ctx->saved_data["shared"] = shared;
    ctx->mark_non_differentiable({o.count});
    ctx->set_materialize_grads(false);
    return {o.y, o.count, o.mean, o.var};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    at::AutoDispatchBelowADInplaceOrView below;
    const auto saved = ctx->get_saved_variables();
    // (saved-tensor hooks may hand back any layout)
    const Tensor x = saved[0].contiguous(), mean0 = saved[1].contiguous(), count = saved[2].contiguous(),
                 cummean = saved[3].contiguous(), cumrstd = saved[4].contiguous(), weight = saved[5].contiguous();
    c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), L = x.size(1), D = x.size(2), groups = ctx->saved_data["groups"].toInt();
    const bool shared = ctx->saved_data["shared"].toBool();
    const Tensor dy = g[0].defined() ? g[0].contiguous() : at::zeros_like(x);
    const Tensor dm = g[2].defined() ? g[2].contiguous() : Tensor(), dv = g[3].defined() ? g[3].contiguous() : Tensor();
    const Tensor mask = saved[6].defined() ? saved[6].contiguous() : Tensor();
    require(dy.scalar_type() == x.scalar_type(), "timestep_norm: y_grad must have x's dtype");
    Tensor dx = at::empty_like(x), dpm = at::empty({B, groups}, x.options()), dpv = at::empty({B, groups}, x.options()), dw = at::empty_like(weight), db = at::empty_like(weight);
    const Tensor ws = tsn_workspace(x, groups, true);
    check(mega_timestep_norm_layer_bwd(dy.data_ptr(), ptr(dm), ptr(dv), x.data_ptr(), kernel_code(x), mean0.data_ptr(), shared, count.data_ptr<int64_t>(), fptr(cummean), fptr(cumrstd), weight.data_ptr(), static_cast<const uint8_t*>(ptr(mask)), B, L, D, groups, dx.data_ptr(), dpm.data_ptr(), dpv.data_ptr(), dw.data_ptr(), db.data_ptr(), ws.data_ptr(), stream_of(x)), "mega_timestep_norm_layer_bwd");
    if (shared) dpm = dpv = Tensor();  // the prior is no parameter here
    return {dx, Tensor(), dpm, dpv, Tensor(), dw, db, Tensor(), Tensor(), Tensor()};
  }
};
// (y, count, mean, var), or None where the layer has to prepare its operands itself (other element
// types of weights or statistics, a prior that is trained)
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> timestep_norm_layer(const Tensor& x, const Optional& prev_count, const Optional& prev_mean, const Optional& prev_var, const Tensor& prior_count, const Tensor& prior_mean, const Tensor& prior_logv, const Tensor& weight, const Tensor& bias, const Optional& mask, int64_t groups, double eps) {
  const bool shared = !prev_count.has_value();
  if (!x.is_cuda() || x.dim() != 3 || code_of(x.scalar_type()) < 0 || x.size(0) < 1 || x.size(1) < 1) return std::nullopt;
  if (prev_mean.has_value() == shared || prev_var.has_value() == shared) return std::nullopt;
  const Tensor &count = shared ? prior_count : *prev_count, &mean = shared ? prior_mean : *prev_mean, &var = shared ? prior_logv : *prev_var;
  if (shared && at::GradMode::is_enabled() && (mean.requires_grad() || var.requires_grad())) return std::nullopt;
  const int64_t B = x.size(0), D = x.size(2);
  const auto is = [&](const Tensor& t, at::ScalarType type, int64_t n) { return t.scalar_type() == type && t.device() == x.device() && t.numel() == n && t.is_contiguous(); };
  if (!is(weight, x.scalar_type(), D) || !is(bias, x.scalar_type(), D) || !is(count, at::kLong, shared ? 1 : B) || !is(mean, x.scalar_type(), shared ? groups : B * groups) || !is(var, x.scalar_type(), shared ? groups : B * groups)) return std::nullopt;
  if (mask.has_value()) {
    if (mask->scalar_type() != at::kBool) fail("padding_mask must be a bool tensor");
    if (mask->device() != x.device() || mask->numel() != B * x.size(1)) return std::nullopt;
  }
  c10::DeviceGuard guard(x.device());
  if (wants_grad({&x, &mean, &var, &weight, &bias})) {
    auto o = TsnFn::apply(x, count, mean, var, shared, weight, bias, mask, groups, eps);
    return std::make_tuple(o[0], o[1], o[2], o[3]);
  }
  TsnOut o = tsn_raw(x.contiguous(), count, mean, var, shared, weight, bias, mask, groups, eps);
  return std::make_tuple(o.y, o.count, o.mean, o.var);
}

// ---- the EMA layer without a carried state ------------------------------------------------------
// Coefficients in one float32 buffer (p, log q, gamma_hat), then the recurrence.
Tensor cema_coeffs(const Tensor& alpha, const Tensor& delta, const Tensor& theta, const Tensor& gamma, int64_t D, int64_t N) {
  Tensor c = floats({5 * D * N}, alpha);
  float* p = c.data_ptr<float>();
  check(mega_cema_layer_coeffs_fwd(kernel_code(alpha), alpha.data_ptr(), delta.data_ptr(), theta.data_ptr(), gamma.data_ptr(), D, N, p, p + D * N, p + 3 * D * N, stream_of(alpha)), "mega_cema_layer_coeffs_fwd");
  return c;
}
Tensor scan_raw(const Tensor& x, const float* p, const float* log_q, const float* gamma_hat, const float* omega, const float* h0, float* h_last, int64_t N) {
  Tensor y = at::empty_like(x);
  check(mega_cema_layer_scan_fwd(x.data_ptr(), kernel_code(x), p, log_q, gamma_hat, omega, h0, x.size(0), x.size(1), N, x.size(2), y.data_ptr(), h_last, stream_of(x)), "mega_cema_layer_scan_fwd");
  return y;
}
// float32 (contiguous) form of the skip weight
Tensor as_float(const Tensor& t) { return t.to(at::kFloat).contiguous(); }
// rows as the recurrence kernels take them: float32 ones on 16-byte boundaries
Tensor rows_of(const Tensor& x) {
  Tensor c = x.contiguous();
  if (c.scalar_type() == at::kFloat && reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 != 0) c = c.clone(at::MemoryFormat::Contiguous);
  return c;
}
// a float32 tensor in two bfloat16 pieces, or in three; all in one tensor, each on a 16-byte boundary
Tensor split(const Tensor& t, int pieces) {
  const int64_t n = t.numel(), n8 = (n + 7) / 8 * 8;
  Tensor out = at::empty({pieces, n8}, t.options().dtype(at::kBFloat16));
  uint16_t* p = static_cast<uint16_t*>(out.data_ptr());
  Tensor whole = t;
  if (n != n8) whole = at::constant_pad_nd(t.reshape({-1}), {0, n8 - n});
  if (pieces == 2) check(mega_split_bf16(whole.data_ptr(), kernel_code(t), n8, p, p + n8, stream_of(t)), "mega_split_bf16");
  else check(mega_split_bf16_three(whole.data_ptr<float>(), n8, p, p + n8, p + 2 * n8, stream_of(t)), "mega_split_bf16_three");
  return out;
}
struct CemaFn : Function<CemaFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& alpha, const Tensor& delta, const Tensor& theta, const Tensor& gamma, const Tensor& omega) {
    at::AutoDispatchBelowADInplaceOrView below;
    const int64_t D = x.size(1), N = alpha.size(1);
    const Tensor xc = rows_of(x), w = as_float(omega), c = cema_coeffs(alpha, delta, theta, gamma, D, N);
    const float* p = c.data_ptr<float>();
    Tensor y = scan_raw(xc, p, p + D * N, p + 3 * D * N, fptr(w), nullptr, nullptr, N);
    ctx->save_for_backward({xc, alpha, delta, theta, gamma, omega, c, w});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    at::AutoDispatchBelowADInplaceOrView below;
    const auto saved = ctx->get_saved_variables();
    const Tensor x = rows_of(saved[0]), alpha = saved[1].contiguous(), delta = saved[2].contiguous(), theta = saved[3].contiguous(), gamma = saved[4].contiguous(), omega = saved[5].contiguous(), c = saved[6].contiguous(), w = saved[7].contiguous();
    require(g[0].sizes() == x.sizes() && g[0].scalar_type() == x.scalar_type(), "cema: y_grad must match x in shape and dtype");
    c10::DeviceGuard guard(x.device());
    const Tensor dy = rows_of(g[0]);
    const int64_t B = x.size(0), D = x.size(1), L = x.size(2), N = alpha.size(1), DN = D * N;
    const float *p = c.data_ptr<float>(), *lq = p + DN, *gh = p + 3 * DN;
    void* s = stream_of(x);
    // gradients of the launches' groups of rows, stacked: (dp, dq, dgamma_hat, domega); the coefficients'
    // backward adds the stack up
    const bool wide = x.scalar_type() == at::kFloat;
    const bool thirds = wide && L % 8 != 0;
    const int64_t per = mega_cema_layer_scan_sets(B, D, L), launches = thirds ? 6 : wide ? 3 : 1, sets = launches * per;
    const Tensor stack = floats({sets * (5 * DN + D)}, x);
    float *dp = stack.data_ptr<float>(), *dq = dp + sets * DN, *dg = dq + 2 * sets * DN, *dw = dg + 2 * sets * DN;
    Tensor dx = wide ? floats(x.sizes(), x) : at::empty_like(x);
    if (!wide) {
      const int mode = x.scalar_type() == at::kHalf ? 3 : 0;
      check(mega_cema_layer_scan_bwd(dy.data_ptr(), x.data_ptr(), p, lq, gh, fptr(w), B, D, N, L, dx.data_ptr(), mode, dp, dq, dg, dw, s), "mega_cema_layer_scan_bwd");
    } else {
      // linear in dy and, for the parameter gradients, in x: pairs of bfloat16 pieces.  dx is linear in dy alone and is
      // added up in float32 over the pairs with x's first piece.  Lengths that are a multiple of 8 take two pieces and leave out
      // (dy_lo, x_lo), 2e-6 of the parameter gradients; the others, which came from a float32 convolution, three and leave
      // out what is below 2^-25 (forward and backward of 2048 x 52327 12.2 -> 2.1 ms, 2048 x 22185 1.72 -> 1.01).
      static constexpr int pairs[6][2] = {{0, 0}, {1, 0}, {0, 1}, {2, 0}, {1, 1}, {0, 2}};
      const Tensor gp = split(dy, thirds ? 3 : 2), xp = split(x, thirds ? 3 : 2);
      const int64_t n8 = gp.size(1);
      const uint16_t *g0 = static_cast<const uint16_t*>(gp.data_ptr()), *x0 = static_cast<const uint16_t*>(xp.data_ptr());
      for (int i = 0; i < launches; ++i) {
        const bool to_dx = pairs[i][1] == 0;
        check(mega_cema_layer_scan_bwd(g0 + pairs[i][0] * n8, x0 + pairs[i][1] * n8, p, lq, gh, fptr(w), B, D, N, L, to_dx ? dx.data_ptr() : nullptr, to_dx && i > 0 ? 2 : 1, dp + i * per * DN, dq + 2 * i * per * DN, dg + 2 * i * per * DN, dw + i * per * D, s), "mega_cema_layer_scan_bwd");
      }
    }
    Tensor da = at::empty_like(alpha), dd = at::empty_like(delta), dt = at::empty_like(theta), dga = at::empty_like(gamma), dom = at::empty_like(omega);
    check(mega_cema_layer_coeffs_bwd(kernel_code(alpha), dp, dq, dg, dw, sets, alpha.data_ptr(), delta.data_ptr(), theta.data_ptr(), D, N, da.data_ptr(), dd.data_ptr(), dt.data_ptr(), dga.data_ptr(), dom.data_ptr(), s), "mega_cema_layer_coeffs_bwd");
    return {dx, da, dd, dt, dga, dom};
  }
};
// rows of this shape and type run on the recurrence kernels in one launch per piece
bool cema_takes(const Tensor& x, int64_t N) {
  return x.is_cuda() && x.dim() == 3 && N >= 1 && N <= 16 && code_of(x.scalar_type()) >= 0 && x.size(2) >= 1 && x.size(0) * x.size(1) <= 0x7fffffff;
}
// float32 rows whose length is no multiple of 8: whether the recurrence is ahead of the convolution (kernel row, float32 transforms).
// A row of one chunk costs the recurrence a tile like one of 24 of them, and the backward six launches, each of which sets
// up its channels; the transforms' cost follows the power of two above 2 L.  us, recurrence / convolution: forward 64 x 1024 rows of 9
// steps 220 / 46, 16 x 4096 of 193 225 / 151, of 385 228 / 309; 4 x 2048 of 9 35 / 47.  Forward and backward 64 x 1024 of 9 1669 / 152, of 513
// 1912 / 1588, of 1021 2145 / 3276; 16 x 1024 of 65 520 / 255, of 700 611 / 593, of 850 628 / 829; 2048 of 1100 357 / 271, 2 x 1024 220 / 253; 4 x 2048
// of 3001 741 / 674, of 5001 987 / 1184, of 8191 1503 / 1415, 1024 x 16383 485 / 490, x 20001 523 / 900.  Few rows take the host longer than the
// device, four launches and Python where the recurrence is one call: 4 x 64 rows of 65 108 / 150 - 260.  Batches of narrow layers
// add the convolution's weight gradient up slowly: 256 x 64 of 129 steps 544 / 675, 64 x 16 of 257 178 / 347.
bool recurrence_ahead(int64_t B, int64_t D, int64_t L, bool train) {
  const int64_t rows = B * D;
  if (!train) return L > 288 || B <= 4 || rows <= 6144;
  if (L <= 512) return (B <= 8 && D <= 512 && rows <= 2048) || (B >= 16 && D <= 128 && L > 128);
  if (L <= 1024) return (D <= 512 && (B >= 8 || rows <= 2048)) || (B >= 4 && L > 736);
  if (L <= 2048) return B >= 2 || D <= 512 || L > 1400;
  if (L <= 4096) return (B <= 8 && D <= 512 && rows <= 1024) || (B >= 4 && L <= 2304);
  if (L <= 6144) return B >= 2 || D <= 512;
  return L > 8192 || rows <= 512;
}
Optional cema(const Tensor& x, const Tensor& alpha, const Tensor& delta, const Tensor& theta, const Tensor& gamma, const Tensor& omega) {
  if (alpha.dim() != 3 || !cema_takes(x, alpha.size(1))) return std::nullopt;
  const int64_t D = x.size(1), N = alpha.size(1);
  const auto is = [&](const Tensor& t, int64_t n) { return t.scalar_type() == alpha.scalar_type() && t.device() == x.device() && t.numel() == n && t.is_contiguous(); };
  if (code_of(alpha.scalar_type()) < 0 || !is(alpha, D * N) || !is(delta, D * N) || !is(theta, D) || !is(gamma, 2 * D * N) || !is(omega, D)) return std::nullopt;
  const bool train = wants_grad({&x, &alpha, &delta, &theta, &gamma, &omega});
  if (x.scalar_type() == at::kFloat && x.size(2) % 8 != 0 && !recurrence_ahead(x.size(0), D, x.size(2), train)) return std::nullopt;
  c10::DeviceGuard guard(x.device());
  if (train) return CemaFn::apply(x, alpha, delta, theta, gamma, omega);
  const Tensor xc = rows_of(x), ws = floats({5 * D * N}, x);
  Tensor y = at::empty_like(xc);
  if (y.numel() == 0) return y;
  check(mega_cema_layer_fwd(xc.data_ptr(), kernel_code(x), kernel_code(alpha), alpha.data_ptr(), delta.data_ptr(), theta.data_ptr(), gamma.data_ptr(), omega.data_ptr(), x.size(0), D, N, x.size(2), y.data_ptr(), ws.data_ptr(), stream_of(x)), "mega_cema_layer_fwd");
  return y;
}
// with a carried state and / or the last state wanted, without gradients; p, log_q, gamma_hat float32 / complex64
std::optional<std::tuple<Tensor, Optional>> cema_state(const Tensor& x, const Tensor& p, const Tensor& log_q, const Tensor& gamma_hat, const Tensor& omega, const Optional& h0, bool last) {
  const int64_t N = p.size(1);
  if (!cema_takes(x, N)) return std::nullopt;
  // (with a carried state these lengths take the convolution)
  if (h0.has_value() && x.scalar_type() == at::kFloat && x.size(2) % 8 != 0) return std::nullopt;
  const int64_t B = x.size(0), D = x.size(1);
  require(p.numel() == D * N && log_q.numel() == D * N && gamma_hat.numel() == D * N && omega.numel() == D, "cema: x and the parameters must have the same number of channels");
  if (h0.has_value()) require(h0->scalar_type() == at::kComplexFloat && h0->numel() == B * D * N && h0->device() == x.device(), "cema: the carried state must be complex64 (B, D, N)");
  c10::DeviceGuard guard(x.device());
  const Tensor xc = rows_of(x), w = as_float(omega), h = h0.has_value() ? stored(*h0).contiguous() : Tensor();
  Tensor h_last;
  if (last) h_last = at::empty({B, D, N}, x.options().dtype(at::kComplexFloat));
  Tensor y = scan_raw(xc, p.data_ptr<float>(), fptr(log_q), fptr(gamma_hat), fptr(w), fptr(h), fptr(h_last), N);
  return std::make_tuple(y, last ? Optional(h_last) : std::nullopt);
}

// ---- attention ------------------------------------------------------------------------------------
struct AttnDims {
  int64_t B, L1, L2, NH, H1, H2;
};
AttnDims attn_dims(const Tensor& q, const Tensor& k, const Tensor& v) {
  need_gpu({&q, &k, &v});
  require(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k, v must be (B, L, N, H)");
  const AttnDims d{q.size(0), q.size(1), k.size(1), q.size(2), q.size(3), v.size(3)};
  require(k.size(0) == d.B && k.size(2) == d.NH && k.size(3) == d.H1 && v.size(0) == d.B && v.size(1) == d.L2 && v.size(2) == d.NH, "attention: inconsistent shapes");
  require(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(), "q, k, v must share one dtype");
  return d;
}
// contiguous, on a 16-byte boundary
Tensor attn_operand(const Tensor& t) {
  Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone(at::MemoryFormat::Contiguous);
}
std::tuple<Tensor, Tensor> attention_raw(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
  const AttnDims d = attn_dims(q, k, v);
  const int code = kernel_code(q);
  Tensor y = at::empty({d.B, d.L1, d.NH, d.H2}, v.options());
  Tensor saved = at::empty({mega_attention_layer_saved_elements(code, d.B, d.L1, d.L2, d.NH, d.H1, d.H2, scale)}, v.options());
  check(mega_attention_layer_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), code, d.B, d.L1, d.L2, d.NH, d.H1, d.H2, scale, causal, y.data_ptr(), saved.data_ptr(), stream_of(q)), "mega_attention_layer_fwd");
  return {y, saved};
}
struct AttentionFn : Function<AttentionFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor qc = attn_operand(q), kc = attn_operand(k), vc = attn_operand(v);
    auto [y, w] = attention_raw(qc, kc, vc, scale, causal);
    ctx->save_for_backward({qc, kc, vc, w});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["causal"] = causal;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    at::AutoDispatchBelowADInplaceOrView below;
    const auto saved = ctx->get_saved_variables();
    const Tensor q = attn_operand(saved[0]), k = attn_operand(saved[1]), v = attn_operand(saved[2]), w = attn_operand(saved[3]);
    const AttnDims d = attn_dims(q, k, v);
    c10::DeviceGuard guard(q.device());
    const Tensor dy = attn_operand(g[0]);
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const Tensor ws = at::empty_like(w);
    check(mega_attention_layer_bwd(dy.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), kernel_code(q), d.B, d.L1, d.L2, d.NH, d.H1, d.H2, ctx->saved_data["scale"].toDouble(), ctx->saved_data["causal"].toBool(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), stream_of(q)), "mega_attention_layer_bwd");
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};
Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
  attn_dims(q, k, v);
  c10::DeviceGuard guard(q.device());
  if (wants_grad({&q, &k, &v})) return AttentionFn::apply(q, k, v, scale, causal);
  return std::get<0>(attention_raw(attn_operand(q), attn_operand(k), attn_operand(v), scale, causal));
}

// ---- linear layers --------------------------------------------------------------------------------
// Whether the thread shows its operations to something beside autograd: the TorchScript tracer, a mode that counts flops
// or makes fake tensors, a functorch transform.  A launch is no operation -- a trace of one holds the allocation of its
// result and nothing that fills it -- so these are given the library's products.
bool watched() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return (tls.included_ - tls.excluded_ - c10::default_included_set).highestFunctionalityKey() != c10::DispatchKey::Undefined;
}
// Whether a tensor is what its memory holds and nothing more: dispatch keys of a dense tensor, no subclass, functional
// wrapper, zeros without memory or batch.
bool plain(const Tensor& t) {
  constexpr auto usual = c10::default_included_set | c10::autograd_dispatch_keyset | c10::autocast_dispatch_keyset | c10::DispatchKeySet(c10::DispatchKey::Dense);
  return (t.key_set() - usual).highestFunctionalityKey() == c10::DispatchKey::Undefined && t.has_storage();
}
// A matrix as the library's products take it: its own memory, whole rows, 16-byte boundary.
bool dense16(const Tensor& t) {
  if (!plain(t) || watched() || !t.is_contiguous()) return false;
  const void* memory = t.data_ptr();
  return memory != nullptr && reinterpret_cast<uintptr_t>(memory) % 16 == 0;
}
enum { kLinearForward, kLinearInputGrad, kLinearWeightGrad };
// memory for the parts of products that are cut along their reduction axis
Tensor parts_of(int kind, const Tensor& x, int64_t tokens, int64_t n_in, const std::vector<int64_t>& n_out) {
  const int64_t size = mega_linear_workspace_bytes(kind, tokens, n_in, static_cast<int>(n_out.size()), n_out.data());
  return size > 0 ? at::empty({size}, x.options().dtype(at::kByte)) : Tensor();
}
// dW_i = g_i^T x, (out_i, in) from (tokens, out_i) and (tokens, in), for layers of one input in one launch.
variable_list weight_grads(variable_list gs, const Tensor& x) {
  const int64_t tokens = x.size(0), n_in = x.size(1);
  const int code = code_of(x.scalar_type());
  bool taken = !gs.empty() && gs.size() <= 3 && x.has_storage();
  for (const Tensor& g : gs) taken = taken && g.has_storage() && g.scalar_type() == x.scalar_type() && g.size(0) == tokens;
  std::vector<int64_t> n_out;
  for (const Tensor& g : gs) n_out.push_back(g.size(1));
  taken = taken && mega_linear_takes(kLinearWeightGrad, code, tokens, n_in, static_cast<int>(gs.size()), n_out.data());
  variable_list dw;
  if (taken) {
    const Tensor xc = x.contiguous();
    std::vector<const void*> from;
    std::vector<void*> to;
    taken = dense16(xc);
    for (Tensor& g : gs) {
      g = g.contiguous();
      taken = taken && dense16(g);
    }
    if (taken) {
      for (const Tensor& g : gs) {
        dw.push_back(at::empty({g.size(1), n_in}, x.options()));
        from.push_back(g.data_ptr());
        to.push_back(dw.back().data_ptr());
      }
      const Tensor ws = parts_of(kLinearWeightGrad, x, tokens, n_in, n_out);
      check(mega_linear_weight_grads(from.data(), xc.data_ptr(), code, tokens, n_in, static_cast<int>(gs.size()), n_out.data(), to.data(), ptr(ws), stream_of(x)), "mega_linear_weight_grads");
      return dw;
    }
  }
  for (const Tensor& g : gs) dw.push_back(at::mm(g.t(), x));
  return dw;
}
Tensor flat(const Tensor& t) { return t.reshape({-1, t.size(-1)}); }
// the bias gradient: column sums of g (tokens, out)
Tensor bias_grad(const Tensor& g) {
  const int64_t rows = g.size(0), cols = g.size(1);
  const bool taken = rows >= 1 && cols >= 1 && cols % 8 == 0 && cols <= (1 << 24) &&
                     (g.scalar_type() == at::kBFloat16 || g.scalar_type() == at::kHalf) && dense16(g);
  if (!taken) return g.sum(0);
  Tensor out = at::empty({cols}, g.options()), ws = bytes(mega_column_sums_workspace_bytes(rows, cols), g);
  check(mega_column_sums(g.data_ptr(), kernel_code(g), rows, cols, out.data_ptr(), ws.data_ptr(), stream_of(g)), "mega_column_sums");
  return out;
}
// Whether dx = g W goes through a transposed copy of W, after which both operands run along the reduction axis:
// the library's product is then faster by more than the copy takes where the product is large.  The copy
// included / without it, in us: 4096 tokens x 2048 x 1024 30 / 25, 4096 x 2752 x 1024 37 / 32, 4096 x 4096 x 2048 (2^35
// products) 68 / 66; 8192 x 4096 x 2048 102 / 107, 32768 x 2048 x 1024 109 / 120, 8192 x 4096 x 4096 194 / 217.
bool turned(const Tensor& g, const Tensor& w) {
  return static_cast<double>(g.size(0)) * w.size(0) * w.size(1) > static_cast<double>(1ll << 35) && plain(w) && !watched();
}
// dx = g W, added to `sum` (in place) where there is one
Tensor input_grad(const Tensor& g, const Tensor& w, const Tensor& sum) {
  const int64_t tokens = g.size(0), n_out = g.size(1), n_in = w.size(1);
  const int code = code_of(g.scalar_type());
  if (w.scalar_type() == g.scalar_type() && w.size(0) == n_out && mega_linear_takes(kLinearInputGrad, code, tokens, n_in, 1, &n_out) &&
      dense16(g) && dense16(w) && (!sum.defined() || dense16(sum))) {
    const Tensor dx = sum.defined() ? sum : at::empty({tokens, n_in}, g.options());
    const void *gp = g.data_ptr(), *wp = w.data_ptr();
    check(mega_linear_input_grad(&gp, &wp, ptr(sum), code, tokens, n_in, 1, &n_out, dx.data_ptr(), stream_of(g)), "mega_linear_input_grad");
    return dx;
  }
  if (!sum.defined()) return turned(g, w) ? at::linear(g, transpose_raw(w)) : at::mm(g, w);
  const Tensor wt = turned(g, w) ? transpose_raw(w).t() : w;
  Tensor dx = sum;
  at::addmm_out(dx, sum, g, wt);
  return dx;
}
// sum_i g_i W_i, (tokens, out_i) x (out_i, in): one product along all of the outputs where its launch takes them
Tensor input_grads(const variable_list& gs, const variable_list& ws) {
  const int64_t tokens = gs[0].size(0), n_in = ws[0].size(1);
  const int code = code_of(gs[0].scalar_type()), count = static_cast<int>(gs.size());
  bool taken = count >= 2 && count <= 3;
  std::vector<int64_t> n_out;
  std::vector<const void*> gp, wp;
  for (size_t i = 0; i < gs.size(); ++i) {
    n_out.push_back(gs[i].size(1));
    taken = taken && gs[i].scalar_type() == gs[0].scalar_type() && ws[i].scalar_type() == gs[0].scalar_type() && gs[i].size(0) == tokens &&
            ws[i].size(0) == n_out[i] && ws[i].size(1) == n_in && dense16(gs[i]) && dense16(ws[i]);
    if (taken) {
      gp.push_back(gs[i].data_ptr());
      wp.push_back(ws[i].data_ptr());
    }
  }
  if (taken && mega_linear_takes(kLinearInputGrad, code, tokens, n_in, count, n_out.data())) {
    const Tensor dx = at::empty({tokens, n_in}, gs[0].options());
    check(mega_linear_input_grad(gp.data(), wp.data(), nullptr, code, tokens, n_in, count, n_out.data(), dx.data_ptr(), stream_of(gs[0])), "mega_linear_input_grad");
    return dx;
  }
  Tensor dx;
  for (size_t i = 0; i < gs.size(); ++i) dx = input_grad(gs[i], ws[i], dx);
  return dx;
}
// y_i = x W_i^T (+ bias_i), + residual with one layer, in one launch; nothing where the library's products are faster or
// the operands are not what the launch takes
std::optional<variable_list> products(const Tensor& x, const variable_list& w, const std::vector<Optional>& bias, const Optional& residual) {
  const auto type = x.scalar_type();
  if (!x.is_cuda() || x.dim() < 1 || (type != at::kBFloat16 && type != at::kHalf) || w.size() > 3 || at::autocast::is_autocast_enabled(at::kCUDA)) return std::nullopt;
  const int64_t n_in = x.size(-1), tokens = n_in > 0 ? x.numel() / n_in : 0;
  const auto fits = [&](const Tensor& t) { return t.scalar_type() == type && t.device() == x.device() && dense16(t); };
  if (tokens < 1 || !fits(x)) return std::nullopt;
  std::vector<int64_t> n_out;
  for (size_t i = 0; i < w.size(); ++i) {
    if (w[i].dim() != 2 || w[i].size(1) != n_in || !fits(w[i])) return std::nullopt;
    if (bias[i].has_value() && (bias[i]->dim() != 1 || bias[i]->size(0) != w[i].size(0) || !fits(*bias[i]))) return std::nullopt;
    n_out.push_back(w[i].size(0));
  }
  auto shape = x.sizes().vec();
  shape.back() = n_out[0];
  if (residual.has_value() && (w.size() != 1 || residual->sizes() != at::IntArrayRef(shape) || !fits(*residual))) return std::nullopt;
  const int code = code_of(type), count = static_cast<int>(w.size());
  if (!mega_linear_takes(kLinearForward, code, tokens, n_in, count, n_out.data())) return std::nullopt;
  c10::DeviceGuard guard(x.device());
  variable_list y;
  std::vector<const void*> wp, bp;
  std::vector<void*> yp;
  for (size_t i = 0; i < w.size(); ++i) {
    shape.back() = n_out[i];
    y.push_back(at::empty(shape, x.options()));
    wp.push_back(w[i].data_ptr());
    bp.push_back(bias[i].has_value() ? bias[i]->data_ptr() : nullptr);
    yp.push_back(y.back().data_ptr());
  }
  const Tensor ws = parts_of(kLinearForward, x, tokens, n_in, n_out);
  check(mega_linear_fwd(x.data_ptr(), wp.data(), bp.data(), residual.has_value() ? residual->data_ptr() : nullptr, code, tokens, n_in, count, n_out.data(), yp.data(), ptr(ws), stream_of(x)), "mega_linear_fwd");
  return y;
}
// x W^T (+ bias), or x W^T + residual with the residual as the product's accumulator input
Tensor linear_raw(const Tensor& x, const Tensor& weight, const Optional& bias, const Optional& residual) {
  if (auto y = products(x, {weight}, {bias}, residual); y.has_value()) return (*y)[0];
  if (!residual.has_value()) return at::linear(x, weight, bias);
  require(x.dim() >= 1 && residual->dim() >= 1, "linear: x and residual need at least one dimension");
  auto shape = x.sizes().vec();
  shape.back() = weight.size(0);
  return at::addmm(flat(*residual), flat(x), weight.t()).view(shape);
}
// A layer's gradients (dx, dW, db) as recorded operations: under create_graph the backward is itself
// differentiated, so nothing in it may go below autograd or to a kernel that autograd does not know.
struct LinearGrads {
  Tensor dx, dw, db;
};
LinearGrads linear_recorded(const Tensor& g, const Tensor& x, const Tensor& weight, bool dx, bool dw, bool db) {
  const Tensor g2 = flat(g);
  return {dx ? at::mm(g2, weight).view(x.sizes()) : Tensor(), dw ? at::mm(g2.t(), flat(x)) : Tensor(), db ? g2.sum(0) : Tensor()};
}
struct LinearFn : Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const Optional& bias, const Optional& residual) {
    at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({x, weight});
    ctx->saved_data["bias"] = bias.has_value();
    ctx->saved_data["residual"] = residual.has_value();
    return linear_raw(x, weight, bias, residual);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &weight = saved[1];
    const bool has_bias = ctx->saved_data["bias"].toBool(), has_residual = ctx->saved_data["residual"].toBool();
    c10::DeviceGuard guard(x.device());
    if (at::GradMode::is_enabled()) {
      auto r = linear_recorded(g[0], x, weight, ctx->needs_input_grad(0), ctx->needs_input_grad(1), has_bias && ctx->needs_input_grad(2));
      return {r.dx, r.dw, r.db, has_residual && ctx->needs_input_grad(has_bias ? 3 : 2) ? g[0] : Tensor()};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor g2 = flat(g[0]);
    Tensor dx, dw, db, dr;
    if (ctx->needs_input_grad(0)) dx = input_grad(g2, weight, Tensor()).view(x.sizes());
    if (ctx->needs_input_grad(1)) dw = weight_grads({g2}, flat(x))[0];
    if (has_bias && ctx->needs_input_grad(2)) db = bias_grad(g2);
    if (has_residual && ctx->needs_input_grad(has_bias ? 3 : 2)) dr = g[0];
    return {dx, dw, db, dr};
  }
};
Tensor linear(const Tensor& x, const Tensor& weight, const Optional& bias, const Optional& residual) {
  if (wants_grad({&x, &weight, maybe(bias), maybe(residual)})) return LinearFn::apply(x, weight, bias, residual);
  return linear_raw(x, weight, bias, residual);
}

// several layers of one input: products, input gradient and weight gradients in one launch each where that is the faster form
struct LinearGroupFn : Function<LinearGroupFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, at::TensorList params, std::vector<bool> has_bias) {
    at::AutoDispatchBelowADInplaceOrView below;
    variable_list keep{x}, weights;
    std::vector<Optional> biases;
    size_t at_ = 0;
    std::vector<int64_t> bias_flags;
    for (const bool b : has_bias) {
      weights.push_back(params[at_++]);
      biases.push_back(b ? Optional(params[at_++]) : Optional());
      keep.push_back(weights.back());
      bias_flags.push_back(b);
    }
    variable_list out;
    if (auto y = products(x, weights, biases, Optional()); y.has_value()) out = *y;
    else
      for (size_t i = 0; i < weights.size(); ++i) out.push_back(linear_raw(x, weights[i], biases[i], Optional()));
    ctx->save_for_backward(keep);
    ctx->saved_data["bias"] = bias_flags;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const auto has_bias = ctx->saved_data["bias"].toIntVector();
    const Tensor& x = saved[0];
    c10::DeviceGuard guard(x.device());
    Tensor dx;
    variable_list grads{Tensor()};
    size_t edge = 1;
    if (at::GradMode::is_enabled()) {
      for (size_t i = 0; i < has_bias.size(); ++i) {
        const bool dw = ctx->needs_input_grad(edge++), db = has_bias[i] && ctx->needs_input_grad(edge++);
        auto r = linear_recorded(g[i], x, saved[1 + i], ctx->needs_input_grad(0), dw, db);
        if (r.dx.defined()) dx = dx.defined() ? dx + r.dx : r.dx;
        grads.push_back(r.dw);
        if (has_bias[i]) grads.push_back(r.db);
      }
      grads[0] = dx;
      grads.push_back(Tensor());
      return grads;
    }
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor x2 = flat(x);
    variable_list wanted;             // the gradients whose layers want a weight gradient,
    std::vector<size_t> place;        // and where in `grads` it goes
    variable_list all, weights;
    for (size_t i = 0; i < has_bias.size(); ++i) {
      const Tensor& w = saved[1 + i];
      const Tensor g2 = flat(g[i]);
      all.push_back(g2);
      weights.push_back(w);
      if (ctx->needs_input_grad(edge++)) {
        wanted.push_back(g2);
        place.push_back(grads.size());
      }
      grads.push_back(Tensor());
      if (has_bias[i]) grads.push_back(ctx->needs_input_grad(edge++) ? bias_grad(g2) : Tensor());
    }
    if (ctx->needs_input_grad(0)) dx = input_grads(all, weights);
    if (wanted.size() <= 3) {
      const variable_list dw = wanted.empty() ? variable_list() : weight_grads(wanted, x2);
      for (size_t i = 0; i < dw.size(); ++i) grads[place[i]] = dw[i];
    } else {
      for (size_t i = 0; i < wanted.size(); ++i) grads[place[i]] = weight_grads({wanted[i]}, x2)[0];
    }
    grads[0] = dx.defined() ? dx.view(x.sizes()) : Tensor();
    grads.push_back(Tensor());
    return grads;
  }
};
std::vector<Tensor> linear_group(const Tensor& x, const std::vector<Tensor>& params, const std::vector<bool>& has_bias) {
  bool recorded = wants_grad({&x});
  for (const Tensor& t : params) recorded = recorded || wants_grad({&t});
  if (recorded) return LinearGroupFn::apply(x, at::TensorList(params), has_bias);
  variable_list weights;
  std::vector<Optional> biases;
  size_t at_ = 0;
  for (const bool b : has_bias) {
    weights.push_back(params[at_++]);
    biases.push_back(b ? Optional(params[at_++]) : Optional());
  }
  if (auto y = products(x, weights, biases, Optional()); y.has_value()) return *y;
  variable_list out;
  for (size_t i = 0; i < weights.size(); ++i) out.push_back(linear_raw(x, weights[i], biases[i], Optional()));
  return out;
}

}  // namespace

void bind_ops(py::module_& m) {
  // a launch may wait for room in the stream's queue: not with the interpreter held
  using free = py::call_guard<py::gil_scoped_release>;
  m.def("transpose_last2", &transpose_last2, free());
  m.def("silu_mul", &silu_mul, free());
  m.def("layer_norm_plus_one", &layer_norm_plus_one, free());
  m.def("qk_norm_rotary", &qk_norm_rotary, free());
  m.def("timestep_norm_layer", &timestep_norm_layer, free());
  m.def("tsn_last_workspaces", &tsn_last_workspaces, free());
  m.def("cema", &cema, free());
  m.def("cema_state", &cema_state, free());
  m.def("attention", &attention, free());
  m.def("linear", &linear, free());
  m.def("linear_group", &linear_group, free());
}

}  // namespace mega_host
