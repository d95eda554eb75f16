// The one-token step of a block on a cache (csrc/block_decode.hip).
#include "host.hpp"

#include <tuple>
#include <vector>

namespace mega_host {
namespace {

using Optional = std::optional<Tensor>;
// (out, ((keys, values, length), (count, mean, var), state))
using Step = std::tuple<Tensor, std::tuple<std::tuple<Tensor, Tensor, int64_t>, std::tuple<Tensor, Tensor, Tensor>, Tensor>>;

// The step, or None where the step kernels do not take the sizes, types or layouts (the caller then
// goes operator by operator).  `weights` in the order of the enumeration below.
enum { kTsnW, kTsnB, kOmega, kRmsW, kWz, kBz, kWr, kBr, kWh1, kBh1, kWv, kBv, kWh2, kGamma, kBeta, kLnW, kLnB, kFc1, kFc2, kFc3, kWeights };

std::optional<Step> block_decode_step(const Tensor& x, const Tensor& k, const Tensor& v, const Tensor& prev_count,
                             const Tensor& prev_mean, const Tensor& prev_var, const Tensor& hx, const Optional& freqs,
                             const std::vector<Optional>& weights, const Tensor& p, const Tensor& q, const Tensor& gamma_hat,
                             int64_t heads, int64_t groups, int64_t chunk, double tsn_eps, double rms_eps, double z_eps,
                             double ln_eps) {
  const auto type = x.scalar_type();
  const int dtype = code_of(type);
  if (dtype != MEGA_BF16 && dtype != MEGA_F16) return std::nullopt;
  const auto dev = x.device();
  if (!x.is_cuda() || static_cast<int>(weights.size()) != kWeights) return std::nullopt;
  if (x.dim() != 3 || x.size(1) != 1 || k.dim() != 4 || p.dim() < 2 || heads < 1) return std::nullopt;
  // a forward-mode tangent goes to the operators, which refuse it, and so does a lazily conjugated or negated
  // view, which they resolve
  for (const Tensor* t : {&x, &k, &v, &prev_count, &prev_mean, &prev_var, &hx})
    if (has_tangent(*t) || lazy(*t)) return std::nullopt;
  if (freqs.has_value() && lazy(*freqs)) return std::nullopt;
  const auto aligned = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  for (int i = 0; i < kWeights; ++i) {
    const Optional& w = weights[i];
    const bool may_lack = i == kRmsW || i == kBz || i == kBr || i == kBh1 || i == kBv || i == kLnW || i == kLnB;
    if (!w.has_value()) {
      if (may_lack) continue;
      return std::nullopt;
    }
    if (has_tangent(*w) || lazy(*w) || w->scalar_type() != type || w->device() != dev || !w->is_contiguous() || !aligned(*w)) return std::nullopt;
  }
  const int64_t B = x.size(0), D = x.size(2), S = weights[kWz]->size(0), E = weights[kWv]->size(0), F = weights[kFc1]->size(0),
                N = p.size(1), n = k.size(1);
  const int64_t rows[kWeights] = {1, 1, 1, 1, S, 1, E, 1, D, 1, E, 1, D, 2, 2, 1, 1, F, D, F};
  const int64_t cols[kWeights] = {D, D, D, D, D, S, D, E, D, D, D, E, E, S, S, D, D, D, F, D};
  for (int i = 0; i < kWeights; ++i)  // (the operators refuse what does not fit)
    if (weights[i].has_value() && (weights[i]->numel() != rows[i] * cols[i] || (rows[i] > 1 && weights[i]->size(-1) != cols[i]))) return std::nullopt;
  if (!mega_block_decode_supported(dtype, B, D, S, E, F, heads, groups, N)) return std::nullopt;
  const auto is = [&](const Tensor& t, at::ScalarType ty, at::IntArrayRef shape) {
    return t.scalar_type() == ty && t.device() == dev && t.sizes() == shape && t.is_contiguous();
  };
  if (!is(prev_count, at::kLong, {B}) || !is(prev_mean, type, {B, groups}) || !is(prev_var, type, {B, groups}) ||
      !is(hx, at::kComplexFloat, {B, D, N}) || !aligned(hx) || !x.is_contiguous())
    return std::nullopt;
  if (k.scalar_type() != type || v.scalar_type() != type || k.device() != dev || v.device() != dev ||
      k.sizes() != at::IntArrayRef({B, n, heads, S / heads}) || v.sizes() != at::IntArrayRef({B, n, heads, E / heads}) || n < 1)
    return std::nullopt;
  if (p.scalar_type() != at::kFloat || q.scalar_type() != at::kComplexFloat || gamma_hat.scalar_type() != at::kComplexFloat ||
      p.numel() != D * N || q.numel() != D * N || gamma_hat.numel() != D * N || !p.is_contiguous() || !q.is_contiguous() ||
      !gamma_hat.is_contiguous() || !aligned(p) || !aligned(q) || !aligned(gamma_hat) || p.device() != dev)
    return std::nullopt;
  if (freqs.has_value() && !is(*freqs, at::kComplexFloat, {1, S / heads / 2})) return std::nullopt;

  c10::DeviceGuard guard(dev);
  const auto dense = [&](const Tensor& t) {
    const Tensor c = t.contiguous();
    return aligned(c) ? c : c.clone(at::MemoryFormat::Contiguous);
  };
  const Tensor k_in = dense(k), v_in = dense(v);
  // the cache that is handed back is the caller's own, as a concatenation would be: it shares nothing with
  // the old one, whatever streams, threads or later writes the two meet
  Tensor k_out = at::empty({B, n + 1, heads, S / heads}, x.options()), v_out = at::empty({B, n + 1, heads, E / heads}, x.options());
  const auto ptr = [](const Optional& t) { return t.has_value() ? t->data_ptr() : nullptr; };
  Tensor y = at::empty_like(x), count = at::empty_like(prev_count), mean = at::empty_like(prev_mean),
         var = at::empty_like(prev_var), h = at::empty_like(hx);
  mega_block_decode_args a{};
  a.dtype = dtype;
  a.B = B, a.D = D, a.S = S, a.E = E, a.F = F, a.heads = heads, a.G = groups, a.N = N;
  a.length = n;
  a.tsn_eps = tsn_eps, a.rms_eps = rms_eps, a.z_eps = z_eps, a.ln_eps = ln_eps;
  a.x = x.data_ptr();
  a.prev_count = prev_count.data_ptr<int64_t>(), a.prev_mean = prev_mean.data_ptr(), a.prev_var = prev_var.data_ptr();
  a.tsn_weight = ptr(weights[kTsnW]), a.tsn_bias = ptr(weights[kTsnB]);
  a.p = p.data_ptr<float>(), a.q = static_cast<const float*>(q.data_ptr()),
  a.gamma_hat = static_cast<const float*>(gamma_hat.data_ptr()), a.omega = ptr(weights[kOmega]);
  a.h_in = static_cast<const float*>(hx.data_ptr()), a.rms_weight = ptr(weights[kRmsW]);
  a.wz = ptr(weights[kWz]), a.bz = ptr(weights[kBz]), a.wr = ptr(weights[kWr]), a.br = ptr(weights[kBr]);
  a.wh1 = ptr(weights[kWh1]), a.bh1 = ptr(weights[kBh1]), a.wv = ptr(weights[kWv]), a.bv = ptr(weights[kBv]);
  a.wh2 = ptr(weights[kWh2]), a.qk_gamma = ptr(weights[kGamma]), a.qk_beta = ptr(weights[kBeta]);
  a.freqs = freqs.has_value() ? static_cast<const float*>(freqs->data_ptr()) : nullptr;
  a.ln_weight = ptr(weights[kLnW]), a.ln_bias = ptr(weights[kLnB]);
  a.fc1 = ptr(weights[kFc1]), a.fc2 = ptr(weights[kFc2]), a.fc3 = ptr(weights[kFc3]);
  a.k_in = k_in.data_ptr(), a.v_in = v_in.data_ptr(), a.k_out = k_out.data_ptr(), a.v_out = v_out.data_ptr();
  a.y = y.data_ptr(), a.count = count.data_ptr<int64_t>(), a.mean = mean.data_ptr(), a.var = var.data_ptr();
  a.h_out = static_cast<float*>(h.data_ptr());
  Tensor ws = at::empty({mega_block_decode_workspace_bytes(&a)}, x.options().dtype(at::kByte));
  a.workspace = ws.data_ptr();
  check(mega_block_decode(&a, stream_of(x)), "mega_block_decode");
  const int64_t total = n + 1, tail = total % chunk;  // (0: the chunk is closed and its cache given up)
  return Step{y, {{k_out.narrow(1, total - tail, tail), v_out.narrow(1, total - tail, tail), tail}, {count, mean, var}, h}};
}

}  // namespace

void bind_decode(py::module_& m) {
  // a launch may wait for room in the stream's queue: not with the interpreter held
  m.def("block_decode_step", &block_decode_step, py::call_guard<py::gil_scoped_release>());
}

}  // namespace mega_host
