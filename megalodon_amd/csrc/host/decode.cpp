// Generation from a cache: room for new keys and values behind the old ones, and the one-token
// step of a block (csrc/block_decode.hip).
#include "host.hpp"

#include <algorithm>
#include <memory>
#include <vector>

namespace mega_host {
namespace {

// Storage behind a cache's keys and values with room for tokens to come.  The cache that a
// caller holds is a view of its first tokens; the buffer travels with that view (attribute
// `_mega_kv` of the key tensor) and goes when the last view goes.  `used` tokens are taken by the
// longest view handed out: a caller that continues from an older, shorter cache while
// the longer one is alive gets a copy, so nothing that was returned ever changes.
struct KvBuffer {
  Tensor k, v;
  int64_t used = 0;
};
constexpr const char* kAttr = "_mega_kv";
constexpr int64_t kRoom = 256;  // room is made in steps of this many tokens: one copy of the cache per step

// whether `view` is the first tokens of `whole`
bool starts(const Tensor& view, const Tensor& whole) {
  return view.data_ptr() == whole.data_ptr() && view.dim() == 4 && view.strides() == whole.strides() &&
         view.size(0) == whole.size(0) && view.size(1) <= whole.size(1) && view.sizes().slice(2) == whole.sizes().slice(2);
}

// A buffer that holds the old tokens of (k, v) and has room for `more` behind them; `chunk` is the
// length at which the cache is given up.
std::shared_ptr<KvBuffer> room_for(const py::object& k_obj, const Tensor& k, const Tensor& v, int64_t more, int64_t chunk) {
  const int64_t n = k.size(1);
  py::object held = py::getattr(k_obj, kAttr, py::none());
  if (!held.is_none()) {
    auto buf = held.cast<std::shared_ptr<KvBuffer>>();
    // nothing lies behind the old tokens, or nobody holds it any more: the buffer and this
    // cache are then the only owners of the storage
    const bool free = buf->used == n || (buf->k.storage().use_count() == 2 && buf->v.storage().use_count() == 2);
    if (free && n + more <= buf->k.size(1) && starts(k, buf->k) && starts(v, buf->v)) return buf;
  }
  auto buf = std::make_shared<KvBuffer>();
  const int64_t total = n + more;
  // (strides of whole 16-byte pieces come with head widths that are multiples of 8)
  const int64_t cap = total >= chunk ? total : std::min(chunk, (total + kRoom / 4 + kRoom - 1) / kRoom * kRoom);
  buf->k = at::empty({k.size(0), cap, k.size(2), k.size(3)}, k.options());
  buf->v = at::empty({v.size(0), cap, v.size(2), v.size(3)}, v.options());
  if (n > 0) {
    buf->k.narrow(1, 0, n).copy_(k);
    buf->v.narrow(1, 0, n).copy_(v);
  }
  buf->used = n;
  return buf;
}

// the views of `buf` that hold tokens lo .. hi - 1
py::tuple views_of(const std::shared_ptr<KvBuffer>& buf, int64_t lo, int64_t hi) {
  py::object k = py::cast(buf->k.narrow(1, lo, hi - lo)), v = py::cast(buf->v.narrow(1, lo, hi - lo));
  if (lo == 0) py::setattr(k, kAttr, py::cast(buf));
  return py::make_tuple(k, v);
}

// (keys, values) of the old and the new tokens together, in storage with room for more; None for
// operands that are not one batch of one type (the caller concatenates)
py::object kv_append(const py::object& k_obj, const Tensor& v, const Tensor& k_new, const Tensor& v_new, int64_t chunk) {
  const Tensor k = k_obj.cast<Tensor>();
  const auto joins = [](const Tensor& a, const Tensor& b) {
    return a.dim() == 4 && b.dim() == 4 && a.size(0) == b.size(0) && a.sizes().slice(2) == b.sizes().slice(2) &&
           a.scalar_type() == b.scalar_type() && a.device() == b.device() && !has_tangent(a) && !has_tangent(b);
  };
  if (!joins(k, k_new) || !joins(v, v_new) || k.size(1) != v.size(1) || k_new.size(1) != v_new.size(1)) return py::none();
  const int64_t n = k.size(1), more = k_new.size(1);
  auto buf = room_for(k_obj, k, v, more, chunk);
  buf->k.narrow(1, n, more).copy_(k_new);
  buf->v.narrow(1, n, more).copy_(v_new);
  buf->used = n + more;
  return views_of(buf, 0, n + more);
}

using Optional = std::optional<Tensor>;

// The step, or None where the step kernels do not take the sizes, types or layouts (the caller then
// goes operator by operator).  `weights` in the order of the enumeration below.
enum { kTsnW, kTsnB, kOmega, kRmsW, kWz, kBz, kWr, kBr, kWh1, kBh1, kWv, kBv, kWh2, kGamma, kBeta, kLnW, kLnB, kFc1, kFc2, kFc3, kWeights };

py::object block_decode_step(const Tensor& x, const py::object& k_obj, const Tensor& v, const Tensor& prev_count,
                             const Tensor& prev_mean, const Tensor& prev_var, const Tensor& hx, const Optional& freqs,
                             const std::vector<Optional>& weights, const Tensor& p, const Tensor& q, const Tensor& gamma_hat,
                             int64_t heads, int64_t groups, int64_t chunk, double tsn_eps, double rms_eps, double z_eps,
                             double ln_eps) {
  const Tensor k = k_obj.cast<Tensor>();
  const auto type = x.scalar_type();
  const int dtype = code_of(type);
  if (dtype != MEGA_BF16 && dtype != MEGA_F16) return py::none();
  const auto dev = x.device();
  if (!x.is_cuda() || static_cast<int>(weights.size()) != kWeights) return py::none();
  // a forward-mode tangent goes to the operators, which refuse it
  for (const Tensor* t : {&x, &k, &v, &prev_mean, &prev_var, &hx})
    if (has_tangent(*t)) return py::none();
  const auto aligned = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  for (int i = 0; i < kWeights; ++i) {
    const Optional& w = weights[i];
    const bool may_lack = i == kRmsW || i == kBz || i == kBr || i == kBh1 || i == kBv || i == kLnW || i == kLnB;
    if (!w.has_value()) {
      if (may_lack) continue;
      return py::none();
    }
    if (has_tangent(*w) || w->scalar_type() != type || w->device() != dev || !w->is_contiguous() || !aligned(*w)) return py::none();
  }
  const int64_t B = x.size(0), D = x.size(2), S = weights[kWz]->size(0), E = weights[kWv]->size(0), F = weights[kFc1]->size(0),
                N = p.size(1), n = k.size(1);
  if (!mega_block_decode_supported(dtype, B, D, S, E, F, heads, groups, N)) return py::none();
  const auto is = [&](const Tensor& t, at::ScalarType ty, at::IntArrayRef shape) {
    return t.scalar_type() == ty && t.device() == dev && t.sizes() == shape && t.is_contiguous();
  };
  if (!is(prev_count, at::kLong, {B}) || !is(prev_mean, type, {B, groups}) || !is(prev_var, type, {B, groups}) ||
      !is(hx, at::kComplexFloat, {B, D, N}) || !aligned(hx) || !x.is_contiguous())
    return py::none();
  if (k.scalar_type() != type || v.scalar_type() != type || k.device() != dev || v.device() != dev ||
      k.sizes() != at::IntArrayRef({B, n, heads, S / heads}) || v.sizes() != at::IntArrayRef({B, n, heads, E / heads}) || n < 1)
    return py::none();
  if (p.scalar_type() != at::kFloat || q.scalar_type() != at::kComplexFloat || gamma_hat.scalar_type() != at::kComplexFloat ||
      p.numel() != D * N || q.numel() != D * N || gamma_hat.numel() != D * N || !p.is_contiguous() || !q.is_contiguous() ||
      !gamma_hat.is_contiguous() || !aligned(p) || !aligned(q) || !aligned(gamma_hat) || p.device() != dev)
    return py::none();
  if (freqs.has_value() && !is(*freqs, at::kComplexFloat, {1, S / heads / 2})) return py::none();

  c10::DeviceGuard guard(dev);
  auto buf = room_for(k_obj, k, v, 1, chunk);
  const auto ptr = [](const Optional& t) { return t.has_value() ? t->data_ptr() : nullptr; };
  Tensor y = at::empty_like(x), count = at::empty_like(prev_count), mean = at::empty_like(prev_mean),
         var = at::empty_like(prev_var), h = at::empty_like(hx);
  mega_block_decode_args a{};
  a.dtype = dtype;
  a.B = B, a.D = D, a.S = S, a.E = E, a.F = F, a.heads = heads, a.G = groups, a.N = N;
  a.length = n, a.k_stride = buf->k.stride(0), a.v_stride = buf->v.stride(0);
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
  a.k_cache = buf->k.data_ptr(), a.v_cache = buf->v.data_ptr();
  a.y = y.data_ptr(), a.count = count.data_ptr<int64_t>(), a.mean = mean.data_ptr(), a.var = var.data_ptr();
  a.h_out = static_cast<float*>(h.data_ptr());
  Tensor ws = at::empty({mega_block_decode_workspace_bytes(&a)}, x.options().dtype(at::kByte));
  a.workspace = ws.data_ptr();
  check(mega_block_decode(&a, stream_of(x)), "mega_block_decode");
  buf->used = n + 1;
  const int64_t total = n + 1, tail = total % chunk;
  py::tuple kv = views_of(buf, total - tail, total);
  return py::make_tuple(y, py::make_tuple(py::make_tuple(kv[0], kv[1], tail), py::make_tuple(count, mean, var), h));
}

}  // namespace

void bind_decode(py::module_& m) {
  py::class_<KvBuffer, std::shared_ptr<KvBuffer>>(m, "KvBuffer").def_readonly("used", &KvBuffer::used);
  m.def("kv_append", &kv_append);
  m.def("block_decode_step", &block_decode_step);
}

}  // namespace mega_host
