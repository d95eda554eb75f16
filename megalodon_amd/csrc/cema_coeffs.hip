// CEMA coefficients from the raw parameters and their gradients, one launch each.
//
// Follows MultiHeadComplexEMA._calc_coeffs
// (megalodon/modules/complex_exponential_moving_average.py:100-117):
//   a = sigmoid(alpha), d = sigmoid(delta), t = sigmoid(theta)
//   p = a,  q = rho e^(i phi) with rho = 1 - a d, phi = n t 2 pi / N  (n = 1 .. N)
//   gamma_hat = (gamma_0 + i gamma_1) sqrt(1 / N)
// The weight operator wants log q, which is (ln rho, phi): it is written
// directly, no complex logarithm.  In the reference (and in the module's
// general path here) these are ~30 elementwise PyTorch kernels on (D, N)
// tensors per training step, forward and backward, each bound by its launch.
//
// Backward: with (dq_r, dq_i) the gradient of the loss w.r.t. (Re q, Im q)
// (PyTorch's convention for complex gradients), dp real, dgamma_hat complex,
//   drho = dq_r cos phi + dq_i sin phi,     dphi = rho (dq_i cos phi - dq_r sin phi)
//   dalpha = (dp - d drho) a (1 - a),       ddelta = -a drho d (1 - d)
//   dtheta = t (1 - t) (2 pi / N) sum_n n dphi_n
//   dgamma = sqrt(1 / N) (Re dgamma_hat, Im dgamma_hat)
#include "common.hpp"
#include "cema_pow.hpp"

namespace mega {
namespace {

constexpr int kThreads = 256;

template <int DT>
__global__ __launch_bounds__(kThreads) void cema_coeffs_fwd_kernel(
    const typename Elem<DT>::type* __restrict__ alpha, const typename Elem<DT>::type* __restrict__ delta,
    const typename Elem<DT>::type* __restrict__ theta, const typename Elem<DT>::type* __restrict__ gamma, int64_t D, int N,
    float* __restrict__ p, float* __restrict__ log_q, float* __restrict__ gamma_hat) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= D * N) return;
  const int64_t ch = i / N;
  const int n = static_cast<int>(i % N);
  using E = Elem<DT>;
  const CemaCoeffs c = cema_coeffs(E::load(alpha + i), E::load(delta + i), E::load(theta + ch), n, N);
  p[i] = c.p;
  log_q[2 * i] = c.log_rho;
  log_q[2 * i + 1] = c.phi;
  gamma_hat[2 * i] = E::load(gamma + 2 * i) * c.scale;
  gamma_hat[2 * i + 1] = E::load(gamma + 2 * i + 1) * c.scale;
}

// One thread per (channel, mode); the sum over the modes of a channel runs
// through LDS (N <= 64, a workgroup holds whole channels).  The incoming gradients
// are `sets` stacks (one per sequence, and per piece of a split tensor) that are added up
// here, in order: separate sums over the batch would be four more launches.
template <int DT>
__global__ __launch_bounds__(kThreads) void cema_coeffs_bwd_kernel(
    const float* __restrict__ dp, const float2* __restrict__ dq, const float2* __restrict__ dgamma_hat,
    const float* __restrict__ dskip, int64_t sets, const typename Elem<DT>::type* __restrict__ alpha,
    const typename Elem<DT>::type* __restrict__ delta, const typename Elem<DT>::type* __restrict__ theta, int64_t D,
    int N, int ch_per_block, typename Elem<DT>::type* __restrict__ dalpha, typename Elem<DT>::type* __restrict__ ddelta,
    typename Elem<DT>::type* __restrict__ dtheta, typename Elem<DT>::type* __restrict__ dgamma,
    typename Elem<DT>::type* __restrict__ domega) {
  using E = Elem<DT>;
  __shared__ float s_phi[kThreads];
  const int local_ch = threadIdx.x / N, n = threadIdx.x % N;
  const int64_t ch = static_cast<int64_t>(blockIdx.x) * ch_per_block + local_ch;
  const bool on = local_ch < ch_per_block && ch < D;
  float contrib = 0.f;
  if (on) {
    const int64_t i = ch * N + n;
    float gp = 0.f, qr = 0.f, qi = 0.f, hr = 0.f, hi = 0.f, gw = 0.f;
    for (int64_t k = 0; k < sets; ++k) {
      const int64_t j = k * D * N + i;
      const float2 q = dq[j], h = dgamma_hat[j];
      gp += dp[j];
      qr += q.x;
      qi += q.y;
      hr += h.x;
      hi += h.y;
      if (n == 0 && dskip != nullptr) gw += dskip[k * D + ch];
    }
    const float a = cema_sigmoid(E::load(alpha + i)), d = cema_sigmoid(E::load(delta + i)), t = cema_sigmoid(E::load(theta + ch));
    const float rho = 1.f - a * d;
    const float phi = static_cast<float>(n + 1) * (t * (6.283185307179586f / static_cast<float>(N)));
    float sn, cs;
    sincosf(phi, &sn, &cs);
    const float drho = qr * cs + qi * sn;
    const float dphi = rho * (qi * cs - qr * sn);
    E::store(dalpha + i, (gp - d * drho) * a * (1.f - a));
    E::store(ddelta + i, -a * drho * d * (1.f - d));
    const float scale = sqrtf(1.f / static_cast<float>(N));
    E::store(dgamma + 2 * i, hr * scale);
    E::store(dgamma + 2 * i + 1, hi * scale);
    if (n == 0 && domega != nullptr) E::store(domega + ch, gw);
    contrib = static_cast<float>(n + 1) * dphi;
  }
  s_phi[threadIdx.x] = contrib;
  __syncthreads();
  if (on && n == 0) {
    float s = 0.f;
    for (int k = 0; k < N; ++k) s += s_phi[local_ch * N + k];
    const float t = cema_sigmoid(E::load(theta + ch));
    E::store(dtheta + ch, t * (1.f - t) * (6.283185307179586f / static_cast<float>(N)) * s);
  }
}

template <int DT>
int launch_fwd(const void* alpha, const void* delta, const void* theta, const void* gamma, int64_t D, int64_t N,
               float* p, float* log_q, float* gamma_hat, hipStream_t s) {
  using T = typename Elem<DT>::type;
  const int64_t blocks = (D * N + kThreads - 1) / kThreads;
  cema_coeffs_fwd_kernel<DT><<<dim3(static_cast<unsigned>(blocks)), kThreads, 0, s>>>(
      static_cast<const T*>(alpha), static_cast<const T*>(delta), static_cast<const T*>(theta),
      static_cast<const T*>(gamma), D, static_cast<int>(N), p, log_q, gamma_hat);
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}
template <int DT>
int launch_bwd(const float* dp, const float* dq, const float* dgamma_hat, const float* dskip, int64_t sets,
               const void* alpha, const void* delta, const void* theta, int64_t D, int64_t N, void* dalpha,
               void* ddelta, void* dtheta, void* dgamma, void* domega, hipStream_t s) {
  using T = typename Elem<DT>::type;
  const int cpb = kThreads / static_cast<int>(N);
  const int64_t blocks = (D + cpb - 1) / cpb;
  MEGA_CHECK_ARG(blocks <= 0x7fffffff, "mega_cema_coeffs_bwd: too many channels");
  cema_coeffs_bwd_kernel<DT><<<dim3(static_cast<unsigned>(blocks)), kThreads, 0, s>>>(
      dp, reinterpret_cast<const float2*>(dq), reinterpret_cast<const float2*>(dgamma_hat), dskip, sets,
      static_cast<const T*>(alpha), static_cast<const T*>(delta), static_cast<const T*>(theta), D,
      static_cast<int>(N), cpb, static_cast<T*>(dalpha), static_cast<T*>(ddelta), static_cast<T*>(dtheta),
      static_cast<T*>(dgamma), static_cast<T*>(domega));
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_cema_layer_coeffs_fwd(int dtype, const void* alpha, const void* delta, const void* theta,
                                          const void* gamma, int64_t D, int64_t N, float* p, float* log_q,
                                          float* gamma_hat, void* stream) {
  MEGA_CHECK_ARG(valid_dtype(dtype), "mega_cema_coeffs_fwd: bad dtype %d", dtype);
  MEGA_CHECK_ARG(alpha && delta && theta && gamma && p && log_q && gamma_hat,
                 "mega_cema_coeffs_fwd: null pointer");
  MEGA_CHECK_ARG(D >= 0 && N >= 1 && N <= 64, "mega_cema_coeffs_fwd: need D >= 0 and 1 <= N <= 64");
  if (D == 0) return MEGA_OK;
  MEGA_CHECK_ARG(D * N <= (1ll << 38), "mega_cema_coeffs_fwd: too many elements");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MEGA_F32) return launch_fwd<MEGA_F32>(alpha, delta, theta, gamma, D, N, p, log_q, gamma_hat, s);
  if (dtype == MEGA_BF16) return launch_fwd<MEGA_BF16>(alpha, delta, theta, gamma, D, N, p, log_q, gamma_hat, s);
  return launch_fwd<MEGA_F16>(alpha, delta, theta, gamma, D, N, p, log_q, gamma_hat, s);
}

extern "C" int mega_cema_layer_coeffs_bwd(int dtype, const float* dp, const float* dq, const float* dgamma_hat,
                                          const float* dskip, int64_t sets, const void* alpha, const void* delta,
                                          const void* theta, int64_t D, int64_t N, void* dalpha, void* ddelta,
                                          void* dtheta, void* dgamma, void* domega, void* stream) {
  MEGA_CHECK_ARG(valid_dtype(dtype), "mega_cema_coeffs_bwd: bad dtype %d", dtype);
  MEGA_CHECK_ARG(dp && dq && dgamma_hat && alpha && delta && theta && dalpha && ddelta && dtheta &&
                     dgamma,
                 "mega_cema_coeffs_bwd: null pointer");
  MEGA_CHECK_ARG(D >= 0 && N >= 1 && N <= 64 && sets >= 0, "mega_cema_coeffs_bwd: need D >= 0 and 1 <= N <= 64");
  MEGA_CHECK_ARG(domega == nullptr || dskip != nullptr, "mega_cema_coeffs_bwd: domega without its rows");
  if (D == 0) return MEGA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto go = dtype == MEGA_F32 ? launch_bwd<MEGA_F32> : dtype == MEGA_BF16 ? launch_bwd<MEGA_BF16> : launch_bwd<MEGA_F16>;
  return go(dp, dq, dgamma_hat, dskip, sets, alpha, delta, theta, D, N, dalpha, ddelta, dtheta, dgamma, domega, s);
}

extern "C" int mega_cema_coeffs_fwd(const float* alpha, const float* delta, const float* theta,
                                    const float* gamma, int64_t D, int64_t N, float* p,
                                    float* log_q, float* gamma_hat, void* stream) {
  return mega_cema_layer_coeffs_fwd(MEGA_F32, alpha, delta, theta, gamma, D, N, p, log_q, gamma_hat, stream);
}

extern "C" int mega_cema_coeffs_bwd(const float* dp, const float* dq, const float* dgamma_hat,
                                    const float* alpha, const float* delta, const float* theta,
                                    int64_t D, int64_t N, float* dalpha, float* ddelta,
                                    float* dtheta, float* dgamma, void* stream) {
  return mega_cema_layer_coeffs_bwd(MEGA_F32, dp, dq, dgamma_hat, nullptr, 1, alpha, delta, theta, D, N, dalpha, ddelta,
                                    dtheta, dgamma, nullptr, stream);
}
