// Causal FFT convolution for gfx950.
//
// Semantics follow megalodon/modules/fused_ops/fftconv.py:30-75:
//   forward   y  = irfft(rfft(x, 2N) * rfft(k, 2N))[:L]
//   backward  dx = flip(conv(flip(dy), k)),  dk = sum_b flip(conv(flip(dy_b), x_b))
// One workgroup convolves one (batch, channel) row entirely on chip: the row
// is read once per half (see fftconv_core.hpp), transformed with 32 complex
// points per lane in registers, multiplied with the parked spectrum of the
// other operand and transformed back; nothing but the rows themselves touches
// HBM (the reference's torch.fft path at L > 16384 makes ~7 full round trips
// and saves the 1 GiB spectra x_f / k_f for backward; here backward recomputes
// the spectra from x and k).
//
// Rows with L <= 2048 use a direct time-domain kernel (exact, O(L^2) per row).
#include "common.hpp"
#include "fftconv_mfma.hpp"
#include "fftconv_rows.hpp"

#include <mutex>

namespace mega {

TableCache fft_tables;

namespace {

// ------------------------------ direct kernel --------------------------------
// L <= 2048 (the transforms are as accurate and from some 1200 steps on faster, but these sums are causal to the last bit,
// also around values that are not finite, and need no tables under capture): time-domain sums with both rows staged in LDS, each output's terms in ascending order of
// the first row's index.  Bound by the multiply-adds: a thread owns R neighbouring outputs and moves a
// window of the second row through registers, so that four steps cost two 16-byte LDS reads and 4 R
// multiply-adds (one output at a time, two reads fed one).  Eight outputs per
// thread cover 2048 with the workgroup's four waves; rows of at most 1024 take four, so that
// their waves all have work.  A wave's share grows with its outputs' index, so the waves of a workgroup
// take the shares in an order that turns with the workgroup: the SIMDs of a compute unit get equal sums.
// Forward / backward of 2 x 1024 rows in bfloat16: 600 steps 49 / 152 -> 24 / 49 us, 1024 steps
// 103 / 326 -> 41 / 85, 2048 steps 374 / 1177 -> 132 / 269, the same bits.
constexpr int kDirectMaxL = 2048;
constexpr int kDirectThreads = 256;

template <int DT, int MODE, int R>
__global__ __launch_bounds__(kDirectThreads) void direct_conv_kernel(
    const void* __restrict__ a, const void* __restrict__ b, void* __restrict__ out, int B, int D,
    int L, int flip, const float* __restrict__ omega) {
  constexpr int kMax = kDirectThreads * R;  // L <= kMax
  __shared__ __align__(16) float sa[kMax];
  __shared__ __align__(16) float sb[kMax];
  const int64_t esz = DT == MEGA_F32 ? 4 : 2;
  const int nb = MODE == 0 ? 1 : B;
  const int64_t d = MODE == 0 ? blockIdx.x % D : blockIdx.x;
  const bool fl = MODE == 1 || flip != 0;
  const int i0 = R * static_cast<int>((threadIdx.x + (blockIdx.x % (kDirectThreads / kWave)) * kWave) % kDirectThreads);
  float total[R];
  for (int bb = 0; bb < nb; ++bb) {
    const int64_t row = MODE == 0 ? blockIdx.x : static_cast<int64_t>(bb) * D + d;
    const char* arow = static_cast<const char*>(a) + row * L * esz;
    __syncthreads();
    for (int i = threadIdx.x; i < L; i += kDirectThreads) {
      sa[i] = ld<DT>(arow, fl ? L - 1 - i : i);
      if (MODE == 0)
        sb[i] = static_cast<const float*>(b)[d * L + i];
      else
        sb[i] = ld<DT>(static_cast<const char*>(b) + row * L * esz, i);
    }
    __syncthreads();
    if (i0 < L) {
      // (values behind L reach only outputs behind L)
      float acc[R], win[R + 4];  // win[4 + r] = sb[i0 + r - s]
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] = 0.f;
#pragma unroll
      for (int r = 0; r < R; r += 4) {
        const float4 v = *reinterpret_cast<const float4*>(sb + i0 + r);
        win[4 + r] = v.x, win[5 + r] = v.y, win[6 + r] = v.z, win[7 + r] = v.w;
      }
#pragma unroll 3
      for (int s = 0; s < i0; s += 4) {
        const float4 v = *reinterpret_cast<const float4*>(sb + (i0 - s - 4));
        const float4 u = *reinterpret_cast<const float4*>(sa + s);
        win[0] = v.x, win[1] = v.y, win[2] = v.z, win[3] = v.w;
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = fmaf(win[4 + r], u.x, acc[r]);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = fmaf(win[3 + r], u.y, acc[r]);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = fmaf(win[2 + r], u.z, acc[r]);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = fmaf(win[1 + r], u.w, acc[r]);
#pragma unroll
        for (int i = R + 3; i >= 4; --i) win[i] = win[i - 4];
      }
#pragma unroll
      for (int u = 0; u < R; ++u)
#pragma unroll
        for (int r = u; r < R; ++r) acc[r] = fmaf(win[4 + r - u], sa[i0 + u], acc[r]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (MODE == 0) {
          const int i = i0 + r;
          if (omega != nullptr) acc[r] = fmaf(omega[d], sa[i], acc[r]);  // sa[i] is a[o]
          if (i < L) st<DT>(static_cast<char*>(out) + row * L * esz, fl ? L - 1 - i : i, acc[r]);
        } else {
          total[r] = bb == 0 ? acc[r] : total[r] + acc[r];
        }
      }
    }
  }
  if (MODE == 1) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (i0 + r < L) static_cast<float*>(out)[d * L + L - 1 - (i0 + r)] = total[r];
  }
}

// The transforms are float32 unless MEGA_FFTCONV_F16_STAGES is set (to anything
// but "0") in the environment: then 16-bit rows the matrix-core engine can take
// run its fp16-operand DFT stages (3x faster, error ~1e-3 of the largest
// output instead of ~1e-6).  Read per call.
bool f16_stages_enabled() {
  const char* v = getenv("MEGA_FFTCONV_F16_STAGES");
  return v != nullptr && !(v[0] == '0' && v[1] == 0);
}

template <int DT, int MODE>
int launch_conv(const void* a, const void* b, void* out, int64_t B, int64_t D, int64_t L, int flip,
                const float* omega, hipStream_t stream) {
  if (L <= kDirectMaxL) {
    const int64_t rows = MODE == 0 ? B * D : D;
    MEGA_CHECK_ARG(rows <= 0x7fffffff, "fftconv: too many rows");
    const auto kernel = L <= 4 * kDirectThreads ? direct_conv_kernel<DT, MODE, 4> : direct_conv_kernel<DT, MODE, 8>;
    kernel<<<dim3(static_cast<unsigned>(rows)), kDirectThreads, 0, stream>>>(
        a, b, out, static_cast<int>(B), static_cast<int>(D), static_cast<int>(L), flip, omega);
    MEGA_CHECK_LAUNCH();
    return MEGA_OK;
  }
  // opt-in: 16-bit rows run their DFT stages on the matrix cores with fp16 operands
  if (f16_stages_enabled() && fftm::applicable(DT, L, a, b, out))
    return fftm::launch_conv(DT, MODE, a, b, out, B, D, L, flip, omega, stream);
  if (L <= 4096) return fftconv_rows<11>(DT, MODE, a, b, out, B, D, L, flip, omega, stream);
  if (L <= 8192) return fftconv_rows<12>(DT, MODE, a, b, out, B, D, L, flip, omega, stream);
  if (L <= 16384) return fftconv_rows<13>(DT, MODE, a, b, out, B, D, L, flip, omega, stream);
  return fftconv_rows<14>(DT, MODE, a, b, out, B, D, L, flip, omega, stream);
}

template <int MODE>
int dispatch_conv(int dtype, const void* a, const void* b, void* out, int64_t B, int64_t D,
                  int64_t L, int flip, const float* omega, hipStream_t stream) {
  switch (dtype) {
    case MEGA_F32: return launch_conv<MEGA_F32, MODE>(a, b, out, B, D, L, flip, omega, stream);
    case MEGA_BF16: return launch_conv<MEGA_BF16, MODE>(a, b, out, B, D, L, flip, omega, stream);
    case MEGA_F16: return launch_conv<MEGA_F16, MODE>(a, b, out, B, D, L, flip, omega, stream);
  }
  return set_error(MEGA_ERR_INVALID_ARG, "fftconv: bad dtype %d", dtype);
}

constexpr int64_t kMaxL = 32768;

__global__ void zero_fill_kernel(float* p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_fftconv_max_length(void) { return static_cast<int>(kMaxL); }

extern "C" int mega_fftconv_prepare(int64_t L, void* stream) {
  MEGA_CHECK_ARG(L >= 0, "mega_fftconv_prepare: negative size");
  if (L > kMaxL)
    return set_error(MEGA_ERR_UNSUPPORTED, "mega_fftconv_prepare: L=%lld exceeds the supported %lld",
                     (long long)L, (long long)kMaxL);
  if (L <= kDirectMaxL) return MEGA_OK;  // the time-domain kernel needs neither tables nor scratch
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (L <= 4096) return fftconv_tables<11>(s);
  if (L <= 8192) return fftconv_tables<12>(s);
  if (L <= 16384) return fftconv_tables<13>(s);
  return fftconv_tables<14>(s);
}

// Scratch blocks held on the current device for the transform size that rows
// of L samples take (0 for rows the time-domain kernel takes).
extern "C" int mega_fftconv_scratch_blocks(int64_t L) {
  if (L <= kDirectMaxL || L > kMaxL) return 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kFftDevices) return 0;
  const int size = L <= 4096 ? 0 : L <= 8192 ? 1 : L <= 16384 ? 2 : 3;
  std::lock_guard<std::mutex> lock(fft_tables.mu);
  return static_cast<int>(fft_tables.scratch[dev][size].size());
}

namespace {
int fftconv_fwd_impl(const char* who, const void* x, int dtype, const float* k, const float* omega,
                     int64_t B, int64_t D, int64_t L, void* y, void* stream) {
  MEGA_CHECK_ARG(x && k && y, "%s: null pointer", who);
  MEGA_CHECK_ARG(valid_dtype(dtype), "%s: bad dtype %d", who, dtype);
  MEGA_CHECK_ARG(B >= 0 && D >= 0 && L >= 0, "%s: negative size", who);
  if (L > kMaxL)
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: L=%lld exceeds the supported %lld", who,
                     (long long)L, (long long)kMaxL);
  if (B == 0 || D == 0 || L == 0) return MEGA_OK;
  return dispatch_conv<0>(dtype, x, k, y, B, D, L, 0, omega, static_cast<hipStream_t>(stream));
}

int fftconv_bwd_impl(const char* who, const void* dy, const void* x, int dtype, const float* k,
                     const float* omega, int64_t B, int64_t D, int64_t L, void* dx, float* dk,
                     void* stream) {
  MEGA_CHECK_ARG(dy && x && k && dx && dk, "%s: null pointer", who);
  MEGA_CHECK_ARG(valid_dtype(dtype), "%s: bad dtype %d", who, dtype);
  MEGA_CHECK_ARG(B >= 0 && D >= 0 && L >= 0, "%s: negative size", who);
  if (L > kMaxL)
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: L=%lld exceeds the supported %lld", who,
                     (long long)L, (long long)kMaxL);
  if (D == 0 || L == 0) return MEGA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (B == 0) {
    const int64_t n = D * L;
    zero_fill_kernel<<<dim3(static_cast<unsigned>((n + 255) / 256)), 256, 0, s>>>(dk, n);
    MEGA_CHECK_LAUNCH();
    return MEGA_OK;
  }
  if (fftm::applicable(dtype, L, dy, x, dx) && reinterpret_cast<uintptr_t>(k) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(dk) % 16 == 0 && f16_stages_enabled())
    return fftm::launch_backward(dtype, dy, x, k, dx, dk, B, D, L, omega, s);
  int rc = dispatch_conv<0>(dtype, dy, k, dx, B, D, L, 1, omega, s);
  if (rc != MEGA_OK) return rc;
  return dispatch_conv<1>(dtype, dy, x, dk, B, D, L, 1, nullptr, s);
}
}  // namespace

extern "C" int mega_fftconv_fwd(const void* x, int dtype, const float* k, int64_t B, int64_t D,
                                int64_t L, void* y, void* stream) {
  return fftconv_fwd_impl("mega_fftconv_fwd", x, dtype, k, nullptr, B, D, L, y, stream);
}

extern "C" int mega_fftconv_bwd(const void* dy, const void* x, int dtype, const float* k,
                                int64_t B, int64_t D, int64_t L, void* dx, float* dk,
                                void* stream) {
  return fftconv_bwd_impl("mega_fftconv_bwd", dy, x, dtype, k, nullptr, B, D, L, dx, dk, stream);
}

extern "C" int mega_fftconv_residual_fwd(const void* x, int dtype, const float* k,
                                         const float* omega, int64_t B, int64_t D, int64_t L,
                                         void* y, void* stream) {
  MEGA_CHECK_ARG(omega, "mega_fftconv_residual_fwd: null omega");
  return fftconv_fwd_impl("mega_fftconv_residual_fwd", x, dtype, k, omega, B, D, L, y, stream);
}

extern "C" int mega_fftconv_residual_bwd(const void* dy, const void* x, int dtype, const float* k,
                                         const float* omega, int64_t B, int64_t D, int64_t L,
                                         void* dx, float* dk, void* stream) {
  MEGA_CHECK_ARG(omega, "mega_fftconv_residual_bwd: null omega");
  return fftconv_bwd_impl("mega_fftconv_residual_bwd", dy, x, dtype, k, omega, B, D, L, dx, dk,
                          stream);
}

// ---- forward that keeps the spectra of x and k, backward that uses them ----------
extern "C" int64_t mega_fftconv_spectrum_bytes(int dtype, int64_t B, int64_t D, int64_t L) {
  if (B <= 0 || D <= 0 || L <= 0 || !f16_stages_enabled()) return 0;
  return fftm::spectrum_bytes(dtype, B, D, L);
}

extern "C" int mega_fftconv_residual_fwd_saving(const void* x, int dtype, const float* k,
                                                const float* omega, int64_t B, int64_t D,
                                                int64_t L, void* y, void* spec_x, void* spec_k,
                                                void* stream) {
  const char* who = "mega_fftconv_residual_fwd_saving";
  MEGA_CHECK_ARG(x && k && y && spec_x && spec_k, "%s: null pointer", who);
  MEGA_CHECK_ARG(fftm::spectrum_bytes(dtype, B, D, L) > 0 && fftm::applicable(dtype, L, x, k, y) &&
                     reinterpret_cast<uintptr_t>(spec_x) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(spec_k) % 16 == 0,
                 "%s: shape, dtype or alignment outside the saved-spectrum path "
                 "(mega_fftconv_spectrum_bytes returns 0 for it)", who);
  return fftm::launch_forward_saving(dtype, x, k, y, B, D, L, omega, spec_x, spec_k,
                                     static_cast<hipStream_t>(stream));
}

extern "C" int mega_fftconv_residual_bwd_saved(const void* dy, int dtype, const void* spec_x,
                                               const void* spec_k, const float* omega, int64_t B,
                                               int64_t D, int64_t L, void* dx, float* dk,
                                               void* stream) {
  const char* who = "mega_fftconv_residual_bwd_saved";
  MEGA_CHECK_ARG(dy && spec_x && spec_k && dx && dk, "%s: null pointer", who);
  MEGA_CHECK_ARG(fftm::spectrum_bytes(dtype, B, D, L) > 0 && fftm::applicable(dtype, L, dy, dx, dk) &&
                     reinterpret_cast<uintptr_t>(spec_x) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(spec_k) % 16 == 0,
                 "%s: shape, dtype or alignment outside the saved-spectrum path", who);
  return fftm::launch_backward_saved(dtype, dy, spec_x, spec_k, dx, dk, B, D, L, omega,
                                     static_cast<hipStream_t>(stream));
}
