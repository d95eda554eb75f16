// LayerNorm / RMSNorm over the last axis with the reference's parameterisation:
// the stored weight is gamma - 1 (megalodon/modules/layer_norm.py:14-66 adds 1
// before calling apex's fused_layer_norm_cuda, which is not part of the
// reference tree).  y = (x - mean) * rstd * (weight + 1) + bias with biased
// variance and rstd = 1 / sqrt(var + eps); RMSNorm drops the mean and the bias
// and uses mean(x^2).  Rows are independent, so the kernels are streaming:
// a row (or 2-4 short rows) sits in the registers of one wavefront, x is read
// once and y written once; the backward reads x and dy once, writes dx once and
// leaves per-workgroup column sums for the parameter gradients, which a second
// small kernel reduces in a fixed order (no float atomics).
#include "common.hpp"

namespace mega {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kMaxGroups = 1024;  // workgroups of the backward = partial-sum rows


// hides a register from common-subexpression elimination: values derived from it
// afterwards are recomputed instead of being kept alive across the row reduction
__device__ __forceinline__ void opaque(uint4& q) {
  asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(q.z), "+v"(q.w));
}

struct NormParams {
  const void* x;
  const void* dy;
  const void* weight;  // gamma - 1, may be null (gamma = 1)
  const void* bias;    // may be null
  void* y;             // forward: y, backward: dx
  float* mean;         // per row (unused for RMS)
  float* rstd;         // per row
  float* part_w;       // backward: (groups, D) partial sums of dy * xhat
  float* part_b;       // backward: (groups, D) partial sums of dy
  int64_t rows;
  int D;
  float eps;
};

// ---- rows in registers: D = LPR * 8 * NCH, 64 / LPR rows per wavefront --------
template <int DT, int LPR, int NCH, bool RMS>
__global__ __launch_bounds__(kThreads) void norm_fwd_vec_kernel(NormParams p) {
  constexpr int RPW = kWave / LPR;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int lr = lane % LPR, slot = lane / LPR;
  const uint16_t* x = static_cast<const uint16_t*>(p.x);
  uint16_t* y = static_cast<uint16_t*>(p.y);
  const float inv_d = 1.f / static_cast<float>(p.D);
  // weight and bias stay packed (one register per element pair)
  // A wave has one row up to 65536 rows of them, so what counts beside its chain of loads is how many waves there are: the
  // next row is not asked for before this one has left its registers (LayerNorm at width 4096 200 of them so, two waves per
  // SIMD, now a third: 4096 rows 15.1 us, now 13.5).  Wide rows are asked for in front of the weights, narrow ones
  // behind them, in us: RMSNorm 4096 x 4096 11.3 / 11.6, 32768 x 4096 92.9 / 96.0 (99.7 with a wait for each piece of the
  // weights), 16384 x 1024 11.2 / 11.8, but 16384 x 512 6.2 / 5.8; LayerNorm 4096 x 2048 7.1 / 7.3, but 16384 x 1024 12.9 / 12.1 and, of few rows,
  // 1531 x 4096 6.7 / 6.4, 2048 7.6 / 7.4, 8192 23.0 / 23.2, 32768 93.9 / 97.3.
  constexpr bool kRowFirst = NCH >= 4 || (RMS && NCH == 2);
  const bool row_first = kRowFirst && (RMS || NCH < 8 || p.rows > 8192);
  const int64_t step = static_cast<int64_t>(gridDim.x) * kWaves * RPW;
  int64_t row = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * RPW + slot;
  uint4 piece[NCH];
  auto request = [&](int64_t at) {  // rows behind the last: the last one again, unused
    const uint16_t* src = x + (at < p.rows ? at : p.rows - 1) * p.D;
#pragma unroll
    for (int i = 0; i < NCH; ++i) piece[i] = *reinterpret_cast<const uint4*>(src + (lr + LPR * i) * 8);
  };
  if (row_first) request(row);
  uint4 gq[NCH], bq[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) gq[i] = bq[i] = make_uint4(0, 0, 0, 0);
  // (one branch for all of them: with a branch to each the loads are waited for one by one)
  if (p.weight)
#pragma unroll
    for (int i = 0; i < NCH; ++i) gq[i] = reinterpret_cast<const uint4*>(p.weight)[lr + LPR * i];
  if (!RMS && p.bias)
#pragma unroll
    for (int i = 0; i < NCH; ++i) bq[i] = reinterpret_cast<const uint4*>(p.bias)[lr + LPR * i];
  for (; row - slot < p.rows; row += step) {
    const bool live = row < p.rows;
    if (!row_first) request(row);
    float v[NCH][8];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      unpack8<DT>(piece[i], v[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += RMS ? v[i][e] * v[i][e] : v[i][e];
    }
    s = group_sum<LPR>(s) * inv_d;
    float mu = 0.f, var = s;
    if (!RMS) {
      mu = s;
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[i][e] -= mu;
          ss += v[i][e] * v[i][e];
        }
      var = group_sum<LPR>(ss) * inv_d;
    }
    const float r = rsqrtf(var + p.eps);
    if (live) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        float g[8], b[8];
        opaque(gq[i]);  // unpacked per row, not hoisted out of the row loop
        unpack8<DT>(gq[i], g);
        if (!RMS) {
          opaque(bq[i]);
          unpack8<DT>(bq[i], b);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = v[i][e] * r * (g[e] + 1.f) + (RMS ? 0.f : b[e]);
        *reinterpret_cast<uint4*>(y + row * p.D + (lr + LPR * i) * 8) = pack8<DT>(v[i]);
      }
      if (lr == 0) {
        p.rstd[row] = r;
        if (!RMS) p.mean[row] = mu;
      }
    }
    if (row_first && row - slot + step < p.rows) request(row + step);
  }
}

template <int DT, int LPR, int NCH, bool RMS>
__global__ __launch_bounds__(kThreads) void norm_bwd_vec_kernel(NormParams p) {
  constexpr int RPW = kWave / LPR;
  extern __shared__ float acc[];  // D floats (x 2 with a bias)
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int lr = lane % LPR, slot = lane / LPR;
  const uint16_t* x = static_cast<const uint16_t*>(p.x);
  const uint16_t* dy = static_cast<const uint16_t*>(p.dy);
  uint16_t* dx = static_cast<uint16_t*>(p.y);
  const float inv_d = 1.f / static_cast<float>(p.D);
  // weights stay packed; x and dy of the row stay packed too and are unpacked once
  // for the row sums and once more for dx, so that the two accumulator sets
  // (2 x D / 64 floats per lane) fit beside them
  uint4 gq[NCH];
  float aw[NCH][8], ab[RMS ? 1 : NCH][8];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    gq[i] = make_uint4(0, 0, 0, 0);
    if (p.weight)
      gq[i] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.weight) + (lr + LPR * i) * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      aw[i][e] = 0.f;
      if (!RMS) ab[i][e] = 0.f;
    }
  }
  const int64_t step = static_cast<int64_t>(gridDim.x) * kWaves * RPW;
  for (int64_t row = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * RPW + slot;
       row - slot < p.rows; row += step) {
    const bool live = row < p.rows;
    const float r = live ? p.rstd[row] : 0.f;
    const float mu = (!RMS && live) ? p.mean[row] : 0.f;
    uint4 qx[NCH], qg[NCH];
    float s1 = 0.f, s0 = 0.f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      qx[i] = make_uint4(0, 0, 0, 0);
      qg[i] = make_uint4(0, 0, 0, 0);
      if (live) {
        qx[i] = *reinterpret_cast<const uint4*>(x + row * p.D + (lr + LPR * i) * 8);
        qg[i] = *reinterpret_cast<const uint4*>(dy + row * p.D + (lr + LPR * i) * 8);
      }
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      float xh[8], gy[8], g[8];
      unpack8<DT>(qx[i], xh);
      unpack8<DT>(qg[i], gy);
      opaque(gq[i]);  // unpacked per row, not hoisted out of the row loop
      unpack8<DT>(gq[i], g);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float h = (xh[e] - mu) * r;
        aw[i][e] += gy[e] * h;
        if (!RMS) ab[i][e] += gy[e];
        const float gw = gy[e] * (g[e] + 1.f);
        s1 += gw * h;
        if (!RMS) s0 += gw;
      }
    }
    s1 = group_sum<LPR>(s1) * inv_d;
    if (!RMS) s0 = group_sum<LPR>(s0) * inv_d;
    if (live) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        opaque(qx[i]);
        opaque(qg[i]);
        opaque(gq[i]);
        float xh[8], gy[8], g[8];
        unpack8<DT>(qx[i], xh);
        unpack8<DT>(qg[i], gy);
        unpack8<DT>(gq[i], g);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          gy[e] = r * (gy[e] * (g[e] + 1.f) - (xh[e] - mu) * r * s1 - s0);
        *reinterpret_cast<uint4*>(dx + row * p.D + (lr + LPR * i) * 8) = pack8<DT>(gy);
      }
    }
  }
  if (p.part_w == nullptr) return;  // no affine parameters
  // column sums of this workgroup, added slot by slot in a fixed order
  for (int s = 0; s < kWaves * RPW; ++s) {
    if (wave * RPW + slot == s) {
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int c = (lr + LPR * i) * 8 + e;
          if (s == 0) {
            acc[c] = aw[i][e];
            if (!RMS) acc[p.D + c] = ab[i][e];
          } else {
            acc[c] += aw[i][e];
            if (!RMS) acc[p.D + c] += ab[i][e];
          }
        }
    }
    __syncthreads();
  }
  for (int c = threadIdx.x; c < p.D; c += kThreads) {
    p.part_w[static_cast<int64_t>(blockIdx.x) * p.D + c] = acc[c];
    if (!RMS && p.part_b) p.part_b[static_cast<int64_t>(blockIdx.x) * p.D + c] = acc[p.D + c];
  }
}

// D = 512 W: a workgroup of W waves takes kRowsAtOnce rows at a time, a lane the same eight columns of each.  The column sums
// stay in its registers from the first row to the last (16 instead of D / 32 of a wave that owns a row, which at D = 4096
// left one wave per SIMD) and need no reduction over the workgroup; the row sums meet in LDS, one barrier for the rows at
// once, while the next rows are on their way.  LayerNorm backward, with a wave to a row / so: 32768 x 4096 239 / 175 us,
// 4096 x 2048 38.9 / 19.2, 4096 x 1024 20.9 / 15.2; RMSNorm 165 / 161, 21.1 / 16.5, 13.8 / 11.9 (see by_columns).
constexpr int kRowsAtOnce = 4;
typedef float float4_any __attribute__((ext_vector_type(4), aligned(4)));  // (a workspace is a caller's, at any float)
template <int DT, int W, bool RMS>
__global__ __launch_bounds__(W * kWave) void norm_bwd_columns_kernel(NormParams p) {
  constexpr int R = kRowsAtOnce;
  __shared__ float2 sums[2][R][W];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int col = threadIdx.x * 8;
  const uint16_t* x = static_cast<const uint16_t*>(p.x) + col;
  const uint16_t* dy = static_cast<const uint16_t*>(p.dy) + col;
  uint16_t* dx = static_cast<uint16_t*>(p.y) + col;
  const float inv_d = 1.f / static_cast<float>(p.D);
  float g[8], aw[8], ab[8];
  uint4 gq = make_uint4(0, 0, 0, 0);
  if (p.weight) gq = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.weight) + col);
  unpack8<DT>(gq, g);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    g[e] += 1.f;
    aw[e] = ab[e] = 0.f;
  }
  uint4 qx[R], qg[R], nx[R], ng[R];
  float rs[R], mu[R], nr[R], nm[R];
  auto request = [&](int64_t row0) {  // rows behind the last: the last one again, unused
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t row = row0 + i < p.rows ? row0 + i : p.rows - 1;
      nx[i] = *reinterpret_cast<const uint4*>(x + row * p.D);
      ng[i] = *reinterpret_cast<const uint4*>(dy + row * p.D);
      nr[i] = p.rstd[row];
      nm[i] = RMS ? 0.f : p.mean[row];
    }
  };
  const int64_t step = static_cast<int64_t>(gridDim.x) * R;
  int64_t row0 = static_cast<int64_t>(blockIdx.x) * R;
  request(row0);
  for (int par = 0; row0 < p.rows; row0 += step, par ^= 1) {
#pragma unroll
    for (int i = 0; i < R; ++i) qx[i] = nx[i], qg[i] = ng[i], rs[i] = nr[i], mu[i] = nm[i];
    if (row0 + step < p.rows) request(row0 + step);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      float xh[8], gy[8], s1 = 0.f, s0 = 0.f;
      unpack8<DT>(qx[i], xh);
      unpack8<DT>(qg[i], gy);
      if (row0 + i < p.rows) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float h = (xh[e] - mu[i]) * rs[i], gw = gy[e] * g[e];
          aw[e] = fmaf(gy[e], h, aw[e]);
          if (!RMS) ab[e] += gy[e];
          s1 = fmaf(gw, h, s1);
          if (!RMS) s0 += gw;
        }
      }
      s1 = wave_sum(s1);
      if (!RMS) s0 = wave_sum(s0);
      if (lane == 0) sums[par][i][wave] = make_float2(s1, s0);
    }
    __syncthreads();  // (the other of the two sets is read until here)
#pragma unroll
    for (int i = 0; i < R; ++i) {
      float s1 = 0.f, s0 = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float2 s = sums[par][i][w];
        s1 += s.x;
        if (!RMS) s0 += s.y;
      }
      s1 *= inv_d;
      s0 *= inv_d;
      if (row0 + i < p.rows) {
        opaque(qx[i]);  // unpacked once more: kept as floats the rows would take 64 registers
        opaque(qg[i]);
        float xh[8], gy[8];
        unpack8<DT>(qx[i], xh);
        unpack8<DT>(qg[i], gy);
#pragma unroll
        for (int e = 0; e < 8; ++e) gy[e] = rs[i] * (gy[e] * g[e] - (xh[e] - mu[i]) * rs[i] * s1 - s0);
        *reinterpret_cast<uint4*>(dx + (row0 + i) * p.D) = pack8<DT>(gy);
      }
    }
  }
  if (p.part_w == nullptr) return;  // no affine parameters
  auto put = [&](float* part, const float (&a)[8]) {
    float4_any* const to = reinterpret_cast<float4_any*>(part + static_cast<int64_t>(blockIdx.x) * p.D + col);
    to[0] = float4_any{a[0], a[1], a[2], a[3]};
    to[1] = float4_any{a[4], a[5], a[6], a[7]};
  };
  put(p.part_w, aw);
  if (!RMS && p.part_b) put(p.part_b, ab);
}

// ---- any D, any element type: one wavefront per row, row re-read from cache ----
template <int DT, bool RMS>
__global__ __launch_bounds__(kThreads) void norm_fwd_any_kernel(NormParams p) {
  using T = typename Elem<DT>::type;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const T* x = static_cast<const T*>(p.x);
  const T* w = static_cast<const T*>(p.weight);
  const T* b = static_cast<const T*>(p.bias);
  T* y = static_cast<T*>(p.y);
  const float inv_d = 1.f / static_cast<float>(p.D);
  for (int64_t row = static_cast<int64_t>(blockIdx.x) * kWaves + wave; row < p.rows;
       row += static_cast<int64_t>(gridDim.x) * kWaves) {
    const T* xr = x + row * p.D;
    float mu = 0.f;
    if (!RMS) {
      float s = 0.f;
      for (int c = lane; c < p.D; c += kWave) s += Elem<DT>::load(xr + c);
      mu = wave_sum(s) * inv_d;
    }
    float ss = 0.f;
    for (int c = lane; c < p.D; c += kWave) {
      const float d = Elem<DT>::load(xr + c) - mu;
      ss += d * d;
    }
    const float r = rsqrtf(wave_sum(ss) * inv_d + p.eps);
    for (int c = lane; c < p.D; c += kWave) {
      const float gm = w ? Elem<DT>::load(w + c) + 1.f : 1.f;
      const float bs = (!RMS && b) ? Elem<DT>::load(b + c) : 0.f;
      Elem<DT>::store(y + row * p.D + c, (Elem<DT>::load(xr + c) - mu) * r * gm + bs);
    }
    if (lane == 0) {
      p.rstd[row] = r;
      if (!RMS) p.mean[row] = mu;
    }
  }
}

template <int DT, bool RMS>
__global__ __launch_bounds__(kThreads) void norm_bwd_any_kernel(NormParams p, int active) {
  using T = typename Elem<DT>::type;
  extern __shared__ float acc[];  // `active` stripes of D floats (x 2 with a bias), one per working wave
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const T* x = static_cast<const T*>(p.x);
  const T* dy = static_cast<const T*>(p.dy);
  const T* w = static_cast<const T*>(p.weight);
  T* dx = static_cast<T*>(p.y);
  const float inv_d = 1.f / static_cast<float>(p.D);
  const int nacc = RMS ? 1 : 2;
  float* mine = acc + static_cast<int64_t>(wave) * nacc * p.D;
  if (p.part_w && wave < active)
    for (int c = lane; c < nacc * p.D; c += kWave) mine[c] = 0.f;
  for (int64_t row = static_cast<int64_t>(blockIdx.x) * active + wave; wave < active && row < p.rows;
       row += static_cast<int64_t>(gridDim.x) * active) {
    const T* xr = x + row * p.D;
    const T* gr = dy + row * p.D;
    const float r = p.rstd[row], mu = RMS ? 0.f : p.mean[row];
    float s1 = 0.f, s0 = 0.f;
    for (int c = lane; c < p.D; c += kWave) {
      const float xh = (Elem<DT>::load(xr + c) - mu) * r;
      const float go = Elem<DT>::load(gr + c);
      const float gw = go * (w ? Elem<DT>::load(w + c) + 1.f : 1.f);
      s1 += gw * xh;
      s0 += gw;
      if (p.part_w) {
        mine[c] += go * xh;
        if (!RMS) mine[p.D + c] += go;
      }
    }
    s1 = wave_sum(s1) * inv_d;
    s0 = RMS ? 0.f : wave_sum(s0) * inv_d;
    for (int c = lane; c < p.D; c += kWave) {
      const float xh = (Elem<DT>::load(xr + c) - mu) * r;
      const float gw = Elem<DT>::load(gr + c) * (w ? Elem<DT>::load(w + c) + 1.f : 1.f);
      Elem<DT>::store(dx + row * p.D + c, r * (gw - xh * s1 - s0));
    }
  }
  if (p.part_w == nullptr) return;
  __syncthreads();
  for (int c = threadIdx.x; c < p.D; c += kThreads) {
    float sw = 0.f, sb = 0.f;
    for (int v = 0; v < active; ++v) {
      sw += acc[static_cast<int64_t>(v) * nacc * p.D + c];
      if (!RMS) sb += acc[static_cast<int64_t>(v) * nacc * p.D + p.D + c];
    }
    p.part_w[static_cast<int64_t>(blockIdx.x) * p.D + c] = sw;
    if (!RMS && p.part_b) p.part_b[static_cast<int64_t>(blockIdx.x) * p.D + c] = sb;
  }
}

// out[c] = sum over `groups` rows (`stride` floats apart) of part[., c], c < D, for one or two
// (part, out) pairs: 16 columns x 64 row slices per workgroup, so that the few columns of a norm
// still occupy a workgroup per 64 bytes of a row and a thread has all its loads in flight.
// (1024 rows of 4096 columns, two sums: 20 us with 64 columns x 16 slices and a launch each, 4.3 so.)
struct ColumnSums {
  const float* part[2];
  void* out[2];
};
template <int DT>
__global__ __launch_bounds__(1024) void norm_param_grad_kernel(ColumnSums t, int groups, int D, int stride) {
  __shared__ float red[16][17];
  const int cx = threadIdx.x % 16, sy = threadIdx.x / 16, wave = threadIdx.x / kWave;
  const int c = blockIdx.x * 16 + cx;
  const float* part = t.part[blockIdx.y];
  float s = 0.f;
  if (c < D) {
#pragma unroll 8
    for (int gidx = sy; gidx < groups; gidx += 64) s += part[static_cast<int64_t>(gidx) * stride + c];
  }
  s += __shfl_xor(s, 16);
  s += __shfl_xor(s, 32);
  if (threadIdx.x % kWave < 16) red[wave][cx] = s;
  __syncthreads();
  if (threadIdx.x < 16 && c < D) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) v += red[w][cx];
    Elem<DT>::store(static_cast<typename Elem<DT>::type*>(t.out[blockIdx.y]) + c, v);
  }
}
template <int DT>
int launch_param_grad(const ColumnSums& t, int groups, int D, int stride, hipStream_t s) {
  norm_param_grad_kernel<DT><<<dim3((D + 15) / 16, t.part[1] != nullptr ? 2 : 1), 1024, 0, s>>>(t, groups, D, stride);
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

// ---- column sums of 16-bit rows (a linear layer's bias gradient) -------------------
// Bound by reading the rows once.  A workgroup takes 256 columns (512 contiguous bytes of a row) of a
// slice of rows, eight rows at a time, its partial sums go out in float32 and the kernel above adds up the
// slices.  Some 2048 workgroups where the rows give every one of them a row per thread: eight waves per SIMD
// is what keeps enough loads in flight.
// The library's reduction / these two launches, rows x columns in bfloat16: 4096 x 2048 17.4 / 7.3 us (and a
// 4.7 us fill of its semaphores besides), 32768 x 1024 32 / 14, 32768 x 8192 98 / 90 (6.0 TB/s).
constexpr int kSumCols = 256, kSumRows = 8, kSumGroups = 2048;
void column_slices(int64_t rows, int64_t cols, int* slices, int64_t* per) {
  const int64_t blocks = (cols + kSumCols - 1) / kSumCols;
  int64_t n = kSumGroups / blocks;
  if (n > (rows + kSumRows - 1) / kSumRows) n = (rows + kSumRows - 1) / kSumRows;
  if (n < 1) n = 1;
  *per = (rows + n - 1) / n;
  *slices = static_cast<int>((rows + *per - 1) / *per);  // none empty
}

template <int DT>
__global__ __launch_bounds__(kSumCols) void column_part_kernel(const uint16_t* __restrict__ x, int64_t rows, int64_t per,
                                                               int cols, float* __restrict__ part) {
  __shared__ float red[kSumRows][kSumCols + 8];
  const int cx = (threadIdx.x % 32) * 8, ry = threadIdx.x / 32, c = blockIdx.x * kSumCols + cx;
  const int64_t lo = blockIdx.y * per, hi = lo + per < rows ? lo + per : rows;
  float acc[8] = {};
  if (c < cols) {
#pragma unroll 4
    for (int64_t r = lo + ry; r < hi; r += kSumRows) {
      float v[8];
      unpack8<DT>(load_once(x + r * cols + c), v);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += v[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[ry][cx + e] = acc[e];
  __syncthreads();
  const int o = blockIdx.x * kSumCols + static_cast<int>(threadIdx.x);
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < kSumRows; ++r) s += red[r][threadIdx.x];
  if (o < cols) part[static_cast<int64_t>(blockIdx.y) * cols + o] = s;
}

// ---- z -> (q, k): per-head RMSNorm, the two affine maps, rotary ----------------
// megalodon/modules/moving_average_gated_attention.py:319-330 (znorm over each
// head of z, `z.unsqueeze(2) * (gamma + 1) / sqrt(Dh) + beta`, unbind into q, k)
// followed by the rotary product of
// megalodon/modules/rotary_positional_embedding.py:53-77 on both: neighbouring
// elements (2i, 2i+1) of a head are one complex number that is multiplied by
// freqs[p][i], p = (row % L) % P the position inside the chunk.  One wavefront
// holds a row of S = 512 * NCH elements, or 512 / S rows of 64, 128 or 256 (one narrow head
// each: left to the PyTorch expressions they are some 65 small launches per training step,
// 0.5 ms of a block of 1024 channels on 2 x 2048 steps), G = Dh / 8 lanes per head; z is read once and q, k are written once.  The backward undoes the rotation with the
// conjugate factor, forms the gradients of the affine parameters as column
// sums (per-workgroup partials, reduced in a fixed order afterwards) and the
// RMSNorm gradient per head.
struct QkParams {
  const uint16_t* z;
  const uint16_t* gamma;  // (2, S) as stored: the factor is (gamma + 1) / sqrt(Dh)
  const uint16_t* beta;   // (2, S)
  const float* freqs;     // (P, Dh / 2, 2) cos, sin; null = no rotary
  const uint16_t* dq;
  const uint16_t* dk;
  uint16_t* q;  // forward: q, backward: dz
  uint16_t* k;
  float* rstd;  // (rows, S / Dh)
  float* part;  // backward: (groups, 4 S): dgamma_q | dgamma_k | dbeta_q | dbeta_k
  int64_t rows;
  int L, P, S, Dh;
  float eps, inv_sqrt_dh;
};

// Where a lane's 16-byte pieces lie: lanes per row, the row among those of the wavefront.
struct QkLane {
  int lpr, slot, col;
  __device__ __forceinline__ QkLane(int S, int lane)
      : lpr(S < 512 ? S / 8 : kWave), slot(lane / lpr), col((lane - slot * lpr) * 8) {}
  __device__ __forceinline__ int rows() const { return kWave / lpr; }
};

__device__ __forceinline__ void rotate8(float* u, const float4& f0, const float4& f1, bool conj) {
  const float c[4] = {f0.x, f0.z, f1.x, f1.z};
  const float sn[4] = {f0.y, f0.w, f1.y, f1.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float s = conj ? -sn[i] : sn[i];
    const float a = u[2 * i], b = u[2 * i + 1];
    u[2 * i] = a * c[i] - b * s;
    u[2 * i + 1] = a * s + b * c[i];
  }
}

template <int DT, int G, int NCH>
__global__ __launch_bounds__(kThreads) void qk_fwd_kernel(QkParams p) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int heads = p.S / p.Dh;
  const QkLane at(p.S, lane);
  const float inv_dh = 1.f / static_cast<float>(p.Dh);
  uint4 gq[NCH], gk[NCH], bq[NCH], bk[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = at.col + kWave * 8 * i;
    gq[i] = *reinterpret_cast<const uint4*>(p.gamma + c);
    gk[i] = *reinterpret_cast<const uint4*>(p.gamma + p.S + c);
    bq[i] = *reinterpret_cast<const uint4*>(p.beta + c);
    bk[i] = *reinterpret_cast<const uint4*>(p.beta + p.S + c);
  }
  for (int64_t first = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * at.rows(); first < p.rows;
       first += static_cast<int64_t>(gridDim.x) * kWaves * at.rows()) {
    const bool on = first + at.slot < p.rows;  // the last wavefront's spare lanes take its first row
    const int64_t row = on ? first + at.slot : first;
    const int pos = static_cast<int>(row % p.L) % p.P;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = at.col + kWave * 8 * i;
      float v[8], uq[8], uk[8], g[8], b[8];
      unpack8<DT>(*reinterpret_cast<const uint4*>(p.z + row * p.S + c), v);
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
      const float r = rsqrtf(group_sum<G>(ss) * inv_dh + p.eps);
      if (on && lane % G == 0) p.rstd[row * heads + c / p.Dh] = r;
      opaque(gq[i]); opaque(bq[i]); opaque(gk[i]); opaque(bk[i]);
      unpack8<DT>(gq[i], g);
      unpack8<DT>(bq[i], b);
#pragma unroll
      for (int e = 0; e < 8; ++e) uq[e] = v[e] * r * ((g[e] + 1.f) * p.inv_sqrt_dh) + b[e];
      unpack8<DT>(gk[i], g);
      unpack8<DT>(bk[i], b);
#pragma unroll
      for (int e = 0; e < 8; ++e) uk[e] = v[e] * r * ((g[e] + 1.f) * p.inv_sqrt_dh) + b[e];
      if (p.freqs) {
        const float4* f = reinterpret_cast<const float4*>(p.freqs + (static_cast<int64_t>(pos) * p.Dh + c % p.Dh));
        const float4 f0 = f[0], f1 = f[1];
        rotate8(uq, f0, f1, false);
        rotate8(uk, f0, f1, false);
      }
      if (on) {
        *reinterpret_cast<uint4*>(p.q + row * p.S + c) = pack8<DT>(uq);
        *reinterpret_cast<uint4*>(p.k + row * p.S + c) = pack8<DT>(uk);
      }
    }
  }
}

template <int DT, int G, int NCH>
__global__ __launch_bounds__(kThreads) void qk_bwd_kernel(QkParams p) {
  extern __shared__ float acc[];  // 4 S floats
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int heads = p.S / p.Dh;
  const QkLane at(p.S, lane);
  const float inv_dh = 1.f / static_cast<float>(p.Dh);
  uint4 gq[NCH], gk[NCH];
  float a_gq[NCH][8], a_gk[NCH][8], a_bq[NCH][8], a_bk[NCH][8];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = at.col + kWave * 8 * i;
    gq[i] = *reinterpret_cast<const uint4*>(p.gamma + c);
    gk[i] = *reinterpret_cast<const uint4*>(p.gamma + p.S + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) a_gq[i][e] = 0.f, a_gk[i][e] = 0.f, a_bq[i][e] = 0.f, a_bk[i][e] = 0.f;
  }
  for (int64_t first = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * at.rows(); first < p.rows;
       first += static_cast<int64_t>(gridDim.x) * kWaves * at.rows()) {
    const bool on = first + at.slot < p.rows;  // the last wavefront's spare lanes take its first row
    const int64_t row = on ? first + at.slot : first;
    const int pos = static_cast<int>(row % p.L) % p.P;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = at.col + kWave * 8 * i;
      float zn[8], dq[8], dk[8], g[8], dzn[8];
      unpack8<DT>(*reinterpret_cast<const uint4*>(p.z + row * p.S + c), zn);
      unpack8<DT>(*reinterpret_cast<const uint4*>(p.dq + row * p.S + c), dq);
      unpack8<DT>(*reinterpret_cast<const uint4*>(p.dk + row * p.S + c), dk);
      if (!on) {
#pragma unroll
        for (int e = 0; e < 8; ++e) dq[e] = dk[e] = 0.f;
      }
      const float r = p.rstd[row * heads + c / p.Dh];
      if (p.freqs) {
        const float4* f = reinterpret_cast<const float4*>(p.freqs + (static_cast<int64_t>(pos) * p.Dh + c % p.Dh));
        const float4 f0 = f[0], f1 = f[1];
        rotate8(dq, f0, f1, true);
        rotate8(dk, f0, f1, true);
      }
      opaque(gq[i]); opaque(gk[i]);
      unpack8<DT>(gq[i], g);
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        zn[e] *= r;
        a_gq[i][e] += dq[e] * zn[e];
        a_bq[i][e] += dq[e];
        dzn[e] = dq[e] * ((g[e] + 1.f) * p.inv_sqrt_dh);
      }
      unpack8<DT>(gk[i], g);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a_gk[i][e] += dk[e] * zn[e];
        a_bk[i][e] += dk[e];
        dzn[e] += dk[e] * ((g[e] + 1.f) * p.inv_sqrt_dh);
        s += dzn[e] * zn[e];
      }
      s = group_sum<G>(s) * inv_dh;
#pragma unroll
      for (int e = 0; e < 8; ++e) dzn[e] = r * (dzn[e] - zn[e] * s);
      if (on) *reinterpret_cast<uint4*>(p.q + row * p.S + c) = pack8<DT>(dzn);
    }
  }
  // the rows of a wavefront onto its first one's lanes
  if constexpr (NCH == 1)
    for (int off = at.lpr; off < kWave; off *= 2)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a_gq[0][e] += __shfl_xor(a_gq[0][e], off);
        a_gk[0][e] += __shfl_xor(a_gk[0][e], off);
        a_bq[0][e] += __shfl_xor(a_bq[0][e], off);
        a_bk[0][e] += __shfl_xor(a_bk[0][e], off);
      }
  // column sums of this workgroup, wave by wave in a fixed order
  for (int w = 0; w < kWaves; ++w) {
    if (wave == w && at.slot == 0) {
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int c = at.col + kWave * 8 * i + e;
          const float vg0 = a_gq[i][e] * p.inv_sqrt_dh, vg1 = a_gk[i][e] * p.inv_sqrt_dh;
          if (w == 0) {
            acc[c] = vg0; acc[p.S + c] = vg1; acc[2 * p.S + c] = a_bq[i][e]; acc[3 * p.S + c] = a_bk[i][e];
          } else {
            acc[c] += vg0; acc[p.S + c] += vg1; acc[2 * p.S + c] += a_bq[i][e]; acc[3 * p.S + c] += a_bk[i][e];
          }
        }
    }
    __syncthreads();
  }
  for (int c = threadIdx.x; c < 4 * p.S; c += kThreads)
    p.part[static_cast<int64_t>(blockIdx.x) * 4 * p.S + c] = acc[c];
}

template <int DT, bool BWD>
int launch_qk(const QkParams& p, int groups, hipStream_t s) {
  const int G = p.Dh / 8, nch = p.S < 512 ? 1 : p.S / 512;
  const size_t lds = BWD ? static_cast<size_t>(4) * p.S * sizeof(float) : 0;
  bool hit = false;
#define MEGA_QK(GG, NN)                                                      \
  if (G == GG && nch == NN) {                                                \
    hit = true;                                                              \
    if (BWD)                                                                 \
      qk_bwd_kernel<DT, GG, NN><<<groups, kThreads, lds, s>>>(p);            \
    else                                                                     \
      qk_fwd_kernel<DT, GG, NN><<<groups, kThreads, 0, s>>>(p);              \
  }
#define MEGA_QK_G(GG) MEGA_QK(GG, 1) MEGA_QK(GG, 2) MEGA_QK(GG, 4) MEGA_QK(GG, 8)
  MEGA_QK_G(8) MEGA_QK_G(16) MEGA_QK_G(32) MEGA_QK_G(64)
#undef MEGA_QK_G
#undef MEGA_QK
  if (!hit) return set_error(MEGA_ERR_UNSUPPORTED, "qk_norm_rotary: unsupported head size / width");
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

// How a row is split over a wavefront: `lpr` lanes per row, `nch` 16-byte chunks
// per lane (D = lpr * 8 * nch); lpr == 0: no register-resident variant.
struct Shape {
  int lpr, nch;
};
Shape vec_shape(int dtype, int64_t D, const NormParams& p) {
  if (dtype == MEGA_F32) return {0, 0};
  for (const void* q : {p.x, p.dy, p.weight, p.bias, static_cast<const void*>(p.y)})
    if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return {0, 0};
  for (int nch : {1, 2, 4, 8})
    if (D == 512 * nch) return {64, nch};  // one row per wavefront
  if (D == 256) return {32, 1};            // two rows per wavefront
  if (D == 128) return {16, 1};            // four
  return {0, 0};
}

int groups_for(int64_t rows, int rows_per_group) {
  const int64_t g = (rows + rows_per_group - 1) / rows_per_group;
  return static_cast<int>(g < 1 ? 1 : (g > kMaxGroups ? kMaxGroups : g));
}

// Where the backward by columns is ahead of a row to a wave: with parameter gradients, whose sums over a workgroup's waves
// it does without.  Without them it only waits at its barriers (8192 x 1024 16.2 us / 9.1, 1500 x 512 4.5 / 2.5).  Its rows
// come in passes of 2048, which cost the same half full.  By columns / a row to a wave:
//   LayerNorm, 512   100 rows 6.4 / 6.7, 2048 9.0 / 9.4, 3000 11.3 / 11.0, 4096 11.9 / 13.1, 4500 14.1 / 13.2, 8192 17.6 / 14.6
//   RMSNorm, 512     100 5.9 / 4.8, 4096 10.1 / 9.4, 16384 19.0 / 14.6
//   RMSNorm, 1024    1000 8.0 / 7.2, 2300 11.0 / 10.3, 3000 11.1 / 11.5, 4096 11.9 / 13.8, 5000 14.3 / 14.8, 5500 14.9 / 14.6, 7000 17.6 / 15.4
//   RMSNorm, 2048    1531 11.0 / 13.1, 6000 19.7 / 24.3, 12000 30.3 / 32.0, 14000 36.9 / 35.3, 32768 86.3 / 83.3
constexpr bool by_columns(bool rms, bool affine, int nch, int64_t rows) {
  if (!affine) return false;
  if (nch == 1) return !rms && (rows <= 2048 || (rows > 3200 && rows <= 4096));
  if (!rms || nch == 8) return true;
  return nch == 2 ? rows > 2800 && rows <= 5200 : rows <= 12288;
}

// Workgroups of the kernel by columns: each adds a row of partial sums that is written and read again, so more than 512 only
// where each has sixteen rows.
int column_groups(int64_t rows) {
  const int few = groups_for(rows, kRowsAtOnce), many = groups_for(rows, 16);
  return few < 512 ? few : many > 512 ? many : 512;
}

template <int DT, bool RMS, bool BWD>
int launch_vec(const NormParams& p, Shape sh, bool columns, int groups, hipStream_t s) {
  const size_t lds = BWD && p.part_w ? static_cast<size_t>(p.D) * (RMS ? 1 : 2) * sizeof(float) : 0;
#define MEGA_NORM(LPR, NCH)                                                                  \
  if (sh.lpr == LPR && sh.nch == NCH) {                                                      \
    if constexpr (BWD) {                                                                     \
      if (LPR == kWave && columns)                                                           \
        norm_bwd_columns_kernel<DT, NCH, RMS><<<groups, NCH * kWave, 0, s>>>(p);             \
      else                                                                                   \
        norm_bwd_vec_kernel<DT, LPR, NCH, RMS><<<groups, kThreads, lds, s>>>(p);             \
    } else                                                                                   \
      norm_fwd_vec_kernel<DT, LPR, NCH, RMS><<<groups, kThreads, 0, s>>>(p);                 \
  }
  MEGA_NORM(64, 1) MEGA_NORM(64, 2) MEGA_NORM(64, 4) MEGA_NORM(64, 8)
  MEGA_NORM(32, 1) MEGA_NORM(16, 1)
#undef MEGA_NORM
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

template <int DT, bool RMS>
int run_fwd(const NormParams& p, int dtype, hipStream_t s) {
  const Shape sh = vec_shape(dtype, p.D, p);
  if constexpr (DT != MEGA_F32) {
    if (sh.lpr) {
      const int rpg = kWaves * (kWave / sh.lpr);
      const int64_t g = (p.rows + rpg - 1) / rpg;
      return launch_vec<DT, RMS, false>(p, sh, false, static_cast<int>(g > 16384 ? 16384 : g), s);
    }
  }
  const int64_t g = (p.rows + kWaves - 1) / kWaves;
  norm_fwd_any_kernel<DT, RMS><<<static_cast<int>(g > 16384 ? 16384 : g), kThreads, 0, s>>>(p);
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

}  // namespace
}  // namespace mega

using namespace mega;

static int check_norm(const char* who, int dtype, int64_t rows, int64_t D) {
  MEGA_CHECK_ARG(valid_dtype(dtype), "%s: unknown dtype %d", who, dtype);
  MEGA_CHECK_ARG(rows >= 0 && D >= 1, "%s: bad sizes", who);
  MEGA_CHECK_ARG(D <= 65536, "%s: rows longer than 65536 elements are not supported", who);
  return MEGA_OK;
}

extern "C" int64_t mega_layer_norm_workspace_bytes(int64_t rows, int64_t D) {
  if (rows < 0 || D < 1) return 16;
  return 2 * static_cast<int64_t>(kMaxGroups) * D * static_cast<int64_t>(sizeof(float));
}

extern "C" int mega_layer_norm_fwd(const void* x, const void* weight, const void* bias, int dtype,
                                   int64_t rows, int64_t D, double eps, int rms, void* y,
                                   float* mean, float* rstd, void* stream) {
  int rc = check_norm("mega_layer_norm_fwd", dtype, rows, D);
  if (rc != MEGA_OK) return rc;
  if (rows == 0) return MEGA_OK;
  MEGA_CHECK_ARG(x && y && rstd && (rms || mean), "mega_layer_norm_fwd: null pointer");
  NormParams p{};
  p.x = x; p.weight = weight; p.bias = rms ? nullptr : bias; p.y = y; p.mean = mean; p.rstd = rstd;
  p.rows = rows; p.D = static_cast<int>(D); p.eps = static_cast<float>(eps);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define MEGA_DISPATCH(DT)                                   \
  return rms ? run_fwd<DT, true>(p, dtype, s) : run_fwd<DT, false>(p, dtype, s);
  if (dtype == MEGA_F32) { MEGA_DISPATCH(MEGA_F32) }
  if (dtype == MEGA_BF16) { MEGA_DISPATCH(MEGA_BF16) }
  MEGA_DISPATCH(MEGA_F16)
#undef MEGA_DISPATCH
}

template <int DT, bool RMS>
static int run_bwd(NormParams p, int dtype, void* dweight, void* dbias, float* ws, hipStream_t s) {
  const bool affine = dweight != nullptr;
  const Shape sh = vec_shape(dtype, p.D, p);
  const int rpg = sh.lpr ? kWaves * (kWave / sh.lpr) : kWaves;
  const bool columns = sh.lpr == kWave && by_columns(RMS, affine, sh.nch, p.rows);
  const int groups = columns ? column_groups(p.rows) : groups_for(p.rows, rpg);
  p.part_w = affine ? ws : nullptr;
  p.part_b = (affine && !RMS && dbias) ? ws + static_cast<int64_t>(kMaxGroups) * p.D : nullptr;
  bool done = false;
  if constexpr (DT != MEGA_F32) {
    if (sh.lpr) {
      int rc = launch_vec<DT, RMS, true>(p, sh, columns, groups, s);
      if (rc != MEGA_OK) return rc;
      done = true;
    }
  }
  if (!done) {
    // one stripe of column sums per active wave, as many waves as 64 KB of LDS hold
    const size_t stripe = static_cast<size_t>(p.D) * (RMS ? 1 : 2) * sizeof(float);
    int active = kWaves;
    while (affine && active > 1 && active * stripe > 64 * 1024) active /= 2;
    MEGA_CHECK_ARG(!affine || active * stripe <= 64 * 1024,
                   "mega_layer_norm_bwd: parameter gradients for rows of %d elements do not fit", p.D);
    norm_bwd_any_kernel<DT, RMS><<<groups, kThreads, affine ? active * stripe : 0, s>>>(p, active);
    MEGA_CHECK_LAUNCH();
  }
  if (affine) return launch_param_grad<DT>({{p.part_w, p.part_b}, {dweight, dbias}}, groups, p.D, p.D, s);
  return MEGA_OK;
}

extern "C" int mega_layer_norm_bwd(const void* dy, const void* x, const void* weight, const float* mean,
                                   const float* rstd, int dtype, int64_t rows, int64_t D, int rms,
                                   void* dx, void* dweight, void* dbias, void* workspace,
                                   void* stream) {
  int rc = check_norm("mega_layer_norm_bwd", dtype, rows, D);
  if (rc != MEGA_OK) return rc;
  MEGA_CHECK_ARG(rows >= 1, "mega_layer_norm_bwd: no rows");
  MEGA_CHECK_ARG(dy && x && dx && rstd && (rms || mean), "mega_layer_norm_bwd: null pointer");
  MEGA_CHECK_ARG(!dweight || workspace, "mega_layer_norm_bwd: parameter gradients need the workspace");
  MEGA_CHECK_ARG(!dbias || dweight, "mega_layer_norm_bwd: dbias without dweight");
  NormParams p{};
  p.x = x; p.dy = dy; p.weight = weight; p.y = dx; p.mean = const_cast<float*>(mean);
  p.rstd = const_cast<float*>(rstd); p.rows = rows; p.D = static_cast<int>(D);
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* ws = static_cast<float*>(workspace);
#define MEGA_DISPATCH(DT)                                                                       \
  return rms ? run_bwd<DT, true>(p, dtype, dweight, dbias, ws, s)                               \
             : run_bwd<DT, false>(p, dtype, dweight, dbias, ws, s);
  if (dtype == MEGA_F32) { MEGA_DISPATCH(MEGA_F32) }
  if (dtype == MEGA_BF16) { MEGA_DISPATCH(MEGA_BF16) }
  MEGA_DISPATCH(MEGA_F16)
#undef MEGA_DISPATCH
}

// ---- z -> (q, k) -------------------------------------------------------------------
static int check_qk(const char* who, int dtype, int64_t rows, int64_t L, int64_t P, int64_t S, int64_t Dh,
                    const void* freqs) {
  if (dtype != MEGA_BF16 && dtype != MEGA_F16)
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: only bfloat16 / float16 tensors are supported", who);
  MEGA_CHECK_ARG(rows >= 0 && (rows == 0 || L >= 1) && S >= 1 && Dh >= 1, "%s: bad sizes", who);
  MEGA_CHECK_ARG(!freqs || P >= 1, "%s: rotary factors without positions", who);
  if (!(Dh == 64 || Dh == 128 || Dh == 256 || Dh == 512) || S % Dh != 0 ||
      !(S == 64 || S == 128 || S == 256 || S == 512 || S == 1024 || S == 2048 || S == 4096))
    return set_error(MEGA_ERR_UNSUPPORTED,
                     "%s: needs a head size of 64, 128, 256 or 512 and a width of 64 to 4096, a power of two "
                     "(got %lld, %lld)", who, (long long)Dh, (long long)S);
  return MEGA_OK;
}

extern "C" int64_t mega_qk_norm_rotary_workspace_bytes(int64_t S) {
  return S < 1 ? 16 : static_cast<int64_t>(kMaxGroups) * 4 * S * static_cast<int64_t>(sizeof(float));
}

extern "C" int mega_qk_norm_rotary_fwd(const void* z, const void* gamma, const void* beta,
                                       const float* freqs, int dtype, int64_t rows, int64_t L, int64_t P,
                                       int64_t S, int64_t Dh, double eps, void* q, void* k, float* rstd,
                                       void* stream) {
  int rc = check_qk("mega_qk_norm_rotary_fwd", dtype, rows, L, P, S, Dh, freqs);
  if (rc != MEGA_OK) return rc;
  if (rows == 0) return MEGA_OK;
  MEGA_CHECK_ARG(z && gamma && beta && q && k && rstd, "mega_qk_norm_rotary_fwd: null pointer");
  for (const void* ptr : {z, gamma, beta, static_cast<const void*>(freqs), static_cast<const void*>(q),
                          static_cast<const void*>(k)})
    MEGA_CHECK_ARG(reinterpret_cast<uintptr_t>(ptr) % 16 == 0, "mega_qk_norm_rotary_fwd: buffers must be 16-byte aligned");
  QkParams p{};
  p.z = static_cast<const uint16_t*>(z); p.gamma = static_cast<const uint16_t*>(gamma);
  p.beta = static_cast<const uint16_t*>(beta); p.freqs = freqs;
  p.q = static_cast<uint16_t*>(q); p.k = static_cast<uint16_t*>(k); p.rstd = rstd;
  p.rows = rows; p.L = (int)L; p.P = freqs ? (int)P : 1; p.S = (int)S; p.Dh = (int)Dh;
  p.eps = static_cast<float>(eps); p.inv_sqrt_dh = static_cast<float>(1.0 / sqrt(static_cast<double>(Dh)));
  const int rpg = kWaves * static_cast<int>(S < 512 ? 512 / S : 1);
  const int64_t g = (rows + rpg - 1) / rpg;
  const int groups = static_cast<int>(g > 16384 ? 16384 : g);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == MEGA_BF16 ? launch_qk<MEGA_BF16, false>(p, groups, s) : launch_qk<MEGA_F16, false>(p, groups, s);
}

extern "C" int mega_qk_norm_rotary_bwd(const void* dq, const void* dk, const void* z, const void* gamma,
                                       const float* rstd, const float* freqs, int dtype, int64_t rows,
                                       int64_t L, int64_t P, int64_t S, int64_t Dh, void* dz, void* dgamma,
                                       void* dbeta, void* workspace, void* stream) {
  int rc = check_qk("mega_qk_norm_rotary_bwd", dtype, rows, L, P, S, Dh, freqs);
  if (rc != MEGA_OK) return rc;
  MEGA_CHECK_ARG(rows >= 1, "mega_qk_norm_rotary_bwd: no rows");
  MEGA_CHECK_ARG(dq && dk && z && gamma && rstd && dz && dgamma && dbeta && workspace,
                 "mega_qk_norm_rotary_bwd: null pointer");
  for (const void* ptr : {dq, dk, z, gamma, static_cast<const void*>(freqs), static_cast<const void*>(dz)})
    MEGA_CHECK_ARG(reinterpret_cast<uintptr_t>(ptr) % 16 == 0, "mega_qk_norm_rotary_bwd: buffers must be 16-byte aligned");
  QkParams p{};
  p.z = static_cast<const uint16_t*>(z); p.gamma = static_cast<const uint16_t*>(gamma); p.freqs = freqs;
  p.dq = static_cast<const uint16_t*>(dq); p.dk = static_cast<const uint16_t*>(dk);
  p.q = static_cast<uint16_t*>(dz); p.rstd = const_cast<float*>(rstd); p.part = static_cast<float*>(workspace);
  p.rows = rows; p.L = (int)L; p.P = freqs ? (int)P : 1; p.S = (int)S; p.Dh = (int)Dh;
  p.inv_sqrt_dh = static_cast<float>(1.0 / sqrt(static_cast<double>(Dh)));
  const int groups = groups_for(rows, kWaves * static_cast<int>(S < 512 ? 512 / S : 1));
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = dtype == MEGA_BF16 ? launch_qk<MEGA_BF16, true>(p, groups, s) : launch_qk<MEGA_F16, true>(p, groups, s);
  if (rc != MEGA_OK) return rc;
  const int cols = 2 * static_cast<int>(S);
  const ColumnSums sums{{p.part, p.part + cols}, {dgamma, dbeta}};
  return dtype == MEGA_BF16 ? launch_param_grad<MEGA_BF16>(sums, groups, cols, 2 * cols, s)
                            : launch_param_grad<MEGA_F16>(sums, groups, cols, 2 * cols, s);
}

extern "C" int64_t mega_column_sums_workspace_bytes(int64_t rows, int64_t cols) {
  if (rows <= 0 || cols <= 0) return 0;
  int slices;
  int64_t per;
  column_slices(rows, cols, &slices, &per);
  return static_cast<int64_t>(sizeof(float)) * slices * cols;
}

extern "C" int mega_column_sums(const void* x, int dtype, int64_t rows, int64_t cols, void* out, void* workspace, void* stream) {
  const char* who = "mega_column_sums";
  MEGA_CHECK_ARG(x && out && workspace, "%s: null pointer", who);
  MEGA_CHECK_ARG(rows >= 1 && cols >= 1, "%s: sizes must be at least 1", who);
  if ((dtype != MEGA_BF16 && dtype != MEGA_F16) || cols % 8 != 0 || cols > (1 << 24) || reinterpret_cast<uintptr_t>(x) % 16 != 0)
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: takes 16-bit rows on 16-byte boundaries", who);
  int slices;
  int64_t per;
  column_slices(rows, cols, &slices, &per);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int D = static_cast<int>(cols);
  float* part = static_cast<float*>(workspace);
  const dim3 grid((D + kSumCols - 1) / kSumCols, slices);
  const uint16_t* xs = static_cast<const uint16_t*>(x);
  const ColumnSums sums{{part, nullptr}, {out, nullptr}};
  if (dtype == MEGA_BF16) column_part_kernel<MEGA_BF16><<<grid, kSumCols, 0, s>>>(xs, rows, per, D, part);
  else column_part_kernel<MEGA_F16><<<grid, kSumCols, 0, s>>>(xs, rows, per, D, part);
  MEGA_CHECK_LAUNCH();
  return dtype == MEGA_BF16 ? launch_param_grad<MEGA_BF16>(sums, slices, D, D, s) : launch_param_grad<MEGA_F16>(sums, slices, D, D, s);
}
