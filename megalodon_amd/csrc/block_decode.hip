// One new token per sequence through a whole block, for generation from a cache
// (the cache branch of megalodon/modules/moving_average_gated_attention.py:283-348
// followed by normalized_feedforward_network.py:74-90, at sequence length one).
//
// The step is bound by reading the block's weights once and moving the cached keys and
// values once: at width 4096 the weights are 514 MB, and operator by operator a
// step was 59 launches, 0.84 ms for one sequence and 4.1 ms for sixteen (1531 and
// 3000 cached tokens).  Here it is seven launches, and one for each norm that does not come on the products' way: two there, 0.114 and
// 0.43 ms.  They are cut where a whole row is needed by everybody:
//   1. step_kernel    TimestepNorm step, EMA state step
//   2. products       z, r, h1 of the RMSNorm; v = silu(...) straight into the new cache
//   3. attend_kernel  q, k (norm, affine maps, rotary), one softmax part per split; the old keys and values
//                     pass into the new cache as they are read, the new key joins them
//   4. combine_kernel the parts put together, gate silu(r)
//   5. products       wh2 + h1 + residual
//   6. products       fc1, fc3 of the LayerNorm; silu(a) b
//   7. products       fc2 + residual
// The products are rows_kernel's for few sequences, else tiles_kernel's (few_rows).  rows_kernel can normalise on the way, which it does
// for the RMSNorm but with one sequence of more than 3072 features, for the LayerNorm up to 2048; rows_norm_kernel has the others'.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace mega {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxTokens = 32;

template <int DT>
__device__ __forceinline__ floatx4 mma16(u32x4 a, u32x4 b, floatx4 c) {
  if constexpr (DT == MEGA_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <int DT>
__device__ __forceinline__ float round_to(float v) {
  typename Elem<DT>::type t;
  Elem<DT>::store(&t, v);
  return Elem<DT>::load(&t);
}
__device__ __forceinline__ float silu(float v) { return v / (1.f + __expf(-v)); }

// ---- 1: TimestepNorm and EMA, one step -----------------------------------------
// A workgroup owns 32 channels of one sequence: 8 threads per channel, two modes each, so
// the state (16 complex numbers per channel, the kernel's only sizeable traffic) moves in
// 16-byte pieces.  Every wave works out the moments of the group its channels lie in by
// itself: reading at most a few hundred values again costs less than a hand-over.
constexpr int kStepChannels = 32;
constexpr int kModes = 16;

struct StepParams {
  const uint16_t *x, *prev_mean, *prev_var, *weight, *bias, *omega;
  const int64_t* prev_count;
  const float *p, *q, *gamma;
  const float4* h_in;
  uint16_t *tsn, *cema, *mean, *var;
  int64_t* count;
  float4* h_out;
  int D, G, Dg;
  float eps;
};

template <int DT>
__global__ __launch_bounds__(256) void step_kernel(const StepParams a) {
  using E = Elem<DT>;
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int d0 = blockIdx.x * kStepChannels, g = d0 / a.Dg;
  const int d = d0 + (tid >> 3), m2 = tid & 7;  // modes 2 m2, 2 m2 + 1
  const int64_t hidx = (static_cast<int64_t>(b) * a.D + d) * (kModes / 2) + m2;
  const int cidx = d * (kModes / 2) + m2;
  const float4 h = a.h_in[hidx];
  const float4 q = reinterpret_cast<const float4*>(a.q)[cidx], gm = reinterpret_cast<const float4*>(a.gamma)[cidx];
  const float2 p = reinterpret_cast<const float2*>(a.p)[cidx];
  // moments of the group at this step
  const uint16_t* xg = a.x + static_cast<int64_t>(b) * a.D + g * a.Dg;
  float s = 0.f;
  for (int i = lane; i < a.Dg; i += 64) s += E::load(xg + i);
  const float inv = 1.f / static_cast<float>(a.Dg);
  const float gu = wave_sum(s) * inv;
  s = 0.f;
  for (int i = lane; i < a.Dg; i += 64) {
    const float t = E::load(xg + i) - gu;
    s += t * t;
  }
  const float gv = wave_sum(s) * inv;
  // merged with the running statistics (utils.h:154-164)
  const int64_t c0 = a.prev_count[b];
  const float n = static_cast<float>(c0 + 1), c1 = static_cast<float>(c0) / n, c2 = 1.f / n;
  const float u0 = E::load(a.prev_mean + b * a.G + g), v0 = E::load(a.prev_var + b * a.G + g);
  const float delta = gu - u0;
  const float u = c1 * u0 + c2 * gu, v = c1 * v0 + c2 * gv + (c1 * delta) * (c2 * delta);
  const float r = 1.f / sqrtf(v + a.eps);
  if (tid == 0 && d0 % a.Dg == 0) {
    E::store(a.mean + b * a.G + g, u);
    E::store(a.var + b * a.G + g, v);
    if (g == 0) a.count[b] = c0 + 1;
  }
  const float xn = round_to<DT>((E::load(a.x + static_cast<int64_t>(b) * a.D + d) - u) * r *
                                    (E::load(a.weight + d) + 1.f) + E::load(a.bias + d));
  // h <- q h + p x, y = Re sum gamma h + omega x
  float4 o;
  o.x = q.x * h.x - q.y * h.y + p.x * xn;
  o.y = q.x * h.y + q.y * h.x;
  o.z = q.z * h.z - q.w * h.w + p.y * xn;
  o.w = q.z * h.w + q.w * h.z;
  a.h_out[hidx] = o;
  const float y = group_sum<8>(gm.x * o.x - gm.y * o.y + gm.z * o.z - gm.w * o.w);
  const float out = round_to<DT>(y + E::load(a.omega + d) * xn);
  if (m2 == 0) {
    E::store(a.tsn + static_cast<int64_t>(b) * a.D + d, xn);
    E::store(a.cema + static_cast<int64_t>(b) * a.D + d, out);
  }
}

// ---- 2, 5, 6, 7: products of a weight matrix with at most 32 rows --------------
// out[m][n] = sum_k x[m][k] W[n][k].  What counts is that the weights, each read once, stream in at the memory's rate.
enum { kNormNone = 0, kNormRms = 1, kNormLayer = 2 };
constexpr int kMaxSegs = 4;

struct Segment {       // rows of one weight matrix
  const uint16_t* W;   // (rows, K)
  const uint16_t* W2;  // pair mode: second matrix of the same shape
  const uint16_t* bias;
  const uint16_t* x;   // (tokens, K)
  uint16_t* out;
  int64_t out_stride;  // elements between tokens
  int blocks;          // workgroups of this segment
  int norm;
  int act;             // silu on the result
};
struct ProductParams {
  Segment seg[kMaxSegs];
  int segs, K, tokens;
  const uint16_t *norm_weight, *norm_bias;  // stored weight = gamma - 1; may be null
  float eps;
  const uint16_t *add1, *add2;  // (tokens, rows), added to the result
};

// Rows normalised as the layer would, for the products that take them as they are: a workgroup per row, 16 values a thread
// (bound by its launch: 2.8-4.7 us for 9-28 rows of 1024-4096 values).
constexpr int kNormThreads = 512;
template <int DT, int NORM>
__global__ __launch_bounds__(kNormThreads) void rows_norm_kernel(const uint16_t* x, const uint16_t* weight, const uint16_t* bias,
                                                                 uint16_t* out, int K, float eps) {
  constexpr int NW = kNormThreads / kWave;
  __shared__ float sums[NW], squares[NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * K;
  float v[2][8], g[2][8], b[2][8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 8 * (tid + i * kNormThreads);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = g[i][e] = b[i][e] = 0.f;
    if (k < K) {
      unpack8<DT>(*reinterpret_cast<const uint4*>(x + row + k), v[i]);
      if (weight) unpack8<DT>(*reinterpret_cast<const uint4*>(weight + k), g[i]);
      if (NORM == kNormLayer && bias) unpack8<DT>(*reinterpret_cast<const uint4*>(bias + k), b[i]);
    }
  }
  const float inv = 1.f / static_cast<float>(K);
  float mean = 0.f, s = 0.f;
  if (NORM == kNormLayer) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[i][e];
    s = wave_sum(s);
    if (lane == 0) sums[wave] = s;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) mean += sums[w];
    mean *= inv;
  }
  s = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (8 * (tid + i * kNormThreads) < K)
#pragma unroll
      for (int e = 0; e < 8; ++e) s += (v[i][e] - mean) * (v[i][e] - mean);
  s = wave_sum(s);
  if (lane == 0) squares[wave] = s;
  __syncthreads();
  s = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) s += squares[w];
  const float rstd = rsqrtf(s * inv + eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 8 * (tid + i * kNormThreads);
    if (k >= K) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = fmaf((v[i][e] - mean) * rstd, g[i][e] + 1.f, b[i][e]);
    *reinterpret_cast<uint4*>(out + row + k) = pack8<DT>(v[i]);
  }
}

// ---- 2, 5, 6, 7 for few tokens: a workgroup per few weight rows ------------------
// out[m][n] = sum_k x[m][k] W[n][k] again, for at most 4 TT tokens.  A wave's load is four rows by 128 values (256
// contiguous bytes of each), the operand of two 4x4x4 products in sixteen blocks: lane l holds row l % 4, values
// 8 (l / 4) .. + 7, and x in the same arrangement, token l % 4.  The eight waves of a workgroup share its G groups of four rows along k,
// 128 values each in turn, and ask for four pieces at once.
// What the layout is for: 256 bytes of a row in one request with the non-temporal hint, and many small workgroups, which the
// hardware hands out as others end.  Reading alone, 176 MB in four rows a workgroup take 26.5 us (6.6 TB/s; without the hint
// 28.5), in sixteen rows by 64 bytes 33, and by one workgroup per compute unit with an equal share each 52.  With that and x
// through the caches the products of one row take 14.5 us for 67 / 90 MB (in sixteen rows by 64 bytes 18.7).  A norm on the way costs vector
// work per workgroup, so those take 16 rows (while both came so at width 4096, 176 / 180 MB: 32.3 and 36.5 us; in 8 rows 36.4 and 40.5, in sixteen
// by 64 bytes 41.5 and 45).  Their weights come in two pieces at a time, one with more than one token tile: all four would leave one workgroup per unit
// (41.6 us) or spill (84).
template <int DT>
__device__ __forceinline__ floatx4 mma4(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, floatx4 c) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  if constexpr (DT == MEGA_BF16)
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, u32x2{a0, a1}), __builtin_bit_cast(s16x4, u32x2{b0, b1}), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, u32x2{a0, a1}), __builtin_bit_cast(f16x4, u32x2{b0, b1}), c, 0, 0, 0);
}
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// Row q of 16 lanes of the result holds a[q] summed over the four rows of lanes.
__device__ __forceinline__ float rows_sum(floatx4 a) {
  auto half = [](float x, float y) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
  };
  const float even = half(a[0], a[2]), odd = half(a[1], a[3]);
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(even), __float_as_uint(odd), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// Sum over the lanes of one token (l % 4), in all of them.
__device__ __forceinline__ float token_sum(float v) {
  v = dpp_add<0x124>(v);  // row_ror:4
  v = dpp_add<0x128>(v);  // row_ror:8
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
__device__ __forceinline__ u32x4 load_weights(const uint16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

constexpr int kRowsWaves = 8, kRowsPieces = 4;
// Longest row that is normalised on the way with `tt` token tiles: one round of pieces.  Only the RMSNorm of one tile goes up to four a
// wave; the others end at two (see few_rows), and rounds of three and four that nothing reaches took their kernels from 78, 82 and 90 registers
// to 119, 116 and 128, with ten more in scratch (eight tokens of one sequence of two heads of 1024 features 415 -> 410 us, of four 518 -> 513,
// of one head +- 0).
constexpr int norm_row(int norm, int tt) { return kRowsWaves * 128 * (norm == kNormRms && tt == 1 ? kRowsPieces : 2); }

template <int DT, int TT, int G, bool PAIR, int NORM>
__global__ __launch_bounds__(kRowsWaves * kWave, 4) void rows_kernel(const ProductParams a) {
  using E = Elem<DT>;
  constexpr int NW = kRowsWaves, U = kRowsPieces;
  constexpr int kRed = TT * G * 16;
  __shared__ float red[NW][kRed];
  __shared__ float2 moment[NW][4 * TT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int blk = blockIdx.x, si = 0;
  while (blk >= a.seg[si].blocks) blk -= a.seg[si++].blocks;
  const Segment& sg = a.seg[si];
  const int K = a.K, chunks = (K + 127) / 128;
  const int per = (chunks - wave + NW - 1) / NW;  // pieces of this wave: wave, wave + NW, ...
  const int l_row = lane & 3, l_k = (lane >> 2) * 8;
  const int row0 = blk * (PAIR ? 2 * G : 4 * G);

  floatx4 acc[G][TT];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[g][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uint16_t* wp[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
    wp[g] = (PAIR && (g & 1) ? sg.W2 : sg.W) + static_cast<int64_t>(row0 + 4 * (PAIR ? g >> 1 : g) + l_row) * K;
  const uint16_t* xp[TT];
#pragma unroll
  for (int j = 0; j < TT; ++j) xp[j] = sg.x + static_cast<int64_t>(4 * j + l_row < a.tokens ? 4 * j + l_row : 0) * K;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  // value of this lane's piece c (behind the row's end: its last one, which is not used)
  auto at = [&](int c) {
    const int k = 128 * (wave + NW * c) + l_k;
    return k < K ? k : K - 8;
  };
  auto inside = [&](int c) { return 128 * (wave + NW * c) + l_k < K; };

  // n pieces from c0 on
  auto round = [&](int c0, auto count) {
    constexpr int n = decltype(count)::value;
    constexpr int kHeld = NORM == kNormNone ? n : n < 2 || TT > 1 ? 1 : 2;  // pieces of weights in registers
    u32x4 x[n][TT], w[kHeld][G];
    u32x4 gw[NORM != kNormNone ? n : 1], gb[NORM == kNormLayer ? n : 1];
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const int k = at(c0 + i);
#pragma unroll
      for (int j = 0; j < TT; ++j) x[i][j] = *reinterpret_cast<const u32x4*>(xp[j] + k);
    }
    if (NORM != kNormNone) {
#pragma unroll
      for (int i = 0; i < n; ++i) {
        const int k = at(c0 + i);
        gw[i] = a.norm_weight ? *reinterpret_cast<const u32x4*>(a.norm_weight + k) : zero;
        if (NORM == kNormLayer) gb[i] = a.norm_bias ? *reinterpret_cast<const u32x4*>(a.norm_bias + k) : zero;
      }
    }
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
      const int k = at(c0 + i);
#pragma unroll
      for (int g = 0; g < G; ++g) w[i][g] = load_weights(wp[g] + k);
    }
    if (NORM != kNormNone && sg.norm != kNormNone) {
      // a row's moments: of a wave's values in two passes, of the waves' together
      float mean[TT], rstd[TT];
#pragma unroll
      for (int j = 0; j < TT; ++j) {
        float s = 0.f, q = 0.f, mine = 0.f, v[8];
        if (NORM == kNormLayer) {
          int full = 0;
#pragma unroll
          for (int i = 0; i < n; ++i) {
            full += inside(c0 + i) ? 8 : 0;
            unpack8<DT>(__builtin_bit_cast(uint4, x[i][j]), v);
            float t = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) t += v[e];
            s += inside(c0 + i) ? t : 0.f;
          }
          mine = token_sum(s) / token_sum(static_cast<float>(full));
        }
#pragma unroll
        for (int i = 0; i < n; ++i) {
          unpack8<DT>(__builtin_bit_cast(uint4, x[i][j]), v);
          float t = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float d = NORM == kNormLayer ? v[e] - mine : v[e];
            t += d * d;
          }
          q += inside(c0 + i) ? t : 0.f;
        }
        q = token_sum(q);
        if (lane < 4) moment[wave][4 * j + lane] = make_float2(mine, q);
      }
      lds_barrier();
      const float inv = 1.f / static_cast<float>(K);
#pragma unroll
      for (int j = 0; j < TT; ++j) {
        float mu = 0.f, q = 0.f;
        auto count = [&](int w) {  // values of wave w
          const int last = chunks - 1, all = (chunks - w + NW - 1) / NW * 128;
          return static_cast<float>(last % NW == w ? all - (128 * chunks - K) : all);
        };
        if (NORM == kNormLayer) {
#pragma unroll
          for (int w = 0; w < NW; ++w) mu += w < chunks ? count(w) * moment[w][4 * j + l_row].x : 0.f;
          mu *= inv;
        }
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          if (w >= chunks) continue;
          const float2 m = moment[w][4 * j + l_row];
          q += m.y;
          if (NORM == kNormLayer) q += count(w) * (m.x - mu) * (m.x - mu);
        }
        mean[j] = mu;
        rstd[j] = rsqrtf(q * inv + a.eps);
      }
#pragma unroll
      for (int i = 0; i < n; ++i) {
        float g[8], b[8], v[8];
        unpack8<DT>(__builtin_bit_cast(uint4, gw[i]), g);
        if (NORM == kNormLayer) unpack8<DT>(__builtin_bit_cast(uint4, gb[i]), b);
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          unpack8<DT>(__builtin_bit_cast(uint4, x[i][j]), v);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float scale = fmaf(g[e], rstd[j], rstd[j]);
            v[e] = NORM == kNormLayer ? fmaf(v[e] - mean[j], scale, b[e]) : v[e] * scale;
          }
          x[i][j] = __builtin_bit_cast(u32x4, pack8<DT>(v));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const int h = i % kHeld;
      if (128 * (wave + NW * (c0 + i)) + 128 > K) {  // lanes behind the row's end
        const bool in = inside(c0 + i);
#pragma unroll
        for (int j = 0; j < TT; ++j) x[i][j] = in ? x[i][j] : zero;
#pragma unroll
        for (int g = 0; g < G; ++g) w[h][g] = in ? w[h][g] : zero;
      }
#pragma unroll
      for (int j = 0; j < TT; ++j) {
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g][j] = mma4<DT>(w[h][g][0], w[h][g][1], x[i][j][0], x[i][j][1], acc[g][j]);
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g][j] = mma4<DT>(w[h][g][2], w[h][g][3], x[i][j][2], x[i][j][3], acc[g][j]);
      }
      if (i + kHeld < n) {
        const int k = at(c0 + i + kHeld);
#pragma unroll
        for (int g = 0; g < G; ++g) w[h][g] = load_weights(wp[g] + k);
      }
    }
  };
  if (NORM == kNormNone) {
    int c = 0;
    for (; c + U <= per; c += U) round(c, std::integral_constant<int, U>());
    if (per - c == 3) round(c, std::integral_constant<int, 3>());
    else if (per - c == 2) round(c, std::integral_constant<int, 2>());
    else if (per - c == 1) round(c, std::integral_constant<int, 1>());
  } else {  // (at most norm_row values)
    if constexpr (norm_row(NORM, TT) > 2 * NW * 128) {
      if (per == 4) round(0, std::integral_constant<int, 4>());
      else if (per == 3) round(0, std::integral_constant<int, 3>());
    }
    if (per == 2) round(0, std::integral_constant<int, 2>());
    else if (per == 1) round(0, std::integral_constant<int, 1>());
    else if (per == 0 && sg.norm != kNormNone) lds_barrier();  // (a row of fewer pieces than waves)
  }

#pragma unroll
  for (int j = 0; j < TT; ++j)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float v = rows_sum(acc[g][j]);
      v = dpp_add<0x124>(v);
      v = dpp_add<0x128>(v);
      if ((lane & 12) == 0) red[wave][(j * G + g) * 16 + (lane >> 4) * 4 + l_row] = v;
    }
  lds_barrier();
  // 16 results of each (token tile, row group): row (o / 4) % 4, token o % 4
  for (int o = tid; o < (PAIR ? kRed / 2 : kRed); o += NW * kWave) {
    const int q = o >> 4, e = o & 15, j = q / (PAIR ? G / 2 : G), g = q % (PAIR ? G / 2 : G);
    const int m = 4 * j + (e & 3), row = row0 + 4 * g + (e >> 2);
    const int src = (j * G + (PAIR ? 2 * g : g)) * 16 + e;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[w][src];
    if (m >= a.tokens) continue;
    if (PAIR) {
      float c = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) c += red[w][src + 16];
      v = silu(round_to<DT>(v)) * round_to<DT>(c);
    } else {
      if (sg.bias) v += E::load(sg.bias + row);
      if (sg.act) v = silu(round_to<DT>(v));
    }
    const int64_t to = static_cast<int64_t>(m) * sg.out_stride + row;
    if (a.add1) v += E::load(a.add1 + to);
    if (a.add2) v += E::load(a.add2 + to);
    E::store(sg.out + to, v);
  }
}

// ---- 2, 5, 6, 7 for more tokens: strips of 16 weight rows ----------------------
// A wave asks for four rows by 128 values (256 contiguous bytes of each, with the non-temporal hint) at a time, as
// rows_kernel does, but turns four such pieces, 16 rows by 128 values, through LDS of its own into the operands of
// 16x16x32 products with 16 MT tokens: four accumulators a tile, where the 4x4x4 products of rows_kernel would take sixteen
// (with 16 tokens 64 registers for 16 rows, 41 / 42 us for 176 / 180 MB).  A strip's registers take its next piece while
// the products run, and x's its next one behind them: a second set for x and a piece behind the last one asked for again cost 1 to 8 %
// (eight tokens of 16 sequences of four, two, one heads 1151, 575, 375 -> 1113, 567, 365 us; of 32, 24, 24 1528, 700, 449 -> 1490, 679, 416),
// two pieces of everything on their way +- 0.  x comes through the caches and holds up the weights (loads come back in order), so it comes
// normalised and serves two strips (one: 1204 -> 1249 us for the step of four heads on 8 tokens of 16 sequences; four 1293).
// In sixteen rows by 64 bytes straight into the operands, as this was before, that step took 1447 us, 16 sequences of two heads
// 620 (577), of one 396 (374), 32 of four 1977 (1567); eight of four by rows_kernel 1259 (1093), five 1175 (1058).
// Waves: few to a workgroup, so that there is little to add up (that step with 8 / 4 / 2 / 1 waves 1332 / 1256 / 1204 / 1199, 32
// sequences 1781 / 1654 / 1567 / 1804, 16 of two heads 637 / 597 / 577 / 633), but four where fewer than 256 workgroups come
// about (16 of one head 384 / 374 / 387 / 427).  One-strip products of 64 to 256 workgroups: eight (sixteen 1368 for 1332).
// PAIR: the two strips are the same rows of two matrices and silu(a) b is stored; otherwise RT consecutive strips of one.
constexpr int kTileNarrow = 8, kTileFull = 256;
template <int DT, int MT, int RT, bool PAIR, int NW>
__global__ __launch_bounds__(NW * kWave, MT == 1 ? 4 : 3) void tiles_kernel(const ProductParams a) {
  using E = Elem<DT>;
  constexpr int T = NW * kWave, kPitch = 128 + 8;
  constexpr int kStage = NW * 16 * kPitch * 2, kRedBytes = NW * RT * MT * 1024;
  __shared__ __align__(16) unsigned char raw[kStage > kRedBytes ? kStage : kRedBytes];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int blk = blockIdx.x, si = 0;
  while (blk >= a.seg[si].blocks) blk -= a.seg[si++].blocks;
  const Segment& sg = a.seg[si];
  const int K = a.K, chunks = (K + 127) / 128;
  const int per = (chunks - wave + NW - 1) / NW;
  const int row0 = blk * (PAIR ? 16 : 16 * RT);
  const int lq = lane >> 4, lc = (lane & 15) * 8;   // memory side: row of four, values of the piece
  const int r = lane & 15, kg = lane >> 4;          // operand side: row (token), group of eight values
  uint16_t* const stage = reinterpret_cast<uint16_t*>(raw) + wave * 16 * kPitch;
  uint16_t* const put = stage + lq * kPitch + lc;
  const uint16_t* const get = stage + r * kPitch + 8 * kg;

  const uint16_t* wp[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
    wp[t] = (PAIR && t == 1 ? sg.W2 : sg.W) + static_cast<int64_t>(row0 + (PAIR ? 0 : 16 * t) + lq) * K;
  const uint16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = 16 * t + r;
    xp[t] = sg.x + static_cast<int64_t>(m < a.tokens ? m : 0) * K;
  }
  floatx4 acc[RT][MT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = floatx4{0.f, 0.f, 0.f, 0.f};
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 w[RT][4], x[MT][4];
  auto load_w = [&](int c, int t) {
    const int k = 128 * (wave + NW * c) + lc;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[t][i] = load_weights(wp[t] + static_cast<int64_t>(4 * i) * K + (k < K ? k : K - 8));
  };
  auto load_x = [&](int c) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = 128 * (wave + NW * c) + 32 * s + 8 * kg;
#pragma unroll
      for (int m = 0; m < MT; ++m) x[m][s] = *reinterpret_cast<const u32x4*>(xp[m] + (k < K ? k : K - 8));
    }
  };
  // piece c; its registers take the next one as they are read
  auto piece = [&](int c, bool more) {
    const int k0 = 128 * (wave + NW * c);
    const bool cut = k0 + 128 > K;  // lanes behind the row's end
    if (cut)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) x[m][s] = k0 + 32 * s + 8 * kg >= K ? zero : x[m][s];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(put + 4 * i * kPitch) = cut && k0 + lc >= K ? zero : w[t][i];
      if (more) load_w(c + 1, t);
      asm volatile("" ::: "memory");  // (a wave's LDS accesses are served in order)
      u32x4 f[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) f[s] = *reinterpret_cast<const u32x4*>(get + 32 * s);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = mma16<DT>(f[s], x[m][s], acc[t][m]);
      asm volatile("" ::: "memory");
    }
    if (more) load_x(c + 1);
  };
  if (per > 0) {
    load_x(0);
#pragma unroll
    for (int t = 0; t < RT; ++t) load_w(0, t);
    for (int c = 0; c + 1 < per; ++c) piece(c, true);
    piece(per - 1, false);
  }
  __syncthreads();
  float (*red)[RT * MT][4][kWave] = reinterpret_cast<float (*)[RT * MT][4][kWave]>(raw);
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][t * MT + m][i][lane] = acc[t][m][i];
  __syncthreads();
  constexpr int kOuts = (PAIR ? 1 : RT) * MT * 256;
  for (int o = tid; o < kOuts; o += T) {
    const int tile = o >> 8, i = (o >> 6) & 3, ln = o & 63;
    const int rt = tile / MT, m = 16 * (tile % MT) + (ln & 15);
    const int row = row0 + 16 * rt + 4 * (ln >> 4) + i;
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < NW; ++q) v += red[q][tile][i][ln];
    if (PAIR) {
      float c = 0.f;
#pragma unroll
      for (int q = 0; q < NW; ++q) c += red[q][MT + tile][i][ln];
      v = silu(round_to<DT>(v)) * round_to<DT>(c);
    } else {
      if (sg.bias) v += E::load(sg.bias + row);
      if (sg.act) v = silu(round_to<DT>(v));
    }
    if (m < a.tokens) {
      const int64_t at = static_cast<int64_t>(m) * sg.out_stride + row;
      if (a.add1) v += E::load(a.add1 + at);
      if (a.add2) v += E::load(a.add2 + at);
      E::store(sg.out + at, v);
    }
  }
}

// ---- 3: attention of one query row over the cached keys ------------------------
// A workgroup takes a run of keys of one (sequence, head): scores (a key's 8-element pieces on
// LPK neighbouring lanes), softmax over the run, and the run's weighted sum of values, each
// thread owning eight of the value columns so that a value row is one contiguous read of
// the workgroup.  The first value rows are requested before the scores are known.
// The partial (max, sum, weighted values) go out in float32.  Every old key and value is read by
// exactly one workgroup, which writes it to its place in the new cache on the way: a cache that has been
// handed out is never written again, and the one that continues it is contiguous.  (Appended in place to storage
// with room the steps took 0.144 and 0.32 ms, but then a cache shares memory with the one it continues; with
// stores that stay in the caches 0.156 and 0.52.)
// The memory bounds it, old keys and values in and out, and how much of its rate is had depends on how many streams there
// are: a workgroup a CU, all of equal runs (key_runs).  AHEAD value rows and KU pieces of keys are in flight per thread:
// long runs twice as many as short ones, whose requests past the end are for nothing.
constexpr int kAttendThreads = 256;
constexpr int kMaxKeys = 4096;  // keys of a run
constexpr int kLongRun = 300;

struct AttendParams {
  const uint16_t *z, *gamma, *beta;  // (B, S); (2, S)
  const float* freqs;                // (zh / 2) complex, or null
  const uint16_t *k_old, *v_old;     // (B, total - 1, heads, zh | H2)
  uint16_t *k, *v;                   // (B, total, heads, zh | H2); the last row of v is written already
  float* part;                       // (B * heads, splits, H2)
  float2* ml;                        // (B * heads, splits): max and sum
  int heads, H2, total, splits, per; // total keys with the new one; per = keys of a run
  float eps, inv_sqrt;
};

template <int DT, int LPK, int AHEAD, int KU>
__global__ __launch_bounds__(kAttendThreads) void attend_kernel(const AttendParams a) {
  using E = Elem<DT>;
  __shared__ float score[kMaxKeys];
  __shared__ float wred[4];
  __shared__ float osum[kAttendThreads * 8];
  constexpr int zh = LPK * 8, KPW = 64 / LPK;  // keys per wave access
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int split = blockIdx.x, bh = blockIdx.y, b = bh / a.heads, h = bh % a.heads;
  const int k_lo = split * a.per, k_hi = k_lo + a.per < a.total ? k_lo + a.per : a.total;
  const int nk = k_hi - k_lo;
  const bool newest = k_hi == a.total;  // this run ends with the new token
  const int S = a.heads * zh, c = (lane & (LPK - 1)) * 8;

  // value rows: thread column c8 of key group kg
  const int cols = a.H2 >> 3, kgroups = kAttendThreads / cols, c8 = (tid % cols) * 8, kg = tid / cols;
  const int64_t vstep = static_cast<int64_t>(a.heads) * a.H2, vcol = static_cast<int64_t>(h) * a.H2 + c8;
  const int old_hi = newest ? nk - 1 : nk;  // keys of the run that the old cache holds
  const uint16_t* vp = a.v_old + (static_cast<int64_t>(b) * (a.total - 1) + k_lo) * vstep + vcol;
  uint16_t* vq = a.v + (static_cast<int64_t>(b) * a.total + k_lo) * vstep + vcol;
  uint4 ahead[AHEAD];
  auto request = [&](int i0) {  // rows past the run's end: the last one again, unused
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int j = i0 + i * kgroups, at = j < nk ? j : nk - 1;
      ahead[i] = load_once((at < old_hi ? vp : vq) + at * vstep);
    }
  };
  // The first keys and z are asked for in front of the first value rows: loads come back in order.
  const uint16_t* kp = a.k_old + (static_cast<int64_t>(b) * (a.total - 1) + k_lo) * S + h * zh + c;
  uint16_t* kq = a.k + (static_cast<int64_t>(b) * a.total + k_lo) * S + h * zh + c;
  uint4 raw[KU];
  auto request_keys = [&](int j0) {
#pragma unroll
    for (int i = 0; i < KU; ++i) {
      const int j = j0 + i * 4 * KPW;
      raw[i] = old_hi > 0 ? load_once(kp + static_cast<int64_t>(j < old_hi ? j : old_hi - 1) * S)
                          : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  const int at = h * zh + c;
  const uint4 z_raw = *reinterpret_cast<const uint4*>(a.z + static_cast<int64_t>(b) * S + at);
  request_keys(wave * KPW + lane / LPK);
  const uint4 g_raw = *reinterpret_cast<const uint4*>(a.gamma + at), b_raw = *reinterpret_cast<const uint4*>(a.beta + at);
  request(kg);

  // q, and for the run with the new token also k: every wave works them out for itself
  float q[8], kn[8];
  {
    float zv[8], g[8], bt[8];
    unpack8<DT>(z_raw, zv);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += zv[e] * zv[e];
    const float rs = rsqrtf(group_sum<LPK>(ss) / static_cast<float>(zh) + a.eps);
    float f[8];
    if (a.freqs) {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = a.freqs[c + e];
    }
    auto finish = [&](const uint4& gp, const uint4& bp, float* o) {
      unpack8<DT>(gp, g);
      unpack8<DT>(bp, bt);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = zv[e] * rs * ((g[e] + 1.f) * a.inv_sqrt) + bt[e];
      if (a.freqs) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x0 = o[2 * e], x1 = o[2 * e + 1];
          o[2 * e] = x0 * f[2 * e] - x1 * f[2 * e + 1];
          o[2 * e + 1] = x0 * f[2 * e + 1] + x1 * f[2 * e];
        }
      }
    };
    finish(g_raw, b_raw, q);
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = round_to<DT>(q[e]);
    if (newest) {
      finish(*reinterpret_cast<const uint4*>(a.gamma + S + at), *reinterpret_cast<const uint4*>(a.beta + S + at), kn);
      const uint4 packed = pack8<DT>(kn);
      if (tid < LPK)
        *reinterpret_cast<uint4*>(a.k + (static_cast<int64_t>(b) * a.total + a.total - 1) * S + at) = packed;
      unpack8<DT>(packed, kn);
    }
  }
  for (int j0 = wave * KPW + lane / LPK, first = 1; j0 - lane / LPK < old_hi; j0 += 4 * KPW * KU, first = 0) {
    if (!first) request_keys(j0);
#pragma unroll
    for (int i = 0; i < KU; ++i) {
      const int j = j0 + i * 4 * KPW;
      float kv[8], s = 0.f;
      if (j < old_hi) store_streaming(kq + static_cast<int64_t>(j) * S, raw[i]);
      unpack8<DT>(raw[i], kv);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += q[e] * kv[e];
      s = group_sum<LPK>(s);
      if (j < old_hi && c == 0) score[j] = s;
    }
  }
  if (newest) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += q[e] * kn[e];
    s = group_sum<LPK>(s);
    if (tid == 0) score[nk - 1] = s;
  }
  __syncthreads();
  float mx = -INFINITY;
  for (int j = tid; j < nk; j += kAttendThreads) mx = fmaxf(mx, score[j]);
  mx = wave_max(mx);
  if (lane == 0) wred[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(wred[0], wred[1]), fmaxf(wred[2], wred[3]));
  __syncthreads();
  float sum = 0.f;
  for (int j = tid; j < nk; j += kAttendThreads) {
    const float e = __expf(score[j] - mx);
    score[j] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) wred[wave] = sum;
  __syncthreads();
  sum = wred[0] + wred[1] + wred[2] + wred[3];

  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  for (int j0 = kg; j0 < nk; j0 += AHEAD * kgroups) {
    uint4 now[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) now[i] = ahead[i];
    request(j0 + AHEAD * kgroups);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int j = j0 + i * kgroups;
      const float w = j < nk ? score[j] : 0.f;
      if (j < old_hi) store_streaming(vq + j * vstep, now[i]);
      float vv[8];
      unpack8<DT>(now[i], vv);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] += (j < nk ? vv[e] : 0.f) * w;
    }
  }
  if (kgroups > 1) {
#pragma unroll
    for (int e = 0; e < 8; ++e) osum[tid * 8 + e] = o[e];
    __syncthreads();
    if (kg == 0)
      for (int s = 1; s < kgroups; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] += osum[(tid + s * cols) * 8 + e];
  }
  if (kg == 0) {
    float* dst = a.part + (static_cast<int64_t>(bh) * a.splits + split) * a.H2 + c8;
    *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
    *reinterpret_cast<float4*>(dst + 4) = make_float4(o[4], o[5], o[6], o[7]);
  }
  if (tid == 0) a.ml[static_cast<int64_t>(bh) * a.splits + split] = make_float2(mx, sum);
}

// ---- 4: the runs of a row put together, times silu(r) ---------------------------
// 64 columns of one (sequence, head) per workgroup, 16 threads along them (16 bytes each),
// 16 groups of threads along the runs.
struct CombineParams {
  const float* part;
  const float2* ml;
  const uint16_t* r;
  uint16_t* out;
  int heads, H2, splits;
};
template <int DT>
__global__ __launch_bounds__(256) void combine_kernel(const CombineParams a) {
  using E = Elem<DT>;
  __shared__ float4 sums[16][16];
  __shared__ float norm[16];
  const int tid = threadIdx.x, cg = tid & 15, sg = tid >> 4, bh = blockIdx.y, col = blockIdx.x * 64 + cg * 4;
  const float2* ml = a.ml + static_cast<int64_t>(bh) * a.splits;
  float mx = -INFINITY;
  for (int s = cg; s < a.splits; s += 16) mx = fmaxf(mx, ml[s].x);
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  float l = 0.f;
  const float* src = a.part + static_cast<int64_t>(bh) * a.splits * a.H2 + col;
#pragma unroll 4
  for (int s = sg; s < a.splits; s += 16) {
    const float2 m = ml[s];
    const float w = __expf(m.x - mx);
    const float4 v = *reinterpret_cast<const float4*>(src + static_cast<int64_t>(s) * a.H2);
    l += w * m.y;
    o.x += w * v.x;
    o.y += w * v.y;
    o.z += w * v.z;
    o.w += w * v.w;
  }
  sums[sg][cg] = o;
  if (cg == 0) norm[sg] = l;
  __syncthreads();
  if (tid < 64) {
    const int q4 = tid >> 2, e = tid & 3;
    float v = 0.f, n = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      v += reinterpret_cast<const float*>(&sums[s][q4])[e];
      n += norm[s];
    }
    const int64_t at = static_cast<int64_t>(bh) * a.H2 + blockIdx.x * 64 + tid;  // (B, heads * H2)
    v = round_to<DT>(v / n);
    E::store(a.out + at, v * silu(E::load(a.r + at)));
  }
}

// ---- host ----------------------------------------------------------------------
// Runs of keys: a workgroup for every CU, or for as many as equal shares of the pairs leave, where that is two thirds of them;
// else two.  At least 16 keys each (a run's partial result is 4 bytes per value column, a key 2).  Where the score buffer holds fewer, equal
// shares of as many more runs as that takes (us of a step, cut at the buffer's end with the rest in a run of its own / so: 32 sequences of
// eight heads of 512 value columns and 4101 keys 557 / 457, 5001 625 / 556, 24 of 4501 530 / 404, 32 of twenty heads of 128 and 4201 549 / 444).
// More pairs than CUs take two runs each up to half as many again and one above, of at most 1024 keys; a run each, up to the score buffer,
// left CUs with one workgroup where others had two (us, so cut / now, value columns of 256: 261 pairs of 700 keys 95 / 89, of 4090 364 / 320, 300 of
// 2000 221 / 198, of 4090 407 / 339, 341 of 2000 227 / 211, 384 234 / 223, 576 357 / 329; with two runs each 403 of 2000 would take 245 for 238, 480 of
// 64 columns and 700 keys 69 for 66).
// So do more than two thirds of the CUs' number where the keys are more than a fifth of what is read: while a lone workgroup is at its keys or
// between the two, nothing of its CU's is on the way (us, one run / so, key by value columns: 172 pairs of 256 x 64 and 4000 keys 226 / 193, of 1000
// 79 / 70, of 64 x 128 and 4000 132 / 120, 180 of 64 x 64 and 4000 107 / 101, 228 of 128 x 256 and 300 56.1 / 53.5, 256 of 64 x 64 and 2000 78.7 / 80.1; of 64 x
// 512 and 1000, where it does not hold, 180 115 / 119, of 256 x 1024 225 / 233).
// The number of CUs is a constant: the workspace is asked for apart from the launch, and both have to come to the same runs whatever
// device is current then.  With at least 512 workgroups, most of them resident two to a CU and a few left for the end, the step of
// four heads on 8 tokens took, us before / now: 1 x 1531 keys 986 / 968, 5 x 3900 2350 / 2144, 9 x 3000 2868 / 2577, 13 x 3000 3700 / 3260, 16 x
// 3000 3903 / 3738, 22 x 3000 (69 % of the CUs) 5692 / 4983, 32 x 3500 7822 / 7434; of eight heads 24 x 1000 (75 %) 8279 / 8083, 20 x
// 1000 (62 %, so two a CU) 7337 / 7239 where one a CU takes 7457.  With long requests for all 1 x 1531 took 982, with short ones
// 32 x 3500 7531.
constexpr int64_t kCus = 256;
void key_runs(int64_t pairs, int64_t total, int64_t zh, int64_t H2, int* splits, int* per) {
  int64_t want = kCus / pairs, most = kMaxKeys;
  if (pairs > kCus || (3 * pairs > 2 * kCus && H2 < 4 * zh)) want = 2 * pairs <= 3 * kCus ? 2 : 1, most = kMaxKeys / 4;
  else if (3 * want * pairs < 2 * kCus) want = 2 * kCus / pairs;
  int64_t n = (total + want - 1) / want;
  if (n < 16) n = 16;
  if (n > most) {
    const int64_t runs = (total + most - 1) / most;
    n = (total + runs - 1) / runs;
  }
  *per = static_cast<int>(n);
  *splits = static_cast<int>((total + n - 1) / n);
}

struct Layout {
  int64_t tsn, cema, normed, z, r, h1, attn, y1, hidden, ml, part, bytes;
};
Layout layout_of(const mega_block_decode_args& a) {
  int splits, per;
  key_runs(a.B * a.heads, a.length + 1, a.S / a.heads, a.E / a.heads, &splits, &per);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  Layout l;
  l.tsn = take(2 * a.B * a.D);
  l.cema = take(2 * a.B * a.D);
  l.normed = take(2 * a.B * a.D);
  l.z = take(2 * a.B * a.S);
  l.r = take(2 * a.B * a.E);
  l.h1 = take(2 * a.B * a.D);
  l.attn = take(2 * a.B * a.E);
  l.y1 = take(2 * a.B * a.D);
  l.hidden = take(2 * a.B * a.F);
  l.ml = take(8 * a.B * a.heads * splits);
  l.part = take(4 * a.B * a.E * splits);
  l.bytes = at;
  return l;
}

template <int DT, int MT, int RT, bool PAIR, int NW>
void tiles_as(const ProductParams& p, int blocks, hipStream_t s) {
  tiles_kernel<DT, MT, RT, PAIR, NW><<<blocks, NW * kWave, 0, s>>>(p);
}
template <int DT, int MT, int RT, bool PAIR>
void tiles(const ProductParams& p, hipStream_t s) {
  int blocks = 0;
  for (int i = 0; i < p.segs; ++i) blocks += p.seg[i].blocks;
  if constexpr (RT == 1) tiles_as<DT, MT, RT, PAIR, kTileNarrow>(p, blocks, s);
  else if (blocks < kTileFull) tiles_as<DT, MT, RT, PAIR, 4>(p, blocks, s);
  else tiles_as<DT, MT, RT, PAIR, 2>(p, blocks, s);
}

// Whether the products are rows_kernel's: up to four tokens, up to eight in narrow blocks (us, rows_kernel / tiles_kernel: eight
// sequences of one head of 1024 features 324 / 363, of two 522 / 506, of four 1259 / 1093; one of four 974 / 1090), and up to sixteen where
// the step is its launches, two fewer so (a token of nine / sixteen sequences: 128 features 33.3 / 33.5 and 36.5 / 37.7, 256 33.7 / 34.0 and 37.6 / 39.0,
// 384 34.6 / 34.7 and 38.4 / 39.2; at 480 40.1 / 40.2 and 39.0 / 38.5.  From 17 on those two launches cost 64 features 3 to 4 us of 34).
// Their norms come on the way, each workgroup's for itself, while that costs less than a launch: in front of fc1 and fc3 up to 2048
// features (us, on the way / ahead, four rows of each a workgroup: one sequence of two heads 417 / 417, four 424 / 432; of three 628 / 605, 816 / 807;
// of four 970 / 928, 1604 / 1586), in front of z, r and h1 but for one sequence of rows that give a wave a fourth piece (a token of one sequence
// of 100 keys, us, on the way / ahead: 2304 features 53.7 / 54.9, 2560 60.0 / 59.7, 2816 65.5 / 65.3, 3072 70.0 / 70.8, 3328 82.0 / 80.6, 3584 88.2 / 87.1, 3840
// 95.6 / 94.5, 4096 105.7 / 102.5; eight of two sequences of 4096 877 / 883).
bool few_rows(int B, int D) { return D <= norm_row(kNormRms, 1) && B <= (D <= 384 ? 16 : D < norm_row(kNormRms, 2) ? 8 : 4); }
template <int DT, int TT, int G, bool PAIR, int NORM>
void rows(ProductParams p, hipStream_t s) {
  int blocks = 0;
  for (int i = 0; i < p.segs; ++i) blocks += p.seg[i].blocks;
  rows_kernel<DT, TT, G, PAIR, NORM><<<blocks, kRowsWaves * kWave, 0, s>>>(p);
}

template <int DT, int AHEAD, int KU>
void attend(const AttendParams& p, int zh, dim3 grid, hipStream_t s) {
  if (zh == 64) attend_kernel<DT, 8, AHEAD, KU><<<grid, kAttendThreads, 0, s>>>(p);
  else if (zh == 128) attend_kernel<DT, 16, AHEAD, KU><<<grid, kAttendThreads, 0, s>>>(p);
  else attend_kernel<DT, 32, AHEAD, KU><<<grid, kAttendThreads, 0, s>>>(p);
}

template <int DT, int MT>
int run(const mega_block_decode_args& a, hipStream_t s) {
  const Layout l = layout_of(a);
  char* ws = static_cast<char*>(a.workspace);
  auto u16 = [](const void* p) { return static_cast<const uint16_t*>(p); };
  auto at16 = [&](int64_t off) { return reinterpret_cast<uint16_t*>(ws + off); };
  const int D = static_cast<int>(a.D), B = static_cast<int>(a.B), E = static_cast<int>(a.E), S = static_cast<int>(a.S),
            F = static_cast<int>(a.F), H = static_cast<int>(a.heads);
  {
    StepParams p{u16(a.x), u16(a.prev_mean), u16(a.prev_var), u16(a.tsn_weight), u16(a.tsn_bias), u16(a.omega),
                 a.prev_count, a.p, a.q, a.gamma_hat, reinterpret_cast<const float4*>(a.h_in), at16(l.tsn),
                 at16(l.cema), static_cast<uint16_t*>(a.mean), static_cast<uint16_t*>(a.var), a.count,
                 reinterpret_cast<float4*>(a.h_out), D,
                 static_cast<int>(a.G), static_cast<int>(a.D / a.G), a.tsn_eps};
    step_kernel<DT><<<dim3(D / kStepChannels, B), 256, 0, s>>>(p);
  }
  const uint16_t* none = nullptr;
  const bool few = few_rows(B, D);
  const bool front = !few || (B == 1 && D > 3 * kRowsWaves * 128), behind = !few || D > norm_row(kNormLayer, 1);  // whether the norms have launches of their own
  // rows of a workgroup: of z, r, h1 and v, of fc1 and fc3 (a pair), of wh2 and fc2
  const int wide = !few ? 32 : front ? 4 : 16, pair = !few ? 16 : behind ? 4 : 8, narrow = !few ? 16 : B <= 4 || B > 8 ? 4 : 8;
  auto seg = [&](const void* W, const void* W2, const void* bias, const uint16_t* x, uint16_t* out, int64_t stride,
                 int rows, int strip, int norm, int act) {
    return Segment{u16(W), u16(W2), u16(bias), x, out, stride, rows / strip, norm, act};
  };
  {
    if (front)
      rows_norm_kernel<DT, kNormRms><<<B, kNormThreads, 0, s>>>(at16(l.cema), u16(a.rms_weight), none, at16(l.normed), D, a.rms_eps);
    const uint16_t* row = at16(front ? l.normed : l.cema);
    ProductParams p{};
    // the wide layers first: the narrow one fills the gaps at the end
    p.seg[0] = seg(a.wv, none, a.bv, at16(l.tsn), static_cast<uint16_t*>(a.v_out) + a.length * a.E,
                   (a.length + 1) * a.E, E, wide, kNormNone, 1);
    p.seg[1] = seg(a.wr, none, a.br, row, at16(l.r), E, E, wide, kNormRms, 0);
    p.seg[2] = seg(a.wh1, none, a.bh1, row, at16(l.h1), D, D, wide, kNormRms, 0);
    p.seg[3] = seg(a.wz, none, a.bz, row, at16(l.z), S, S, wide, kNormRms, 0);
    p.segs = 4, p.K = D, p.tokens = B;
    p.norm_weight = u16(a.rms_weight);
    p.eps = a.rms_eps;
    if (!few) tiles<DT, MT, 2, false>(p, s);
    else if (front) rows<DT, 1, 1, false, kNormNone>(p, s);
    else if (B <= 4) rows<DT, 1, 4, false, kNormRms>(p, s);
    else if (B <= 8) rows<DT, 2, 4, false, kNormRms>(p, s);
    else rows<DT, 4, 4, false, kNormRms>(p, s);
  }
  const int zh = S / H, H2 = E / H;
  int splits, per;
  key_runs(static_cast<int64_t>(B) * H, a.length + 1, zh, H2, &splits, &per);
  {
    AttendParams p{at16(l.z), u16(a.qk_gamma), u16(a.qk_beta), a.freqs, u16(a.k_in), u16(a.v_in),
                   static_cast<uint16_t*>(a.k_out), static_cast<uint16_t*>(a.v_out), reinterpret_cast<float*>(ws + l.part),
                   reinterpret_cast<float2*>(ws + l.ml), H, H2, static_cast<int>(a.length + 1), splits, per, a.z_eps,
                   1.f / sqrtf(static_cast<float>(zh))};
    const dim3 grid(splits, B * H);
    if (per >= kLongRun) attend<DT, 16, 8>(p, zh, grid, s);
    else attend<DT, 8, 4>(p, zh, grid, s);
  }
  {
    CombineParams p{reinterpret_cast<const float*>(ws + l.part), reinterpret_cast<const float2*>(ws + l.ml),
                    at16(l.r), at16(l.attn), H, H2, splits};
    combine_kernel<DT><<<dim3(H2 / 64, B * H), 256, 0, s>>>(p);
  }
  {
    ProductParams p{};
    p.seg[0] = seg(a.wh2, none, none, at16(l.attn), at16(l.y1), D, D, narrow, kNormNone, 0);
    p.segs = 1, p.K = E, p.tokens = B;
    p.add1 = at16(l.h1), p.add2 = u16(a.x);
    if (!few) tiles<DT, MT, 1, false>(p, s);
    else if (B <= 4) rows<DT, 1, 1, false, kNormNone>(p, s);
    else if (B <= 8) rows<DT, 2, 2, false, kNormNone>(p, s);
    else rows<DT, 4, 1, false, kNormNone>(p, s);
  }
  {
    if (behind)
      rows_norm_kernel<DT, kNormLayer><<<B, kNormThreads, 0, s>>>(at16(l.y1), u16(a.ln_weight), u16(a.ln_bias), at16(l.normed), D, a.ln_eps);
    ProductParams p{};
    p.seg[0] = seg(a.fc1, a.fc3, none, at16(behind ? l.normed : l.y1), at16(l.hidden), F, F, pair, kNormLayer, 0);
    p.segs = 1, p.K = D, p.tokens = B;
    p.norm_weight = u16(a.ln_weight), p.norm_bias = u16(a.ln_bias);
    p.eps = a.ln_eps;
    if (!few) tiles<DT, MT, 2, true>(p, s);
    else if (behind) rows<DT, 1, 2, true, kNormNone>(p, s);
    else if (B <= 4) rows<DT, 1, 4, true, kNormLayer>(p, s);
    else if (B <= 8) rows<DT, 2, 4, true, kNormLayer>(p, s);
    else rows<DT, 4, 4, true, kNormLayer>(p, s);
  }
  {
    ProductParams p{};
    p.seg[0] = seg(a.fc2, none, none, at16(l.hidden), static_cast<uint16_t*>(a.y), D, D, narrow, kNormNone, 0);
    p.segs = 1, p.K = F, p.tokens = B;
    p.add1 = u16(a.x);
    if (!few) tiles<DT, MT, 1, false>(p, s);
    else if (B <= 4) rows<DT, 1, 1, false, kNormNone>(p, s);
    else if (B <= 8) rows<DT, 2, 2, false, kNormNone>(p, s);
    else rows<DT, 4, 1, false, kNormNone>(p, s);
  }
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_block_decode_supported(int dtype, int64_t B, int64_t D, int64_t S, int64_t E, int64_t F,
                                           int64_t heads, int64_t G, int64_t N) {
  if ((dtype != MEGA_BF16 && dtype != MEGA_F16) || B < 1 || B > kMaxTokens || N != kModes || heads < 1 || G < 1) return 0;
  if (D > 8192 || D % 32 || E % 32 || S % 32 || F % 32 || D % G || S % heads || E % heads) return 0;
  const int64_t Dg = D / G, zh = S / heads, H2 = E / heads;
  if (Dg % kStepChannels || (zh != 64 && zh != 128 && zh != 256)) return 0;
  // value columns: eight per thread, whole key groups in a workgroup
  return H2 == 64 || H2 == 128 || H2 == 256 || H2 == 512 || H2 == 1024 || H2 == 2048;
}

extern "C" int64_t mega_block_decode_workspace_bytes(const mega_block_decode_args* a) {
  return a == nullptr ? -1 : layout_of(*a).bytes;
}

extern "C" int mega_block_decode(const mega_block_decode_args* a, void* stream) {
  const char* who = "mega_block_decode";
  MEGA_CHECK_ARG(a != nullptr, "%s: null arguments", who);
  if (!mega_block_decode_supported(a->dtype, a->B, a->D, a->S, a->E, a->F, a->heads, a->G, a->N))
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: sizes outside what the step kernels take", who);
  MEGA_CHECK_ARG(a->length >= 1 && a->length < (1 << 24), "%s: length must be at least 1", who);
  for (const void* q : {a->x, a->prev_mean, a->prev_var, a->tsn_weight, a->tsn_bias, a->omega, a->wz, a->wr, a->wh1,
                        a->wv, a->wh2, a->qk_gamma, a->qk_beta, a->fc1, a->fc2, a->fc3,
                        static_cast<const void*>(a->p), static_cast<const void*>(a->q),
                        static_cast<const void*>(a->gamma_hat), static_cast<const void*>(a->h_in),
                        a->k_in, a->v_in, static_cast<const void*>(a->k_out), static_cast<const void*>(a->v_out),
                        static_cast<const void*>(a->y), static_cast<const void*>(a->mean),
                        static_cast<const void*>(a->var), static_cast<const void*>(a->h_out),
                        static_cast<const void*>(a->workspace)})
    MEGA_CHECK_ARG(q != nullptr, "%s: null pointer", who);
  MEGA_CHECK_ARG(a->prev_count && a->count, "%s: null pointer", who);
  for (const void* q : {a->wz, a->wr, a->wh1, a->wv, a->wh2, a->fc1, a->fc2, a->fc3, a->rms_weight, a->ln_weight,
                        a->ln_bias, a->qk_gamma, a->qk_beta, static_cast<const void*>(a->p),
                        static_cast<const void*>(a->q), static_cast<const void*>(a->gamma_hat),
                        static_cast<const void*>(a->h_in), static_cast<const void*>(a->h_out),
                        a->k_in, a->v_in, static_cast<const void*>(a->k_out), static_cast<const void*>(a->v_out),
                        static_cast<const void*>(a->workspace)})
    MEGA_CHECK_ARG(reinterpret_cast<uintptr_t>(q) % 16 == 0, "%s: operands must be 16-byte aligned", who);
  MEGA_CHECK_ARG(a->k_in != a->k_out && a->v_in != a->v_out, "%s: the new cache must not be the old one", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == MEGA_BF16) return a->B <= 16 ? run<MEGA_BF16, 1>(*a, s) : run<MEGA_BF16, 2>(*a, s);
  return a->B <= 16 ? run<MEGA_F16, 1>(*a, s) : run<MEGA_F16, 2>(*a, s);
}
