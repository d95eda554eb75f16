// One new token per sequence through a whole block, for generation from a cache
// (the cache branch of megalodon/modules/moving_average_gated_attention.py:283-348
// followed by normalized_feedforward_network.py:74-90, at sequence length one).
//
// The step is bound by reading the block's weights once and moving the cached keys and
// values once: at width 4096 the weights are 514 MB, and operator by operator a
// step was 59 launches, 0.84 ms for one sequence and 4.1 ms for sixteen (1531 and
// 3000 cached tokens).  Here it is seven launches, 0.151 and 0.50 ms, cut where a whole row is needed by everybody:
//   1. step_kernel    TimestepNorm step, EMA state step, partial square sums of the row
//   2. skinny_kernel  RMSNorm folded into z, r, h1; v = silu(...) straight into the new cache
//   3. attend_kernel  q, k (norm, affine maps, rotary), one softmax part per split; the old keys and values
//                     pass into the new cache as they are read, the new key joins them
//   4. combine_kernel the parts put together, gate silu(r)
//   5. skinny_kernel  wh2 + h1 + residual, partial moments of the row
//   6. skinny_kernel  LayerNorm folded into fc1, fc3; silu(a) b
//   7. skinny_kernel  fc2 + residual
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
  float* squares;  // (B, D / 32): sum of squares of the stored EMA outputs
  int D, G, Dg;
  float eps;
};

template <int DT>
__global__ __launch_bounds__(256) void step_kernel(const StepParams a) {
  using E = Elem<DT>;
  __shared__ float part[4];
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
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
  const float sq = wave_sum(m2 == 0 ? out * out : 0.f);
  if (lane == 0) part[wave] = sq;
  __syncthreads();
  if (tid == 0) a.squares[static_cast<int64_t>(b) * gridDim.x + blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// ---- 2, 5, 6, 7: products of a weight matrix with at most 32 rows --------------
// out[m][n] = sum_k x[m][k] W[n][k].  What counts is that the weights stream in at the
// memory's rate: each is read once, 16 bytes per lane straight into the operand of a
// 16x16x32 product (16 weight rows by 16 or 32 tokens; the matrix pipe is idle otherwise,
// so columns without a token cost nothing).  A workgroup of NW waves takes a strip of 16
// rows (RT strips), its waves equal runs of the reduction; two batches of
// loads are kept in flight per wave, 128 or 256 contiguous bytes of every row, and the first is requested
// before the row statistics are put together.  x comes through the caches (at most 700 KB for all).
// A normalisation in front of the product is applied to the operand on its way in.
// Waves per strip.  Two-strip products have 672 and 688 workgroups at width 4096: four waves each
// are all resident at once (eight ran 45.9 / 50.0 us, four 40.6 / 45.6, two 41.5 / 44.4 for 176 / 180 MB).
// One-strip products have one workgroup per compute unit there: eight (16.2 / 20.6 us for 67 / 90 MB;
// sixteen 18.9 / 23.8).
constexpr int kWavesWide = 4, kWavesNarrow = 8;
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
struct SkinnyParams {
  Segment seg[kMaxSegs];
  int segs, K, tokens;
  const uint16_t *norm_weight, *norm_bias;  // stored weight = gamma - 1; may be null
  const float* stats;      // RMS: (tokens, stat_parts) square sums; layer: (stat_parts, tokens) x (mean, M2) of 16 values
  int stat_parts, stat_count;  // partial results per token, values behind one
  float eps;
  const uint16_t *add1, *add2;  // (tokens, rows), added to the result
  float2* moments;         // (workgroups, tokens): mean and M2 of this workgroup's 16 stored values, or null
};

// PAIR: the two strips are the same rows of two matrices and silu(a) b is stored;
// otherwise RT consecutive strips of one.
template <int DT, int MT, int RT, bool PAIR, int NORM, int NW>
__global__ __launch_bounds__(NW * kWave, MT == 1 ? 4 : 2) void skinny_kernel(const SkinnyParams a) {
  using E = Elem<DT>;
  constexpr int T = NW * kWave;
  __shared__ float red[NW][RT * MT][4][kWave];
  __shared__ float st_mean[kMaxTokens], st_rstd[kMaxTokens];
  extern __shared__ __align__(16) uint16_t norm_lds[];  // K values of the norm's weight, K of its bias
  // (uniform to the compiler: a matrix instruction ignores the lane mask, so a step past the wave's
  // end has to be skipped by a branch)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int blk = blockIdx.x, si = 0;
  while (blk >= a.seg[si].blocks) blk -= a.seg[si++].blocks;
  const Segment& sg = a.seg[si];
  constexpr int kRows = PAIR ? 16 : 16 * RT;
  const int row0 = blk * kRows;
  const int r = lane & 15, kg = lane >> 4;
  const int steps = a.K / 32, per = (steps + NW - 1) / NW;
  const int s_lo = wave * per < steps ? wave * per : steps, s_hi = s_lo + per < steps ? s_lo + per : steps;

  const uint16_t* wp[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
    wp[t] = (PAIR && t == 1 ? sg.W2 : sg.W) + static_cast<int64_t>(row0 + (PAIR ? 0 : 16 * t) + r) * a.K + 8 * kg;
  const uint16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = 16 * t + r;
    xp[t] = sg.x + static_cast<int64_t>(m < a.tokens ? m : 0) * a.K + 8 * kg;
  }
  floatx4 acc[RT][MT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = floatx4{0.f, 0.f, 0.f, 0.f};

  constexpr int kSteps = 4 / RT;  // steps of 32 per batch
  // weights and x of a batch of steps are requested together, in the order in which they are waited
  // for: a wait for x would otherwise also wait for the weights requested ahead
  struct Batch {
    u32x4 w[RT][kSteps], x[MT][kSteps];
  };
  Batch b0, b1;
  auto request = [&](Batch& t, int s) {  // steps past the wave's end: the last one again, unused
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const int64_t k = 32 * static_cast<int64_t>(s + i < s_hi ? s + i : (s_hi > 0 ? s_hi - 1 : 0));
#pragma unroll
      for (int j = 0; j < RT; ++j) t.w[j][i] = *reinterpret_cast<const u32x4*>(wp[j] + k);
#pragma unroll
      for (int j = 0; j < MT; ++j) t.x[j][i] = *reinterpret_cast<const u32x4*>(xp[j] + k);
    }
  };
  request(b0, s_lo);

  float mean[MT], rstd[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) mean[t] = 0.f, rstd[t] = 1.f;
  const bool normed = NORM != kNormNone && sg.norm != kNormNone;
  if (NORM != kNormNone) {
    // the norm's weight and bias, read from LDS in the loop
    for (int k = tid * 8; k < a.K; k += T * 8) {
      const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
      *reinterpret_cast<uint4*>(norm_lds + k) =
          a.norm_weight ? *reinterpret_cast<const uint4*>(a.norm_weight + k) : zero;
      if (NORM == kNormLayer)
        *reinterpret_cast<uint4*>(norm_lds + a.K + k) =
            a.norm_bias ? *reinterpret_cast<const uint4*>(a.norm_bias + k) : zero;
    }
    // 16 threads per token put its partial results together
    const int j = tid & 15;
    for (int m = tid >> 4; m < a.tokens; m += T / 16) {
      const float inv = 1.f / static_cast<float>(a.K);
      if (NORM == kNormRms) {
        float s = 0.f;
        for (int i = j; i < a.stat_parts; i += 16) s += a.stats[static_cast<int64_t>(m) * a.stat_parts + i];
        s = group_sum<16>(s);
        if (j == 0) st_mean[m] = 0.f, st_rstd[m] = rsqrtf(s * inv + a.eps);
      } else {
        const float2* st = reinterpret_cast<const float2*>(a.stats);
        float s = 0.f, q = 0.f;
        for (int i = j; i < a.stat_parts; i += 16) s += st[static_cast<int64_t>(i) * a.tokens + m].x;
        const float mu = group_sum<16>(s) / static_cast<float>(a.stat_parts);  // equal counts behind every part
        for (int i = j; i < a.stat_parts; i += 16) {
          const float2 v = st[static_cast<int64_t>(i) * a.tokens + m];
          q += v.y + static_cast<float>(a.stat_count) * (v.x - mu) * (v.x - mu);
        }
        q = group_sum<16>(q);
        if (j == 0) st_mean[m] = mu, st_rstd[m] = rsqrtf(q * inv + a.eps);
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = 16 * t + r < a.tokens ? 16 * t + r : 0;
      mean[t] = st_mean[m];
      rstd[t] = st_rstd[m];
    }
  }

  auto consume = [&](Batch& t, int s) {
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      if (s + i < s_hi) {
        if (NORM != kNormNone && normed) {
          const int k = 32 * (s + i) + 8 * kg;
          float g[8], c[8], v[8];
          unpack8<DT>(*reinterpret_cast<const uint4*>(norm_lds + k), g);
          if (NORM == kNormLayer) unpack8<DT>(*reinterpret_cast<const uint4*>(norm_lds + a.K + k), c);
#pragma unroll
          for (int j = 0; j < MT; ++j) {
            unpack8<DT>(make_uint4(t.x[j][i][0], t.x[j][i][1], t.x[j][i][2], t.x[j][i][3]), v);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              v[e] = NORM == kNormLayer ? (v[e] - mean[j]) * rstd[j] * (g[e] + 1.f) + c[e] : v[e] * rstd[j] * (g[e] + 1.f);
            const uint4 pk = pack8<DT>(v);
            t.x[j][i] = u32x4{pk.x, pk.y, pk.z, pk.w};
          }
        }
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[j][m] = mma16<DT>(t.w[j][i], t.x[m][i], acc[j][m]);
      }
    }
  };
  for (int s = s_lo; s < s_hi; s += 2 * kSteps) {
    request(b1, s + kSteps);
    consume(b0, s);
    if (s + kSteps < s_hi) {
      request(b0, s + 2 * kSteps);
      consume(b1, s + kSteps);
    }
  }

#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][t * MT + m][i][lane] = acc[t][m][i];
  __syncthreads();
  // value (i, lane) of a tile: weight row 4 (lane / 16) + i, token lane % 16
  constexpr int kOuts = (PAIR ? 1 : RT) * MT * 256;
  for (int o = tid; o < kOuts; o += T) {
    const int tile = o >> 8, i = (o >> 6) & 3, ln = o & 63;
    const int rt = tile / MT, m = 16 * (tile % MT) + (ln & 15);
    const int row = row0 + 16 * rt + 4 * (ln >> 4) + i;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[w][tile][i][ln];
    if (PAIR) {
      float c = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) c += red[w][MT + tile][i][ln];
      v = silu(round_to<DT>(v)) * round_to<DT>(c);
    } else {
      if (sg.bias) v += E::load(sg.bias + row);
      if (sg.act) v = silu(round_to<DT>(v));
    }
    const bool on = m < a.tokens;
    if (on) {
      const int64_t at = static_cast<int64_t>(m) * sg.out_stride + row;
      if (a.add1) v += E::load(a.add1 + at);
      if (a.add2) v += E::load(a.add2 + at);
      E::store(sg.out + at, v);
    }
    if (RT == 1 && a.moments) {
      // mean and M2 of the strip's 16 values per token: four of them in this wave's lanes ...
      v = round_to<DT>(v);
      float s1 = v;
      s1 += __shfl_xor(s1, 16, 64);
      s1 += __shfl_xor(s1, 32, 64);
      const float mu4 = 0.25f * s1;
      float q = (v - mu4) * (v - mu4);
      q += __shfl_xor(q, 16, 64);
      q += __shfl_xor(q, 32, 64);
      if (ln < 16) {  // the slots of (tile, i) have been read by this very wave only
        red[0][tile][i][ln] = mu4;
        red[1][tile][i][ln] = q;
      }
    }
  }
  if (RT == 1 && a.moments) {
    __syncthreads();
    if (tid < a.tokens) {
      const int tile = tid >> 4, ln = tid & 15;
      float mu = 0.f, q = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) mu += 0.25f * red[0][tile][i][ln];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float dm = red[0][tile][i][ln] - mu;
        q += red[1][tile][i][ln] + 4.f * dm * dm;
      }
      a.moments[static_cast<int64_t>(blockIdx.x) * a.tokens + tid] = make_float2(mu, q);
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
constexpr int kAttendThreads = 256;
constexpr int kMaxKeys = 1024;  // keys of a run
constexpr int kAhead = 8;       // value rows in flight per thread

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

template <int DT, int LPK>
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
  uint4 ahead[kAhead];
  auto request = [&](int i0) {  // rows past the run's end: the last one again, unused
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int j = i0 + i * kgroups, at = j < nk ? j : nk - 1;
      ahead[i] = load_once((at < old_hi ? vp : vq) + at * vstep);
    }
  };
  request(kg);

  // q, and for the run with the new token also k: every wave works them out for itself
  float q[8], kn[8];
  {
    float zv[8], g[8], bt[8];
    const int at = h * zh + c;
    unpack8<DT>(*reinterpret_cast<const uint4*>(a.z + static_cast<int64_t>(b) * S + at), zv);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += zv[e] * zv[e];
    const float rs = rsqrtf(group_sum<LPK>(ss) / static_cast<float>(zh) + a.eps);
    float f[8];
    if (a.freqs) {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = a.freqs[c + e];
    }
    auto finish = [&](const uint16_t* gp, const uint16_t* bp, float* o) {
      unpack8<DT>(*reinterpret_cast<const uint4*>(gp + at), g);
      unpack8<DT>(*reinterpret_cast<const uint4*>(bp + at), bt);
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
    finish(a.gamma, a.beta, q);
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = round_to<DT>(q[e]);
    if (newest) {
      finish(a.gamma + S, a.beta + S, kn);
      const uint4 packed = pack8<DT>(kn);
      if (tid < LPK)
        *reinterpret_cast<uint4*>(a.k + (static_cast<int64_t>(b) * a.total + a.total - 1) * S + at) = packed;
      unpack8<DT>(packed, kn);
    }
  }
  const uint16_t* kp = a.k_old + (static_cast<int64_t>(b) * (a.total - 1) + k_lo) * S + h * zh + c;
  uint16_t* kq = a.k + (static_cast<int64_t>(b) * a.total + k_lo) * S + h * zh + c;
  constexpr int kU = 4;
  for (int j0 = wave * KPW + lane / LPK; j0 - lane / LPK < old_hi; j0 += 4 * KPW * kU) {
    uint4 raw[kU];
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int j = j0 + i * 4 * KPW;
      raw[i] = old_hi > 0 ? load_once(kp + static_cast<int64_t>(j < old_hi ? j : old_hi - 1) * S)
                          : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int i = 0; i < kU; ++i) {
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
  for (int j0 = kg; j0 < nk; j0 += kAhead * kgroups) {
    uint4 now[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) now[i] = ahead[i];
    request(j0 + kAhead * kgroups);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
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
// Runs of keys: enough workgroups to fill the chip twice over, at least 16 keys each (a run's
// partial result is 4 bytes per value column, a key 2), at most what the score buffer holds.
void key_runs(int64_t pairs, int64_t total, int* splits, int* per) {
  int64_t want = (512 + pairs - 1) / pairs;
  int64_t n = (total + want - 1) / want;
  if (n < 16) n = 16;
  if (n > kMaxKeys) n = kMaxKeys;
  *per = static_cast<int>(n);
  *splits = static_cast<int>((total + n - 1) / n);
}

struct Layout {
  int64_t tsn, cema, z, r, h1, attn, y1, hidden, squares, moments, ml, part, bytes;
};
Layout layout_of(const mega_block_decode_args& a) {
  int splits, per;
  key_runs(a.B * a.heads, a.length + 1, &splits, &per);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  Layout l;
  l.tsn = take(2 * a.B * a.D);
  l.cema = take(2 * a.B * a.D);
  l.z = take(2 * a.B * a.S);
  l.r = take(2 * a.B * a.E);
  l.h1 = take(2 * a.B * a.D);
  l.attn = take(2 * a.B * a.E);
  l.y1 = take(2 * a.B * a.D);
  l.hidden = take(2 * a.B * a.F);
  l.squares = take(4 * a.B * (a.D / kStepChannels));
  l.moments = take(8 * a.B * (a.D / 16));
  l.ml = take(8 * a.B * a.heads * splits);
  l.part = take(4 * a.B * a.E * splits);
  l.bytes = at;
  return l;
}

template <int DT, int MT, int RT, bool PAIR, int NORM, int NW>
void skinny(const SkinnyParams& p, hipStream_t s) {
  int blocks = 0;
  for (int i = 0; i < p.segs; ++i) blocks += p.seg[i].blocks;
  const size_t lds = NORM == kNormNone ? 0 : sizeof(uint16_t) * p.K * (NORM == kNormLayer ? 2 : 1);
  skinny_kernel<DT, MT, RT, PAIR, NORM, NW><<<blocks, NW * kWave, lds, s>>>(p);
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
                 reinterpret_cast<float4*>(a.h_out), reinterpret_cast<float*>(ws + l.squares), D,
                 static_cast<int>(a.G), static_cast<int>(a.D / a.G), a.tsn_eps};
    step_kernel<DT><<<dim3(D / kStepChannels, B), 256, 0, s>>>(p);
  }
  const uint16_t* none = nullptr;
  auto seg = [&](const void* W, const void* W2, const void* bias, const uint16_t* x, uint16_t* out, int64_t stride,
                 int rows, int strip, int norm, int act) {
    return Segment{u16(W), u16(W2), u16(bias), x, out, stride, rows / strip, norm, act};
  };
  {
    SkinnyParams p{};
    // the wide layers first: the narrow one fills the gaps at the end
    p.seg[0] = seg(a.wv, none, a.bv, at16(l.tsn), static_cast<uint16_t*>(a.v_out) + a.length * a.E,
                   (a.length + 1) * a.E, E, 32, kNormNone, 1);
    p.seg[1] = seg(a.wr, none, a.br, at16(l.cema), at16(l.r), E, E, 32, kNormRms, 0);
    p.seg[2] = seg(a.wh1, none, a.bh1, at16(l.cema), at16(l.h1), D, D, 32, kNormRms, 0);
    p.seg[3] = seg(a.wz, none, a.bz, at16(l.cema), at16(l.z), S, S, 32, kNormRms, 0);
    p.segs = 4, p.K = D, p.tokens = B;
    p.norm_weight = u16(a.rms_weight);
    p.stats = reinterpret_cast<const float*>(ws + l.squares), p.stat_parts = D / kStepChannels, p.eps = a.rms_eps;
    skinny<DT, MT, 2, false, kNormRms, kWavesWide>(p, s);
  }
  const int zh = S / H, H2 = E / H;
  int splits, per;
  key_runs(static_cast<int64_t>(B) * H, a.length + 1, &splits, &per);
  {
    AttendParams p{at16(l.z), u16(a.qk_gamma), u16(a.qk_beta), a.freqs, u16(a.k_in), u16(a.v_in),
                   static_cast<uint16_t*>(a.k_out), static_cast<uint16_t*>(a.v_out), reinterpret_cast<float*>(ws + l.part),
                   reinterpret_cast<float2*>(ws + l.ml), H, H2, static_cast<int>(a.length + 1), splits, per, a.z_eps,
                   1.f / sqrtf(static_cast<float>(zh))};
    const dim3 grid(splits, B * H);
    if (zh == 64) attend_kernel<DT, 8><<<grid, kAttendThreads, 0, s>>>(p);
    else if (zh == 128) attend_kernel<DT, 16><<<grid, kAttendThreads, 0, s>>>(p);
    else attend_kernel<DT, 32><<<grid, kAttendThreads, 0, s>>>(p);
  }
  {
    CombineParams p{reinterpret_cast<const float*>(ws + l.part), reinterpret_cast<const float2*>(ws + l.ml),
                    at16(l.r), at16(l.attn), H, H2, splits};
    combine_kernel<DT><<<dim3(H2 / 64, B * H), 256, 0, s>>>(p);
  }
  {
    SkinnyParams p{};
    p.seg[0] = seg(a.wh2, none, none, at16(l.attn), at16(l.y1), D, D, 16, kNormNone, 0);
    p.segs = 1, p.K = E, p.tokens = B;
    p.add1 = at16(l.h1), p.add2 = u16(a.x);
    p.moments = reinterpret_cast<float2*>(ws + l.moments);
    skinny<DT, MT, 1, false, kNormNone, kWavesNarrow>(p, s);
  }
  {
    SkinnyParams p{};
    p.seg[0] = seg(a.fc1, a.fc3, none, at16(l.y1), at16(l.hidden), F, F, 16, kNormLayer, 0);
    p.segs = 1, p.K = D, p.tokens = B;
    p.norm_weight = u16(a.ln_weight), p.norm_bias = u16(a.ln_bias);
    p.stats = reinterpret_cast<const float*>(ws + l.moments), p.stat_parts = D / 16, p.stat_count = 16;
    p.eps = a.ln_eps;
    skinny<DT, MT, 2, true, kNormLayer, kWavesWide>(p, s);
  }
  {
    SkinnyParams p{};
    p.seg[0] = seg(a.fc2, none, none, at16(l.hidden), static_cast<uint16_t*>(a.y), D, D, 16, kNormNone, 0);
    p.segs = 1, p.K = F, p.tokens = B;
    p.add1 = u16(a.x);
    skinny<DT, MT, 1, false, kNormNone, kWavesNarrow>(p, s);
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
