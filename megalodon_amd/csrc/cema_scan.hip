// The CEMA layer as a chunked linear recurrence on the matrix cores.
//
// The layer's convolution kernel is a sum of N damped complex exponentials,
//   k[j] = Re sum_n c_n q_n^j,  c_n = p_n gamma_n
// (megalodon/csrc/ops/ema_parameters.cc:37-52), so
//   y = fftconv(x, k) + omega x  (+ the bias of a carried state)
// (megalodon/modules/complex_exponential_moving_average.py:127-147) is the
// output of the recurrence h[t] = q h[t-1] + p x[t], y[t] = Re sum_n gamma_n
// h_n[t] + omega x[t] (the same states ema_hidden.cc:31-61 returns).  Neither k
// nor any spectrum is formed.  A row is cut into chunks of T = 64 steps; with
// X[c][j] = x[64 c + j]:
//   S[c]    = P X[c],          P[m][j]  = (Re, Im)(p_n q_n^(63-j)),  m = 2 n + part   (local state)
//   H[c]    = q^64 H[c-1] + S[c],  H[-1] = carried state                             (scan over chunks)
//   Y[c]    = K X[c] + Q H[c-1],  K[i][j] = k[i-j] (i >= j),  Q[i][m] = (Re, -Im)(gamma_n q_n^(i+1))
// The three products are MFMAs with the chunks of a tile as the 32 columns
// (v_mfma_f32_32x32x16_bf16); a row of x is read from memory once, straight
// into operand registers (a lane's 16-byte load is 8 consecutive steps of one
// chunk), and y is written once from the accumulators.  Parameter matrices are
// float32 values split into two bf16 pieces (hi + lo, 16 significant bits; some have a third, see kFine); x in
// bf16 is exact, fp16 x is split into two exact bf16 pieces; the states are
// float32 and split the same way (where float32 rows need more, the state's products are float32 ones, see XOpWide);
// accumulation is float32.
//
// One workgroup of four waves owns a channel's rows: one of them, or, where the batch has several,
// as many as still leave a workgroup for every slot of the chip.  Setting up the channel's parameter
// matrices costs as much as half an item, and a row of 2048 steps fills one wave: rows are cut
// into tiles of 32 chunks (2048 steps), the tiles of a channel's rows stand in one line, and a
// workgroup takes four of them at a time, a tile per wave; the recurrence starts anew where a tile
// is the first of its row.  (4 x 2048 rows of 5000 steps, forward and backward: 254 us with a row per
// workgroup, 161 us so; 4096 single rows of 32768 steps 419 and 420.)
#include "common.hpp"
#include "cema_pow.hpp"

#include <initializer_list>
#include <type_traits>

namespace mega {
namespace {

constexpr int kT = 64;         // steps per chunk
constexpr int kThreads = 256;  // four waves
constexpr int kWaves = kThreads / kWave;
constexpr int kHP = 36;        // floats per state row in LDS: 32 + 4 (16-byte rows 8 lanes apart hit 32 banks)
constexpr int kSubs = 16;      // sub-segments of the chunk scan (one per 16 threads)

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx16 mfma_bf16(u32x4 a, u32x4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
template <int DT>
__device__ __forceinline__ floatx16 mfma16(u32x4 a, u32x4 b, floatx16 c) {
  if constexpr (DT == MEGA_BF16) return mfma_bf16(a, b, c);
  else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// 8 floats -> packed bf16 high parts and packed bf16 residuals
__device__ __forceinline__ void split8(const float* v, u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t h = pack_bf16x2(v[2 * e], v[2 * e + 1]);
    const float r0 = v[2 * e] - __uint_as_float(h << 16);
    const float r1 = v[2 * e + 1] - __uint_as_float(h & 0xffff0000u);
    hi[e] = h;
    lo[e] = pack_bf16x2(r0, r1);
  }
}
// the same in float16: 22 significant bits of values of some 2^12 (far below them the residuals end), with `third` 33
// Each piece is taken off as it stands in the packed word, hidden from the optimiser: left alone it packs by one
// instruction and takes the residual from another's result, and the two round ties apart.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t take_f16(float& a, float& b) {
  uint32_t w = __builtin_bit_cast(uint32_t, f16x2{static_cast<_Float16>(a), static_cast<_Float16>(b)});
  asm volatile("" : "+v"(w));
  const f16x2 h = __builtin_bit_cast(f16x2, w);
  a -= static_cast<float>(h[0]);
  b -= static_cast<float>(h[1]);
  return w;
}
template <bool THIRD>
__device__ __forceinline__ void split8_f16(const float* v, u32x4& hi, u32x4& lo, u32x4& third) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float a = v[2 * e], b = v[2 * e + 1];
    hi[e] = take_f16(a, b);
    lo[e] = take_f16(a, b);
    if (THIRD) third[e] = take_f16(a, b);
  }
}
// ... and what is left of them behind that: 24 significant bits in three pieces
__device__ __forceinline__ u32x4 split8_third(const float* v, u32x4 hi, u32x4 lo) {
  u32x4 third;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    third[e] = pack_bf16x2((v[2 * e] - __uint_as_float(hi[e] << 16)) - __uint_as_float(lo[e] << 16),
                           (v[2 * e + 1] - __uint_as_float(hi[e] & 0xffff0000u)) - __uint_as_float(lo[e] & 0xffff0000u));
  return third;
}
// The operand blocks of a channel's powers are written by the threads that form the powers, thread (n, a) those of mode n
// with four exponents.  Four columns 4 quad .. 4 quad + 3 of row m of four blocks (rows m, k-steps of 16 columns):
template <bool THIRD>
__device__ __forceinline__ void put_columns(u32x4 (*blocks)[2][kWave], u32x4 (*third)[kWave], int m, int quad, const float* v) {
  const int blk = quad >> 2, ln = m + 32 * ((quad >> 1) & 1), half = quad & 1;
  uint2 hi, lo, rest;
  uint32_t *const h = &hi.x, *const l = &lo.x, *const t = &rest.x;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    h[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
    const float r0 = v[2 * e] - __uint_as_float(h[e] << 16), r1 = v[2 * e + 1] - __uint_as_float(h[e] & 0xffff0000u);
    l[e] = pack_bf16x2(r0, r1);
    if (THIRD) t[e] = pack_bf16x2(r0 - __uint_as_float(l[e] << 16), r1 - __uint_as_float(l[e] & 0xffff0000u));
  }
  reinterpret_cast<uint2*>(&blocks[blk][0][ln])[half] = hi;
  reinterpret_cast<uint2*>(&blocks[blk][1][ln])[half] = lo;
  if (THIRD) reinterpret_cast<uint2*>(&third[blk][ln])[half] = rest;
}
// ... and the columns 2 n, 2 n + 1 of row i of four blocks (row tile of 32, k-step of 16 columns)
__device__ __forceinline__ void put_pair(u32x4 (*blocks)[2][kWave], int n, int i, float a, float b) {
  const int blk = 2 * (i >> 5) + (n >> 3), ln = (i & 31) + 32 * ((n >> 2) & 1);
  const uint32_t h = pack_bf16x2(a, b);
  reinterpret_cast<uint32_t*>(&blocks[blk][0][ln])[n & 3] = h;
  reinterpret_cast<uint32_t*>(&blocks[blk][1][ln])[n & 3] = pack_bf16x2(a - __uint_as_float(h << 16), b - __uint_as_float(h & 0xffff0000u));
}
// ... as they are, two words of four floats a lane where put_pair has two pieces of eight
__device__ __forceinline__ void put_pair_f32(u32x4 (*blocks)[2][kWave], int n, int i, float a, float b) {
  const int blk = 2 * (i >> 5) + (n >> 3), ln = (i & 31) + 32 * ((n >> 2) & 1);
  reinterpret_cast<float2*>(&blocks[blk][(n >> 1) & 1][ln])[n & 1] = make_float2(a, b);
}
// acc += A B over 16 columns: lane (r, g) holds row (column) r and the values 8 g .. + 7 of both
__device__ __forceinline__ floatx16 mma_f32(const u32x4* a, const float* b, floatx16 acc) {
#pragma unroll
  for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[e >> 2][e & 3]), b[e], acc, 0, 0, 0);
  return acc;
}
// Third pieces of k[0 .. 63] for the Toeplitz blocks, whose lanes read eight consecutive lags each: one table of the
// lags in the blocks' order, zeros at negative ones, and a second one that starts an element later, so that every
// lane reads whole words.
constexpr int kThirdLags = 96;
typedef uint16_t ThirdTable[2][kThirdLags];
// The first two pieces of the lags in such tables (in place of whole operand blocks).
__device__ __forceinline__ void fill_pieces(ThirdTable& hi, ThirdTable& lo, const float* k, int tid) {
  if (tid < 2 * kThirdLags) {
    const int lag = kT - 1 - (tid < kThirdLags ? tid : tid - kThirdLags + 1);
    const float v = lag >= 0 && lag < kT ? k[lag] : 0.f;
    const uint32_t h = pack_bf16x2(v, 0.f);
    hi[0][tid] = static_cast<uint16_t>(h);
    lo[0][tid] = static_cast<uint16_t>(pack_bf16x2(v - __uint_as_float(h << 16), 0.f));
  }
}
template <bool DOWN>  // index i: lag 63 - i, else i - 31
__device__ __forceinline__ void fill_thirds(ThirdTable& t, const float* k, int tid) {
  if (tid < 2 * kThirdLags) {
    const int i = tid < kThirdLags ? tid : tid - kThirdLags + 1, lag = DOWN ? kT - 1 - i : i - 31;
    const float v = lag >= 0 && lag < kT ? k[lag] : 0.f;
    const float r = v - __uint_as_float(pack_bf16x2(v, 0.f) << 16);
    t[0][tid] = static_cast<uint16_t>(pack_bf16x2(r - __uint_as_float(pack_bf16x2(r, 0.f) << 16), 0.f));
  }
}
// elements i .. i + 7
__device__ __forceinline__ u32x4 read_thirds(const ThirdTable& t, int i) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(t[i & 1]) + (i >> 1);
  return u32x4{w[0], w[1], w[2], w[3]};
}
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// a <-> b between the two halves of the wave (v_permlane32_swap_b32): afterwards
// the low half holds (its own a, the high half's a), the high half (the low
// half's b, its own b).  Written as inline assembly: the compiler's builtin
// returned the first result for both outputs here.  The compiler does not
// see what the assembly reads, so it guards none of the hazards: the s_nop
// covers the wait states after a vector write of an operand, and operands
// that come out of an MFMA must first pass through an ordinary vector
// instruction (`settle`), which the compiler does schedule behind the MFMA.
__device__ __forceinline__ void half_swap(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void half_swap(uint32_t& a, uint32_t& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
// two floats -> one word of two 16-bit elements of type DT
template <int DT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if (DT == MEGA_BF16) return pack_bf16x2(lo, hi);
  return static_cast<uint32_t>(float_to_f16_bits(lo)) | (static_cast<uint32_t>(float_to_f16_bits(hi)) << 16);
}
// An accumulator tile (lane <-> chunk, register 4 qd + e <-> step 8 qd + 4 g + e of a 32-step
// row tile) rounded to 16 bits and regrouped so that the lane of half g holds the 8
// consecutive steps 16 pr + 8 g .. + 7: the rounding is the ordinary vector instruction
// that separates the MFMA from the swaps (see half_swap).
template <int DT>
__device__ __forceinline__ uint4 octet_of(const floatx16& acc, int pr) {
  uint32_t a0 = pack2<DT>(acc[8 * pr], acc[8 * pr + 1]), a1 = pack2<DT>(acc[8 * pr + 2], acc[8 * pr + 3]);
  uint32_t b0 = pack2<DT>(acc[8 * pr + 4], acc[8 * pr + 5]), b1 = pack2<DT>(acc[8 * pr + 6], acc[8 * pr + 7]);
  half_swap(a0, b0);
  half_swap(a1, b1);
  return make_uint4(a0, a1, b0, b1);
}
// Makes a lane-derived value opaque to the optimiser.  Offsets, masks and converted indices
// depend only on the lane, not on the row: left alone they are hoisted out of the persistent
// row loop into hundreds of spilled registers; recomputing them per item is cheaper.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
// 1.0f the optimiser cannot see through
__device__ __forceinline__ float opaque_one() {
  float one = 1.0f;
  asm volatile("" : "+v"(one));
  return one;
}

// How the rows of a launch lie in memory.
//   kWhole   every row starts on a 16-byte boundary and its length is a multiple of 8
//   kShifted rows of another length in a tensor that starts on one: a row is taken from the
//            16-byte boundary at or in front of its start, the up to seven steps in front of it
//            as zeros -- with no state before them the recurrence does not see them -- so that
//            every access but those at the two ends is aligned
//   kAny     a carried state, or a tensor that starts or ends off a boundary: the same 16-byte accesses at
//            any element's address (which cost more: 4 x 2048 rows of 5001 steps forward and backward
//            258 us so, 190 shifted; 161 for 5000 steps, whole rows without third pieces)
enum { kWhole = 0, kShifted = 1, kAny = 2 };
// The lengths of the last two came to these kernels from a float32 convolution and keep its precision: P, Pg and K have
// a third bf16 piece, products of two split factors keep their lo * lo term, and the state after the last step is
// summed with powers that are evaluated directly.  Relative errors against 64 bits (2-norm, the largest over 121 .. 32767
// steps) at the layer's initial decays, the convolution's, these kernels' and in brackets two pieces':
//   dx before rounding (y alike)  4.0e-6                   4.7e-7 (2.7e-6)
//   state after the last step     2.6e-7                   2.1e-7 (1.5e-6; of float16 rows 2.2e-6)
//   dalpha, ddelta, dtheta        9.7e-7, 1.2e-6, 1.7e-6   3.4e-7, 6.3e-7, 1.4e-6 (5.3e-7, 1.0e-6, 1.8e-6; 3.0e-6, 3.4e-6, 4.0e-6)
// With decays ten and a hundred times slower, where the float32 coefficients bound every path: dx 4.8e-6 / 3.1e-6 and
// 7.5e-5 both (3.3e-6 instead of 4.0e-6 in rows of 121 steps).  The pieces cost 13 %: 4 x 2048 rows of 5001 steps forward and
// backward 168 -> 190 us.
template <int ROWS> constexpr bool kFine = ROWS != kWhole;
typedef u32x4 u32x4_any __attribute__((aligned(2)));
// of the 16-bit steps elem .. elem + 7 those of lo .. hi - 1, zeros for the others
__device__ __forceinline__ u32x4 keep_steps(u32x4 v, int elem, int lo, int hi) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (elem + e < lo || elem + e >= hi) v[e >> 1] &= e & 1 ? 0x0000ffffu : 0xffff0000u;
  return v;
}
// steps elem .. elem + 7 of a tile of which lo .. hi - 1 exist, zeros elsewhere
template <int ROWS>
__device__ __forceinline__ u32x4 load8_16(const uint16_t* tile, int elem, int lo, int hi) {
  const uint16_t* src = tile + elem;
  u32x4 v = {0u, 0u, 0u, 0u};
  if (ROWS != kAny) {  // (kShifted: a piece with one of the steps is inside the tensor)
    if (elem < hi) v = *reinterpret_cast<const u32x4*>(src);
  } else if (elem + 8 <= hi) {
    v = *reinterpret_cast<const u32x4_any*>(src);
  } else if (elem < hi) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (elem + e < hi) v[e >> 1] |= static_cast<uint32_t>(src[e]) << (16 * (e & 1));
  }
  return v;
}
template <int ROWS>
__device__ __forceinline__ void store8_16(uint16_t* tile, int elem, int lo, int hi, uint4 v) {
  uint16_t* dst = tile + elem;
  if ((ROWS != kShifted || elem >= lo) && elem + 8 <= hi) {
    if (ROWS == kAny) *reinterpret_cast<u32x4_any*>(dst) = u32x4{v.x, v.y, v.z, v.w};
    else *reinterpret_cast<uint4*>(dst) = v;
  } else if (ROWS != kWhole && elem < hi) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (elem + e >= lo && elem + e < hi) dst[e] = static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
  }
}

// Eight consecutive steps of a row as a matrix operand: XP bf16 pieces whose sum
// is the data exactly (bf16: the data itself; fp16: two pieces).
template <int DT> struct XOp;
template <> struct XOp<MEGA_BF16> {
  static constexpr int XP = 1;
  u32x4 pc[1];
  template <int ROWS>
  __device__ __forceinline__ void load(const void* tile, int elem, int lo, int hi) {
    pc[0] = load8_16<ROWS>(static_cast<const uint16_t*>(tile), elem, lo, hi);
  }
  __device__ __forceinline__ void keep(int elem, int lo, int hi) { pc[0] = keep_steps(pc[0], elem, lo, hi); }
  __device__ __forceinline__ void values(float* v) const {
    unpack8<MEGA_BF16>(make_uint4(pc[0][0], pc[0][1], pc[0][2], pc[0][3]), v);
  }
};
template <> struct XOp<MEGA_F16> {
  static constexpr int XP = 2;
  u32x4 pc[2];
  template <int ROWS>
  __device__ __forceinline__ void load(const void* tile, int elem, int lo, int hi) {
    float v[8];
    const u32x4 raw = load8_16<ROWS>(static_cast<const uint16_t*>(tile), elem, lo, hi);
    unpack8<MEGA_F16>(make_uint4(raw[0], raw[1], raw[2], raw[3]), v);
    split8(v, pc[0], pc[1]);
  }
  __device__ __forceinline__ void keep(int elem, int lo, int hi) {
    pc[0] = keep_steps(pc[0], elem, lo, hi);
    pc[1] = keep_steps(pc[1], elem, lo, hi);
  }
  __device__ __forceinline__ void values(float* v) const {
    float a[8], b[8];
    unpack8<MEGA_BF16>(make_uint4(pc[0][0], pc[0][1], pc[0][2], pc[0][3]), a);
    unpack8<MEGA_BF16>(make_uint4(pc[1][0], pc[1][1], pc[1][2], pc[1][3]), b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = a[e] + b[e];
  }
};

// float32 rows: the two leading bf16 pieces (16 significant bits, what the parameter matrices
// carry as well); the rest, 2^-17 of a value, is left out
template <> struct XOp<MEGA_F32> {
  static constexpr int XP = 2;
  u32x4 pc[2];
  template <int ROWS>
  __device__ __forceinline__ void load(const void* tile, int elem, int lo, int hi) {
    static_assert(ROWS == kWhole, "float32 rows are aligned");
    (void)lo;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (elem < hi) {
      const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(tile) + elem);
      a = src[0];
      b = src[1];
    }
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    split8(v, pc[0], pc[1]);
  }
};

// float32 rows of the other layouts: all three pieces, 24 significant bits, as P and K carry.  The state's share of the outputs (Q H, and
// in the backward Qd R) is a product of float32 matrix instructions, whose operands lie where the others' two pieces do: in two
// pieces each it was good to 2^-18, which is most of what y and dx are off where memories are long.  Against 64 bits on the same
// float32 coefficients, all of 64 channels in the 2-norm / the channel that is furthest off, 121 and 4097 steps with and without a mean: at the
// initial decays 1.7e-7 / 2.9e-6 (in pieces 4.8e-7 / 3.1e-5), at ten times slower ones 2.1e-7 / 6.6e-7 (1.8e-6 / 1.2e-5), at a hundred times
// slower 4.6e-7 / 7.2e-7 (4.1e-6 / 6.2e-6).  It costs 3 to 16 %: forward, 1024 rows of 51151 steps 123 -> 128 us, 4096 of 1531 45 -> 51, of 201 41 -> 48;
// forward and backward, 2048 of 22185 956 -> 985, 4 x 2048 of 5001 948 -> 987.  (Through a float32 kernel row and float32 transforms, as
// these lengths went before, 2181, 204, 66, 1717 and 1184; y and dx 2.6e-6 - 3.4e-6 and 2e-5 - 1.4e-4 at the initial decays, in no channel more
// than a tenth nearer at slower ones; gradients of the parameters that are sums of terms of one sign, as rows with a mean have, 0.8e-7 - 4.3e-7 there and
// 1.1e-7 - 5.2e-7 here, the others nowhere nearer.)  The forward of kShifted keeps two registers of ONE in scratch, the others' long walk one.
struct XOpWide {
  static constexpr int XP = 3;
  u32x4 pc[3];
  template <int ROWS>
  __device__ __forceinline__ void load(const void* tile, int elem, int lo, int hi) {
    (void)lo;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef f32x4 f32x4_any __attribute__((aligned(4)));
    const float* src = static_cast<const float*>(tile) + elem;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (ROWS == kShifted ? elem < hi : elem + 8 <= hi) {  // (kShifted: a piece with one of the steps is inside the tensor)
      const f32x4 a = *reinterpret_cast<const f32x4_any*>(src), b = *reinterpret_cast<const f32x4_any*>(src + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
    } else if (elem < hi) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (elem + e < hi) v[e] = src[e];
    }
    split8(v, pc[0], pc[1]);
    pc[2] = split8_third(v, pc[0], pc[1]);
  }
  __device__ __forceinline__ void keep(int elem, int lo, int hi) {
#pragma unroll
    for (int i = 0; i < 3; ++i) pc[i] = keep_steps(pc[i], elem, lo, hi);
  }
};
template <int DT, bool FINE>
using XRow = typename std::conditional<DT == MEGA_F32 && FINE, XOpWide, XOp<DT>>::type;

// acc += (A_hi + A_lo) * x, without FINE the lo * lo term of a two-piece x left out
template <int XP, bool FINE = false>
__device__ __forceinline__ floatx16 mma_split(const u32x4* a, const u32x4* x, floatx16 acc) {
  acc = mfma_bf16(a[0], x[0], acc);
  acc = mfma_bf16(a[1], x[0], acc);
  if (XP >= 2) acc = mfma_bf16(a[0], x[1], acc);
  if (XP >= 2 && FINE) acc = mfma_bf16(a[1], x[1], acc);
  if (XP == 3) acc = mfma_bf16(a[0], x[2], acc);
  return acc;
}

// Operand blocks of the forward kernel (each 64 lanes x 8 values, two pieces; Q of WIDE kernels: 64 lanes x 8 floats):
//   0..3   P, k-step s:            rows m, steps j = 16 s + 8 g + e
//   4..7   K by offset o = 16 (b - 5): rows r, lag = o + r - 8 g - e (zero where negative)
//   8..11  Q, (row tile it, k-step s2): rows i = 32 it + r, state columns m = 16 s2 + 8 g + e
constexpr int kFwdBlocks = 12;

// ONE: a workgroup takes one item (at most four tiles) and ends.  Setting up its channel is a chain of short phases
// with a barrier between them, so what counts is how many workgroups share a compute unit: without the blocks of K,
// whose lags are read out of a table of 96 instead, four fit (128 registers a lane: nothing is loaded ahead).  Half of the
// rest is the issue of vector instructions, 500 a wave: the threads that form the powers write the operand blocks of P and
// Q themselves (no table between), and a wave without a tile does nothing but its share of the set-up.  Rows of 2048
// float32 steps of 1024 channels: 15.8 us three to a compute unit with a launch for the coefficients, 11.2 four, 9.9 so;
// 4096 channels of 1531 bfloat16 steps with their last state 51 -> 34, of 2048 31 -> 25, of 4088 54 -> 35.
template <bool ONE>
struct FwdSmemOf {
  static constexpr int NC = kWaves * 32;       // chunks resident
  static constexpr int kBlocks = ONE ? 8 : kFwdBlocks, kQ = kBlocks - 4;
  union {
    float klocal[kT];                          // k[0 .. 63] (+ omega at lag 0), while a row is set up
    cf sub_end[kWaves * 3][16];                // local end state of each sub-segment but a wave's last
  };
  float pn[16];
  cf gn[16];
  cf wave_end[ONE ? 1 : 2][kWaves][16];        // local end state of each wave's 4 sub-segments, by item parity
  float wave_cin[kWaves][32];                  // state in front of each wave's first chunk
  cf carry[2][16];
  cf pw[12][16];                               // q^(4 k), q^(16 k) (k < 4), q, q^64, q^(64 CPS), q^(256 CPS)
  u32x4 aop[kBlocks][2][kWave];                // ONE: P, then Q
  // row 1 + c: state after chunk c of the segment
  float H[(NC + 1) * kHP];
};
struct FwdSmem : FwdSmemOf<false> {};
struct FwdSmemFine : FwdSmem {
  u32x4 third[4][kWave];  // third pieces of P
  alignas(4) ThirdTable kthird;
};
struct FwdSmemOne : FwdSmemOf<true> {
  cf lq[16];
  alignas(4) ThirdTable kpiece[2];
};
struct FwdSmemOneFine : FwdSmemOne {
  alignas(4) ThirdTable kthird;  // (third pieces of P: in registers)
};
static_assert(sizeof(u32x4) * 4 * kWave <= sizeof(float) * (kWaves * 32 + 1) * kHP, "the third pieces of P pass through the state buffer");
static_assert(3 * sizeof(FwdSmemFine) <= 160 * 1024, "three workgroups per compute unit");
static_assert(4 * sizeof(FwdSmemOneFine) <= 160 * 1024, "four workgroups per compute unit");

// The channels' coefficients: p, log q, gamma in float32, or, where `alpha` is not null, the layer's raw parameters of element type
// `dtype`, turned into them as mega_cema_layer_coeffs_fwd does.
struct Coeffs {
  const float* p;
  const cf *log_q, *gamma;
  const float* omega;
  const void *alpha, *delta, *theta, *raw_gamma, *raw_omega;
  int dtype;
};
__device__ __forceinline__ float load_any(const void* base, int dtype, int64_t i) {
  if (dtype == MEGA_F32) return static_cast<const float*>(base)[i];
  const uint16_t v = static_cast<const uint16_t*>(base)[i];
  return dtype == MEGA_BF16 ? bf16_bits_to_float(v) : f16_bits_to_float(v);
}

// The rows of a launch: groups of `nb` rows of one channel (d = group % D), each a line of tiles.
struct Lines {
  int B, D, nb, groups;  // groups = D ceil(B / nb)
  int tpr;               // tiles per row
  int64_t L;             // steps of a row
  __device__ __forceinline__ int first_row(int group) const { return group / D * nb; }
  __device__ __forceinline__ int tiles(int group) const { return min(nb, B - first_row(group)) * tpr; }
};
// A tile of a group's line: which row, where in it.  Stepping from one of a wave's tiles to the
// next needs no division; lanes address inside it by 32-bit offsets from a base that the wave shares.
struct Tile {
  int64_t row;  // b D + d
  int64_t base; // element where the tile starts (kShifted: a row's first one, up to seven in front of the row)
  int lo, hi;   // its steps lo .. hi - 1 exist (hi = 0: no such tile)
  int t;        // number in the line
  int chunk0;   // first chunk inside the row
  int nc;       // chunks of the row in it
  // whether the tile's data have steps of another row among them (kShifted)
  __device__ __forceinline__ bool cut() const { return lo > 0 || hi < 32 * kT; }
};
template <int ROWS>
__device__ __forceinline__ void tile_row(const Lines& ln, Tile& w, int tiles) {
  const int64_t start = w.row * ln.L;
  const int front = ROWS == kShifted ? static_cast<int>(start & 7) : 0;
  const int64_t behind = static_cast<int64_t>(w.chunk0) * kT - front;  // steps of the row in front of the tile
  w.base = start + behind;
  w.lo = ROWS == kShifted && w.chunk0 == 0 ? front : 0;
  w.hi = w.t >= 0 && w.t < tiles ? static_cast<int>(max(int64_t{0}, min(ln.L - behind, int64_t{32 * kT}))) : 0;
  w.nc = (w.hi + kT - 1) / kT;
}
template <int ROWS>
__device__ __forceinline__ Tile tile_at(const Lines& ln, int group, int t) {
  Tile w;
  const bool on = group < ln.groups;
  const int b = t / ln.tpr;
  w.row = on ? static_cast<int64_t>(ln.first_row(group) + b) * ln.D + group % ln.D : 0;
  w.t = t;
  w.chunk0 = (t - b * ln.tpr) * 32;
  tile_row<ROWS>(ln, w, on ? ln.tiles(group) : 0);
  return w;
}
template <int ROWS>
__device__ __forceinline__ void tile_forward(const Lines& ln, Tile& w, int tiles) {
  w.t += kWaves;
  w.chunk0 += 32 * kWaves;
  while (w.chunk0 >= 32 * ln.tpr) {
    w.chunk0 -= 32 * ln.tpr;
    w.row += ln.D;
  }
  tile_row<ROWS>(ln, w, tiles);
}
template <int ROWS>
__device__ __forceinline__ void tile_backward(const Lines& ln, Tile& w, int tiles) {
  w.t -= kWaves;
  w.chunk0 -= 32 * kWaves;
  while (w.chunk0 < 0) {
    w.chunk0 += 32 * ln.tpr;
    w.row -= ln.D;
  }
  tile_row<ROWS>(ln, w, tiles);
}

// LDS traffic of one wave is processed in order: a wave that has written rows
// and waits for its own LDS operations can read what its other lanes wrote.
__device__ __forceinline__ void wave_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int DT, int ROWS, bool ONE>
__global__ __launch_bounds__(kThreads, ONE ? 4 : 3) void cema_scan_fwd_kernel(
    const void* __restrict__ x, void* __restrict__ y, const Coeffs co,
    const cf* __restrict__ h0, cf* __restrict__ h_last, const Lines ln, int N) {
  constexpr bool FINE = kFine<ROWS>;
  using Smem = typename std::conditional<ONE, typename std::conditional<FINE, FwdSmemOneFine, FwdSmemOne>::type,
                                         typename std::conditional<FINE, FwdSmemFine, FwdSmem>::type>::type;
  constexpr bool WIDE = FINE && DT == MEGA_F32;  // Q and the states as float32 operands
  using Op = XRow<DT, FINE>;
  constexpr int NC = Smem::NC, CPS = NC / kSubs, XP = Op::XP;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Smem& sm = *reinterpret_cast<Smem*>(smem_raw);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane >> 5, r = lane & 31;
  // scan roles: mode sn; sub-segment sa = 4 wave + sl of CPS chunks, inside the wave's own tiles
  const int sn = tid & 15, sa = tid >> 4, sl = sa & 3;

  // The workgroup walks (group, four tiles) items: groups blockIdx.x, + gridDim.x, ..., the tiles
  // of a group in line.  The x tile of the next item and the parameters of the next group are
  // requested ahead.
  auto load_tile = [&](Op (&t)[4], const Tile& w) {
    const typename Elem<DT>::type* xrow = static_cast<const typename Elem<DT>::type*>(x) + w.base;
    const int id = opaque(lane), at = (id & 31) * kT + 8 * (id >> 5);
#pragma unroll
    for (int s = 0; s < 4; ++s) t[s].template load<ROWS>(xrow, at + 16 * s, w.lo, w.hi);
  };
  struct RowParams {
    cf lq, gv;
    float pv, w;
  };
  auto fetch_params = [&](int group) {
    RowParams rp{cf{0.f, 0.f}, cf{0.f, 0.f}, 0.f, 0.f};
    if (group < ln.groups) {
      const int d = group % ln.D;
      if (sn < N && co.p != nullptr) {
        const int i = d * N + sn;
        rp.lq = co.log_q[i];
        rp.gv = co.gamma[i];
        rp.pv = co.p[i];
      }
      if (co.raw_omega != nullptr) rp.w = load_any(co.raw_omega, co.dtype, d);
      else if (co.omega != nullptr) rp.w = co.omega[d];
    }
    return rp;
  };

  u32x4 (*passed)[kWave] = reinterpret_cast<u32x4(*)[kWave]>(sm.H);  // ONE and FINE, setup only: third pieces of P
  u32x4 third_p[4];
  cf qT{0.f, 0.f}, qS{0.f, 0.f}, qW{0.f, 0.f};
  int cur = 0, par = 0;
  RowParams rp = fetch_params(blockIdx.x);

  // tables, operand blocks and scan multipliers of a row's channel, from the
  // parameters fetched ahead; then the next row's parameters are requested
  auto setup_row = [&](int group) {
    // the few powers that are evaluated directly (phase reduced in float64): 12 per mode;
    // everything else is a product of two of them and a short chain of multiplications
    if constexpr (ONE) {
      // one lane per mode forms or fetches its coefficients (238 vector instructions of 1100 when every lane did)
      if (tid < 16) {
        if (co.alpha != nullptr && tid < N) {
          const int d = group % ln.D, i = d * N + tid;
          const CemaCoeffs c = cema_coeffs(load_any(co.alpha, co.dtype, i), load_any(co.delta, co.dtype, i), load_any(co.theta, co.dtype, d), tid, N);
          rp.lq = cf{c.log_rho, c.phi};
          rp.gv = cf{load_any(co.raw_gamma, co.dtype, 2 * i) * c.scale, load_any(co.raw_gamma, co.dtype, 2 * i + 1) * c.scale};
          rp.pv = c.p;
        }
        sm.lq[tid] = rp.lq;
        sm.pn[tid] = rp.pv;
        sm.gn[tid] = rp.gv;
      }
      __syncthreads();
      rp.lq = sm.lq[sn];
      rp.pv = sm.pn[sn];
      rp.gv = sm.gn[sn];
    }
    cf direct{0.f, 0.f};
    if (tid < 12 * 16 && sn < N) {
      const int k = tid >> 4;
      const int e = k < 4 ? 4 * k
                          : (k < 8 ? 16 * (k - 4) : (k == 8 ? 1 : (k == 9 ? kT : (k == 10 ? kT * CPS : 4 * kT * CPS))));
      direct = qpow(rp.lq.x, rp.lq.y, e);
    }
    if constexpr (!ONE) __syncthreads();  // every wave is done with the previous row's tables and carried state
    if (tid < 12 * 16) sm.pw[tid >> 4][sn] = direct;
    if (!ONE && tid < 16) {
      sm.pn[tid] = rp.pv;
      sm.gn[tid] = rp.gv;
    }
    cur = 0;
    __syncthreads();
    {
      // q^(4 sa + e), e < 4, and this mode's share of k at those lags, summed over the 16 modes (the 16 lanes of a row):
      // the skip term omega x rides on k[0].  They are this thread's columns of P, and with q^(4 sa + 4) its rows of Q.
      cf v[5];
      v[0] = cmul(sm.pw[sa & 3][sn], sm.pw[4 + (sa >> 2)][sn]);
      v[4] = sa == 15 ? sm.pw[9][sn] : cmul(sm.pw[(sa + 1) & 3][sn], sm.pw[4 + (((sa + 1) >> 2) & 3)][sn]);
      const cf q1 = sm.pw[8][sn];
      const cf c{rp.pv * rp.gv.x, rp.pv * rp.gv.y};
      const int id = opaque(tid), n = id & 15, quad = id >> 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e > 0) v[e] = cmul(v[e - 1], q1);
        const float kl = group_sum<16>(c.x * v[e].x - c.y * v[e].y);
        if (sn == 0) sm.klocal[4 * sa + e] = (sa == 0 && e == 0) ? kl + rp.w : kl;
      }
      u32x4 (*third)[kWave] = nullptr;
      if constexpr (FINE && ONE) third = passed;
      else if constexpr (FINE) third = sm.third;
#pragma unroll
      for (int part = 0; part < 2; ++part) {  // step j has the exponent 63 - j
        float pv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) pv[e] = rp.pv * (part ? v[3 - e].y : v[3 - e].x);
        put_columns<FINE>(sm.aop, third, 2 * n + part, 15 - quad, pv);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const cf w = cmul(rp.gv, v[e + 1]);
        if constexpr (WIDE) put_pair_f32(sm.aop + Smem::kQ, n, 4 * quad + e, w.x, -w.y);
        else put_pair(sm.aop + Smem::kQ, n, 4 * quad + e, w.x, -w.y);
      }
      qT = sm.pw[9][sn];
      qS = sm.pw[10][sn];
      qW = sm.pw[11][sn];
    }
    RowParams next_rp{};
    if constexpr (!ONE) next_rp = fetch_params(group + static_cast<int>(gridDim.x));
    __syncthreads();
    if constexpr (!ONE) {
      const int b = wave, id = opaque(lane), rr = id & 31, gg = id >> 5, o = 16 * (b - 1);
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int lag = o + rr - 8 * gg - e;
        const float kv = sm.klocal[lag >= 0 ? lag : 0];  // read, then masked: no branch around the load
        v[e] = lag >= 0 ? kv : 0.f;
      }
      u32x4 hi, lo;
      split8(v, hi, lo);
      sm.aop[4 + b][0][lane] = hi;
      sm.aop[4 + b][1][lane] = lo;
    }
    if constexpr (ONE) fill_pieces(sm.kpiece[0], sm.kpiece[1], sm.klocal, tid);
    if constexpr (FINE) fill_thirds<true>(sm.kthird, sm.klocal, tid);
    if constexpr (FINE && ONE)
#pragma unroll
      for (int s = 0; s < 4; ++s) third_p[s] = passed[s][lane];
    __syncthreads();
    rp = next_rp;
  };
  // The operand blocks stay in LDS and are read where a phase needs them (P for the local
  // states, K and Q for the outputs): held in registers across the whole item they cost
  // 96 registers and spill.
  auto load_block = [&](int b, u32x4* dst) {
    dst[0] = sm.aop[b][0][lane];
    dst[1] = sm.aop[b][1][lane];
  };

  // One item.  Its x tile was requested by the previous item (or the prologue); everything that
  // reads it -- the local states and the K X part of the outputs -- comes first, then the
  // same registers are reloaded with the next item's tile while the scan and the state part of
  // the outputs run.
  Op xb[4];
  Tile cur_tile = tile_at<ROWS>(ln, blockIdx.x, wave);  // this wave's tile of the item
  auto item = [&](int group, int t0, int tiles) {
    if (t0 == 0) setup_row(group);
    const Tile w = cur_tile;
    typename Elem<DT>::type* yrow = static_cast<typename Elem<DT>::type*>(y) + w.base;
    const int c0 = wave * 32;
    if constexpr (ROWS == kShifted)
      if (w.cut()) {
        const int id = opaque(lane), at = (id & 31) * kT + 8 * (id >> 5);
#pragma unroll
        for (int s = 0; s < 4; ++s) xb[s].keep(at + 16 * s, w.lo, w.hi);
      }
    // a wave behind the line's end only keeps the barriers (of several items it is the last that has any: not worth the registers)
    const bool on = w.nc > 0, runs = !ONE || on, ends = on && h_last != nullptr && w.base + w.hi == (w.row + 1) * ln.L;
    const int cl = w.nc - 1, rem = w.hi - cl * kT;  // the tile's last chunk, 1 .. 64 steps in it
    // those steps, for the state after them: a lane each
    auto load_end = [&] { return ends && lane < rem ? Elem<DT>::load(static_cast<const typename Elem<DT>::type*>(x) + w.base + cl * kT + lane) : 0.f; };
    float x_end = 0.f;
    if constexpr (ONE) x_end = load_end();
    // the state in front of the wave's row, where that starts among the item's tiles
    const int k = w.chunk0 / 32;
    auto carried = [&] { return h0 != nullptr && k <= wave && w.nc > 0 && sn < N ? h0[w.row * N + sn] : cf{0.f, 0.f}; };
    cf h_in{0.f, 0.f};
    if constexpr (!ONE) h_in = carried();
    floatx16 yacc[2];
    // ---- local states S = P X, into this wave's own rows of the state buffer ----------
    if (runs) {
      u32x4 P[4][2];
#pragma unroll
      for (int s = 0; s < 4; ++s) load_block(s, P[s]);
      if (on) {
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          acc = mma_split<XP, FINE>(P[s], xb[s].pc, acc);
          if constexpr (FINE && ONE) acc = mfma_bf16(third_p[s], xb[s].pc[0], acc);
          else if constexpr (FINE) acc = mfma_bf16(sm.third[s][lane], xb[s].pc[0], acc);
        }
        float* dst = sm.H + (1 + c0 + r) * kHP + 4 * g;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          *reinterpret_cast<float4*>(dst + 8 * qd) =
              make_float4(acc[4 * qd], acc[4 * qd + 1], acc[4 * qd + 2], acc[4 * qd + 3]);
      }
    }
    // ---- the within-chunk part of the outputs, K X (omega x included: K carries omega on
    //      its diagonal); the accumulators wait for the state part ------------------------
    if (runs) {
      u32x4 K[4][2];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if constexpr (ONE) {
#pragma unroll
          for (int h = 0; h < 2; ++h) K[b][h] = read_thirds(sm.kpiece[h], kT - 1 - 16 * (b - 1) - r + 8 * g);
        } else {
          load_block(4 + b, K[b]);
        }
      }
#pragma unroll
      for (int it = 0; it < 2; ++it) {
#pragma unroll
        for (int i = 0; i < 16; ++i) yacc[it][i] = 0.f;
        if (on) {
#pragma unroll
          for (int s = 0; s < 2 + 2 * it; ++s) {
            const int b = 1 + 2 * it - s;
            yacc[it] = mma_split<XP, FINE>(K[b], xb[s].pc, yacc[it]);
            // (block b: lags 16 (b - 1) + r - 8 g - e)
            if constexpr (FINE) yacc[it] = mfma_bf16(read_thirds(sm.kthird, kT - 1 - 16 * (b - 1) - r + 8 * g), xb[s].pc[0], yacc[it]);
          }
        }
      }
    }
    if constexpr (!ONE) {
      // (waited for here: asked for behind the requests of the next tile its wait was theirs too, in the middle of the scan.
      // With a scan of fewer operations that showed: float16, 4096 x 32768 160 -> 154 us, 155 with the longer scan;
      // 8 x 512 x 16384 77.5 -> 76.3, 76.1; bfloat16, 4096 x 32768 138 -> 134)
      asm volatile("" : "+v"(h_in.x), "+v"(h_in.y));
      if (t0 + kWaves < tiles) tile_forward<ROWS>(ln, cur_tile, tiles);
      else cur_tile = tile_at<ROWS>(ln, group + static_cast<int>(gridDim.x), wave);
      load_tile(xb, cur_tile);
    }
    wave_sync();
    // ---- scan over the chunks: a sub-segment per 16 lanes, the wave's four sub-segments are its
    //      own chunks; one workgroup barrier hands over the waves' ends ---------------------------
    //      (chunks behind the row's end need no mask: their X is zero, so their S is, and nothing takes
    //      up a state behind them; what a wave without a tile passes on nobody reads)
    float* const col = sm.H + (1 + sa * CPS) * kHP + 2 * sn;  // state column n of the sub-segment's rows
    float2 sv[CPS];                          // the sub-segment's local states, kept for the second pass
    cf h{0.f, 0.f};
    if (runs) {
#pragma unroll
      for (int i = 0; i < CPS; ++i) sv[i] = *reinterpret_cast<const float2*>(col + i * kHP);
#pragma unroll
      for (int i = 0; i < CPS; ++i) h = cfma(qT, h, cf{sv[i].x, sv[i].y});
      if (sl < 3) sm.sub_end[3 * wave + sl][sn] = h;
      wave_sync();
      if (sl == 3) {
        cf e = sm.sub_end[3 * wave][sn];
        e = cfma(qS, e, sm.sub_end[3 * wave + 1][sn]);
        e = cfma(qS, e, sm.sub_end[3 * wave + 2][sn]);
        sm.wave_end[par][wave][sn] = cfma(qS, e, h);
      }
    }
    lds_barrier();
    if (runs) {
      cf cin = ONE ? cf{0.f, 0.f} : sm.carry[cur][sn];
      // through the tiles in front of this wave's, from the first one of its row if that is among the
      // four (there the carried state enters)
      const int from = k <= wave ? wave - k : 0;
      if (k <= wave) cin = ONE ? carried() : h_in;
#pragma unroll
      for (int v = 0; v < kWaves - 1; ++v)
        if (v >= from && v < wave) cin = cfma(qW, cin, sm.wave_end[par][v][sn]);
      if (!ONE && sa == kSubs - 1) sm.carry[cur ^ 1][sn] = cfma(qW, cin, sm.wave_end[par][kWaves - 1][sn]);
      if (sl == 0) *reinterpret_cast<float2*>(sm.wave_cin[wave] + 2 * sn) = make_float2(cin.x, cin.y);
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const cf e = sm.sub_end[3 * wave + s][sn];
        if (s < sl) cin = cfma(qS, cin, e);
      }
      h = cin;
#pragma unroll
      for (int i = 0; i < CPS; ++i) {
        h = cfma(qT, h, cf{sv[i].x, sv[i].y});
        *reinterpret_cast<float2*>(col + i * kHP) = make_float2(h.x, h.y);
      }
    }
    wave_sync();
    // ---- the state part of the outputs, Q H[c-1], and the stores ------------------------------
    if (runs) {
      u32x4 Q[4][2];
      if constexpr (!WIDE)
#pragma unroll
        for (int b = 0; b < 4; ++b) load_block(Smem::kQ + b, Q[b]);
      if (on) {
        u32x4 hb[WIDE ? 1 : 2][2];
        float hv[2][8];
        // the state in front of chunk c0 + r: the previous row of the buffer, or, for the
        // wave's first chunk, what the scan left in wave_cin
        const float* hrow = r == 0 ? sm.wave_cin[wave] : sm.H + (c0 + r) * kHP;
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const float* src = hrow + 16 * s2 + 8 * g;
          const float4 u = *reinterpret_cast<const float4*>(src);
          const float4 u1 = *reinterpret_cast<const float4*>(src + 4);
          const float v[8] = {u.x, u.y, u.z, u.w, u1.x, u1.y, u1.z, u1.w};
          if constexpr (WIDE) {
#pragma unroll
            for (int e = 0; e < 8; ++e) hv[s2][e] = v[e];
          } else {
            split8(v, hb[s2][0], hb[s2][1]);
          }
        }
        const int id = opaque(lane), at = (id & 31) * kT, ag = id >> 5;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          floatx16 acc = yacc[it];
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            if constexpr (WIDE) {
              load_block(Smem::kQ + 2 * it + s2, Q[0]);
              acc = mma_f32(Q[0], hv[s2], acc);
            } else {
              acc = mma_split<2, FINE>(Q[2 * it + s2], hb[s2], acc);
            }
          }
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            if constexpr (DT == MEGA_F32) {
              // registers 8 pr + 4 h + e hold the steps 16 pr + 8 h + 4 g + e: two 16-byte stores
              // per lane, no exchange between the halves of the wave
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const int elem = at + 16 * (2 * it + pr) + 8 * h + 4 * ag;
                if (ROWS == kWhole ? elem < w.hi : ROWS == kShifted && elem >= w.lo && elem + 4 <= w.hi) {
                  *reinterpret_cast<float4*>(yrow + elem) = make_float4(acc[8 * pr + 4 * h], acc[8 * pr + 4 * h + 1],
                                                                        acc[8 * pr + 4 * h + 2], acc[8 * pr + 4 * h + 3]);
                } else if (ROWS != kWhole) {
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    if (elem + e >= w.lo && elem + e < w.hi) yrow[elem + e] = acc[8 * pr + 4 * h + e];
                }
              }
            } else {
              const uint4 oct = octet_of<DT>(acc, pr);
              store8_16<ROWS>(yrow, at + 16 * (2 * it + pr) + 8 * ag, w.lo, w.hi, oct);
            }
          }
        }
      }
    }
    cur ^= 1;
    par ^= 1;
    if (ends) {  // (every lane: they pass each other the steps)
      // the state after step L - 1 (the row's last chunk may be partial), from this wave's own rows
      if constexpr (!ONE) x_end = load_end();
      if constexpr (FINE) {
        // q^rem h + p sum_e q^e x[rem - 1 - e], h the state in front of that chunk; lane (n, a) = (lane % 16, lane / 16) adds
        // up the exponents 16 a .. 16 a + 15 of mode n.  (Step by step the rounding of q alone costs 1e-6 over a chunk.)
        const int first = cl == 0 ? w.lo : 0, n = lane & 15, a = lane >> 4;
        const cf q1 = sm.pw[8][n];
        cf t{0.f, 0.f};
#pragma unroll(ONE ? 4 : 1)
        for (int k = 0; k < 4; ++k) {
          cf v{0.f, 0.f};
#pragma unroll
          for (int e = 3; e >= 0; --e) {
            const int j = rem - 1 - (16 * a + 4 * k + e);
            const float xv = __shfl(x_end, j & 63, 64);
            v = cmul(q1, v);
            if (j >= first) v.x += xv;
          }
          t = cadd(t, cmul(sm.pw[k][n], v));
        }
        t = cmul(sm.pw[4 + a][n], t);
        t.x += __shfl_xor(t.x, 16, 64);
        t.y += __shfl_xor(t.y, 16, 64);
        t.x += __shfl_xor(t.x, 32, 64);
        t.y += __shfl_xor(t.y, 32, 64);
        cf qr = rem == kT ? sm.pw[9][n] : cmul(sm.pw[(rem >> 2) & 3][n], sm.pw[4 + ((rem >> 4) & 3)][n]);
        for (int e = rem & 3; e > 0; --e) qr = cmul(qr, q1);
        const float* prev = cl == 0 ? sm.wave_cin[wave] + 2 * n : sm.H + (c0 + cl) * kHP + 2 * n;
        const cf h = cmul(qr, cf{prev[0], prev[1]});
        if (lane < N) h_last[w.row * N + lane] = cf{h.x + sm.pn[n] * t.x, h.y + sm.pn[n] * t.y};
      } else {
        const int n = lane & 15;
        cf h;
        if (rem == kT) {
          const float* lastrow = sm.H + (1 + c0 + cl) * kHP + 2 * n;
          h = cf{lastrow[0], lastrow[1]};
        } else {
          const float* prev = cl == 0 ? sm.wave_cin[wave] + 2 * n : sm.H + (c0 + cl) * kHP + 2 * n;
          // the recurrence itself over the last chunk's steps: h <- q h + p x
          h = cf{prev[0], prev[1]};
          const cf q1 = sm.pw[8][n];
          const float pp = sm.pn[n];
          for (int j = 0; j < rem; ++j) {
            const float xv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x_end), j)) * pp;
            h = cmul(q1, h);
            h.x += xv;
          }
        }
        if (lane < N) h_last[w.row * N + lane] = h;
      }
    }
  };

  load_tile(xb, cur_tile);
  if constexpr (ONE) {
    item(blockIdx.x, 0, ln.tiles(blockIdx.x));
    return;
  }
  for (int group = blockIdx.x; group < ln.groups; group += static_cast<int>(gridDim.x)) {
    const int tiles = ln.tiles(group);
    for (int t0 = 0; t0 < tiles; t0 += kWaves) item(group, t0, tiles);
  }
}

// How many rows of a channel a group takes: as many as leave `slots` groups, so that a small
// launch still fills the chip.
Lines make_lines(int64_t B, int64_t D, int64_t L, int64_t slots, bool single, int rows) {
  Lines ln;
  int64_t nb = single ? 1 : B * D / slots;
  nb = nb < 1 ? 1 : (nb > B ? B : nb);
  ln.B = static_cast<int>(B);
  ln.D = static_cast<int>(D);
  ln.nb = static_cast<int>(nb);
  ln.groups = static_cast<int>(D * ((B + nb - 1) / nb));
  ln.L = L;
  const int64_t chunks = (L + (rows == kShifted ? 7 : 0) + kT - 1) / kT;  // of a row with steps in front of it
  ln.tpr = static_cast<int>((chunks + 31) / 32);
  return ln;
}
int compute_units(int* cus) {
  int dev = 0;
  MEGA_CHECK_HIP(hipGetDevice(&dev));
  MEGA_CHECK_HIP(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev));
  return MEGA_OK;
}

template <int DT, int ROWS, bool ONE>
int launch_fwd_as(const void* x, void* y, const Coeffs& co, const cf* h0, cf* h_last, const Lines& ln, unsigned grid, int64_t N, hipStream_t stream) {
  const size_t lds = ONE ? (kFine<ROWS> ? sizeof(FwdSmemOneFine) : sizeof(FwdSmemOne)) : (kFine<ROWS> ? sizeof(FwdSmemFine) : sizeof(FwdSmem));
  MEGA_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&cema_scan_fwd_kernel<DT, ROWS, ONE>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
  cema_scan_fwd_kernel<DT, ROWS, ONE><<<dim3(grid), kThreads, lds, stream>>>(x, y, co, h0, h_last, ln, static_cast<int>(N));
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}
// Whether the groups hold no more than the four tiles of an item each: a workgroup per group then.
int lines_of(int64_t B, int64_t D, int64_t L, int rows, Lines* ln, int64_t* slots, bool* one) {
  int cus = 0;
  if (const int rc = compute_units(&cus); rc != MEGA_OK) return rc;
  *slots = 4 * static_cast<int64_t>(cus);  // workgroups that fit the chip
  *ln = make_lines(B, D, L, *slots, false, rows);
  *one = ln->nb * static_cast<int64_t>(ln->tpr) <= kWaves;
  if (!*one) {
    *slots = 3 * static_cast<int64_t>(cus);
    *ln = make_lines(B, D, L, *slots, false, rows);
  }
  return MEGA_OK;
}
template <int DT, int ROWS>
int launch_fwd(const void* x, void* y, const Coeffs& co, const cf* h0, cf* h_last, int64_t B, int64_t D, int64_t N,
               int64_t L, hipStream_t stream) {
  Lines ln;
  int64_t slots = 0;
  bool one = false;
  if (const int rc = lines_of(B, D, L, ROWS, &ln, &slots, &one); rc != MEGA_OK) return rc;
  if (one) return launch_fwd_as<DT, ROWS, true>(x, y, co, h0, h_last, ln, static_cast<unsigned>(ln.groups), N, stream);
  return launch_fwd_as<DT, ROWS, false>(x, y, co, h0, h_last, ln, static_cast<unsigned>(ln.groups < slots ? ln.groups : slots), N, stream);
}


// ------------------------------ backward ------------------------------------
// With c_n = p_n gamma_n and, per mode,
//   A = sum_{t >= s} dy[t] x[s] q^(t-s),   B = dA / dq
// the gradients the reference forms from dk (ema_parameters.cc:80-98 after
// fftconv.py:53-75) are dp = Re(A gamma), dq = conj(B p gamma), dgamma = conj(A p),
// domega = sum dy x, and dx[s] = sum_{t >= s} k[t-s] dy[t] + omega dy[s].  By chunks, in
// reverse time (DY[c][i] = dy[64 c + i], XR[c][j'] = x[64 c + 63 - j']):
//   (G, G')[c]   = Pg DY[c],     Pg = rows (Re, Im)(q^i), then (Re, Im)(i / 64 q^i), i < 64
//   R[c]  = G[c] + q^64 R[c+1],   R'[c] = G'[c] + q^64 (R[c+1] + R'[c+1])            (scan)
//   (X, X')[c]   = Pg XR[c]
//   W  = sum_c X[c] R[c+1],   W' = sum_c (X'[c] R[c+1] + X[c] R'[c+1])
//   DX[c] = K^T DY[c] + Qd R[c+1],   Qd[j][m] = (Re, -Im)(c_n q_n^(64-j)),  omega on the diagonal of K
//   M     = sum_c DY[c]^T X[c]   (64 x 64, rows i >= columns j), dkin[l] = sum_j M[j+l][j]
//   A = sum_l q^l dkin[l] + q W,   B = sum_l l q^(l-1) dkin[l] + W + 64 W'
// Primed states are derivatives by q times q / 64, so that a step over n chunks multiplies both by one power,
// R' <- G' + q^(64 n) (R' + n R): ten operations a chunk, mode and pass instead of eighteen.
// Segments of 128 chunks are taken from the end of the row to its start; a
// wave holds one chunk tile of the segment.  The chunk-contracted product M
// needs operands with chunks along k: the wave parks its DY and X tiles in a
// private LDS tile and reads them back with the transposing LDS read; the same
// tile hands out the time-reversed x operand.  Everything that reads the dy
// and x tiles comes before the scan, so the next item's tiles load under it.
constexpr int kRP = 68;       // floats per row of the reverse-state buffer: (R, R') = 64 + 4
constexpr int kSP = 72;       // 16-bit elements per row of a wave's staging tile: 64 + 8
constexpr int kBwdNC = kWaves * 32;  // chunks per segment
constexpr int kBwdCPS = kBwdNC / kSubs;
constexpr int kBwdBlocks = 16;  // Pg 0..7 (kind, k-step), K^T 8..11 (by offset), Qd 12..15 (row tile, k-step)

typedef short short4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 lds_read_tr(const uint16_t* q) {
  const short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4v*)(q));
  return __builtin_bit_cast(uint2, v);
}

// Float16 rows are taken as they are: dy and x are matrix operands of their own type, the power matrix two float16 pieces
// (three where the bfloat16 form has three).  Powers are at most 1; brought to 2^15 they have 22 (33) bits there and lose
// nothing above 2^-40, which a float16 dx does not resolve (dy c 2^-40 is its last place where dy c is its largest).  The
// lags of k and the state part stay in bfloat16 pieces, whose range they need: omega stands on the lag at zero and may be any
// multiple of the others.  So the product K^T DY takes dy in two bfloat16 pieces too, split where it is multiplied.  R
// and X are 2^15 times themselves, a scale that Qd and the row's reductions take back.  With rows as bfloat16 pieces three
// launches (four where third pieces are) added up what one gives now: backward of 1024 x 35840 400 / 87 us, 4096 x 32768
// 1334 / 296, 4 x 2048 x 5001 667 / 141, 2 x 512 x 759 82 / 20.  (The lags as two float16 pieces too, scaled with the largest: 84,
// 281, 133, 19.5, but a lag at 2^-20 of omega had 17 bits and one at 2^-26 11.)
constexpr float kPowScale = 32768.f;
// eight 16-bit steps as bfloat16 pieces, whose sum they are exactly
template <int DT>
struct DyPieces {
  static constexpr int XP = DT == MEGA_F16 ? 2 : 1;
  u32x4 pc[XP];
  __device__ __forceinline__ explicit DyPieces(const XOp<MEGA_BF16>& steps) {
    const u32x4 raw = steps.pc[0];
    if constexpr (DT == MEGA_F16) {
      float v[8];
      unpack8<MEGA_F16>(make_uint4(raw[0], raw[1], raw[2], raw[3]), v);
      split8(v, pc[0], pc[1]);
    } else {
      pc[0] = raw;
    }
  }
};
struct BwdSmem {
  u32x4 aop[kBwdBlocks][2][kWave];       // operand blocks, two pieces
  // row c: (R, R') at the start of chunk c of the segment.  A wave's own 32 rows double as its
  // private tile for the parked dy / x data before they are written; between rows the buffer
  // holds the power table (setup) and the reduction scratch (finish).
  float R[kBwdNC * kRP];
  float pn[16];
  cf gn[16];
  cf pw[12][16];                         // powers evaluated directly (see setup_row)
  cf sub_end[kSubs][2][16];              // local (R, R') at the start of each sub-segment
  cf wave_end[2][kWaves][2][16];         // the same for each wave's four sub-segments, by item parity
  float wave_cin[kWaves][64];            // (R, R') behind each wave's last chunk
  cf carry[2][2][16];
};
// a row's reductions, in the place of a wave's own sub-segment ends
struct BwdSums {
  float red[2][32];
  float dpart[kT];
  float dkin[kT];                        // wave 0's
};
static_assert(sizeof(BwdSums) <= sizeof(cf) * 4 * 2 * 16, "a wave's sums fit its four sub-segments");
struct BwdSmemFine : BwdSmem {
  u32x4 third[4][kWave];                 // third pieces of Pg, first kind (the second kind's: in registers)
  alignas(4) ThirdTable kthird;
};
static_assert(sizeof(cf) * 16 * (kT + 2) + sizeof(cf) * 16 * 2 * 16 <= sizeof(float) * kBwdNC * kRP,
              "the power table and the final partial sums live in the state buffer");
static_assert(32 * kSP * 2 <= 32 * kRP * 4 && 16 * kWave * 4 <= 32 * kRP * 4 && kWave * 33 <= 32 * kRP,
              "a wave's parked tile and one accumulator tile fit its own rows of the state buffer");
static_assert(sizeof(cf) * 16 * (kT + 2) + sizeof(u32x4) * 4 * kWave + sizeof(float) * kT <= sizeof(float) * kBwdNC * kRP,
              "the third pieces of the second kind pass through the state buffer, behind the power table, k behind them");
static_assert(sizeof(BwdSmemFine) <= 80 * 1024, "two workgroups per compute unit");

// (h, h') <- (g, g') + m (h, h' + n h): the reverse scan's step over n chunks (m = q^(64 n)): one, a
// sub-segment or a wave's
__device__ __forceinline__ void rstep(cf& h, cf& hd, cf g, cf gd, cf m, float n) {
  const cf t{fmaf(n, h.x, hd.x), fmaf(n, h.y, hd.y)};
  h = cfma(m, h, g);
  hd = cfma(m, t, gd);
}

// DX32: dx is written in float32 (or, with a null pointer, not at all) instead of the rows'
// own type -- for callers that add up the backward of several bfloat16 pieces of one tensor;
// DX32 == 2 adds to what dx holds instead of overwriting it.
template <int DT, int DX32, int ROWS>
__global__ __launch_bounds__(kThreads, 2) void cema_scan_bwd_kernel(
    const void* __restrict__ dy, const void* __restrict__ x, void* __restrict__ dx,
    const float* __restrict__ p, const cf* __restrict__ log_q, const cf* __restrict__ gamma,
    const float* __restrict__ omega, const cf* __restrict__ h0, float* __restrict__ dp, cf* __restrict__ dq,
    cf* __restrict__ dgamma, float* __restrict__ domega, cf* __restrict__ dh0, const Lines ln, int N) {
  static_assert(DT == MEGA_BF16 || (DT == MEGA_F16 && DX32 == 0), "bfloat16 rows, or float16 rows with dx of their type");
  constexpr bool H16 = DT == MEGA_F16;
  constexpr float kScale = H16 ? kPowScale : 1.f;  // of Pg
  using Op = XOp<MEGA_BF16>;                       // eight 16-bit steps as they are
  constexpr int CPS = kBwdCPS;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr bool FINE = kFine<ROWS>;
  constexpr bool WIDE = FINE && DX32 != 0;  // Qd and the states as float32 operands
  using Smem = typename std::conditional<FINE, BwdSmemFine, BwdSmem>::type;
  Smem& sm = *reinterpret_cast<Smem*>(smem_raw);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  // lane-derived indices, re-derived from an opaque thread id wherever a phase starts
#define MEGA_LANE_IDS                                                          \
  const int tid = opaque(threadIdx.x) & (kThreads - 1), lane = tid & (kWave - 1); \
  const int g = lane >> 5, r = lane & 31, sn = tid & 15, sa = tid >> 4, sl = sa & 3; \
  (void)g; (void)r; (void)sn; (void)sa; (void)sl; (void)lane;                   \
  float* const myrows = sm.R + wave * 32 * kRP;                                \
  uint16_t* const stage = reinterpret_cast<uint16_t*>(myrows);                 \
  (void)stage
  cf (*qp)[kT + 2] = reinterpret_cast<cf(*)[kT + 2]>(sm.R);                 // setup and finish only
  cf (*ab)[2][16] = reinterpret_cast<cf(*)[2][16]>(sm.R + 2 * 16 * (kT + 2));  // finish only, behind the table
  u32x4 (*passed)[kWave] = reinterpret_cast<u32x4(*)[kWave]>(sm.R + 2 * 16 * (kT + 2));  // setup only, the same place
  float* const klocal = sm.R + 2 * 16 * (kT + 2) + 4 * 4 * kWave;  // setup only: k[0 .. 63] (+ omega at lag 0)
  auto sums = [&](int wv) -> BwdSums& { return *reinterpret_cast<BwdSums*>(&sm.sub_end[4 * wv][0][0]); };  // finish only
  u32x4 third1[4];  // FINE: third pieces of Pg, second kind
  // the last four tiles of a group's line, where its walk starts
  auto tail_of = [&](int group) { return group < ln.groups ? (ln.tiles(group) - 1) / kWaves * kWaves : 0; };

  Op db[4], xb[4], dn[4];  // dn: the next item's dy tile on its way
  auto load_dy = [&](const Tile& w) {
    MEGA_LANE_IDS;
    const uint16_t* row = static_cast<const uint16_t*>(dy) + w.base;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      dn[s].template load<ROWS>(row, r * kT + 16 * s + 8 * g, w.lo, w.hi);
  };
  auto load_x = [&](const Tile& w) {
    MEGA_LANE_IDS;
    const uint16_t* row = static_cast<const uint16_t*>(x) + w.base;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      xb[s].template load<ROWS>(row, r * kT + 16 * s + 8 * g, w.lo, w.hi);
  };
  struct RowParams {
    cf lq, gv;
    float pv, w;
  };
  auto fetch_params = [&](int group) {
    MEGA_LANE_IDS;
    RowParams rp{cf{0.f, 0.f}, cf{0.f, 0.f}, 0.f, 0.f};
    if (group < ln.groups) {
      const int d = group % ln.D;
      if (sn < N) {
        rp.lq = log_q[d * N + sn];
        rp.gv = gamma[d * N + sn];
        rp.pv = p[d * N + sn];
      }
      if (omega != nullptr) rp.w = omega[d];
    }
    return rp;
  };
  auto load_block = [&](int b, u32x4* dst, int lane) {
    dst[0] = sm.aop[b][0][lane];
    dst[1] = sm.aop[b][1][lane];
  };

  // scan multipliers of this thread's mode: over a chunk, a sub-segment, a wave's chunks
  cf qT{0.f, 0.f}, q1{0.f, 0.f};
  int cur = 0, par = 0;
  RowParams rp = fetch_params(blockIdx.x);


  // per-row accumulators
  floatx16 macc[3];      // M tiles (0,0), (1,0), (1,1) over this wave's chunks
  cf wacc[8], wdacc[8];  // W, W' of modes n = 4 qd + 2 g + b at index 2 qd + b, over this lane's chunks

  auto setup_row = [&](int group) {
    MEGA_LANE_IDS;
    // powers evaluated directly (phase reduced in float64), 12 per mode: q^(4 k), q^(16 k)
    // (k < 4), q, q^64, q^(64 CPS), q^(256 CPS)
    cf direct{0.f, 0.f};
    if (tid < 12 * 16 && sn < N) {
      const int k = tid >> 4;
      const int tab[4] = {1, kT, kT * CPS, 4 * kT * CPS};
      const int e = k < 4 ? 4 * k : (k < 8 ? 16 * (k - 4) : tab[k - 8]);
      direct = qpow(rp.lq.x, rp.lq.y, e);
    }
    __syncthreads();  // every wave is done with the previous row's tables and reductions
    if (tid < 12 * 16) sm.pw[tid >> 4][sn] = direct;
    if (tid < 16) {
      sm.pn[tid] = rp.pv;
      sm.gn[tid] = rp.gv;
      sm.carry[0][0][tid] = cf{0.f, 0.f};
      sm.carry[0][1][tid] = cf{0.f, 0.f};
    }
    cur = 0;
    __syncthreads();
    {
      cf v = cmul(sm.pw[sa & 3][sn], sm.pw[4 + (sa >> 2)][sn]);
      q1 = sm.pw[8][sn];
      const cf c{rp.pv * rp.gv.x, rp.pv * rp.gv.y};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qp[sn][4 * sa + e] = v;
        const float kl = group_sum<16>(c.x * v.x - c.y * v.y);
        if (sn == 0) klocal[4 * sa + e] = (sa == 0 && e == 0) ? kl + rp.w : kl;  // omega on the diagonal
        v = cmul(v, q1);
      }
      if (sa == 15) qp[sn][kT] = sm.pw[9][sn];
      qT = sm.pw[9][sn];
    }
    __syncthreads();
    for (int item = tid; item < kBwdBlocks * kWave; item += kThreads) {
      const int blk = item >> 6, ln = item & 63, rr = ln & 31, gg = ln >> 5;
      float v[8];
      if (blk < 8) {
        const int kind = blk >> 2, s = blk & 3, n = rr >> 1, part = rr & 1;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int i = 16 * s + 8 * gg + e;
          const cf w = qp[n][i];
          const float sc = kScale * (kind ? static_cast<float>(i) / kT : 1.f);
          v[e] = sc * (part ? w.y : w.x);
        }
      } else if (blk < 12) {
        const int o = 16 * (blk - 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int lag = o - rr + 8 * gg + e;
          const float kv = klocal[lag >= 0 ? lag : 0];  // read, then masked: no branch around the load
          v[e] = lag >= 0 ? kv : 0.f;
        }
      } else {
        const int jt = (blk - 12) >> 1, s2 = (blk - 12) & 1, j = 32 * jt + rr;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int m = 16 * s2 + 8 * gg + e, n = m >> 1;
          const cf c = cf{sm.pn[n] * sm.gn[n].x, sm.pn[n] * sm.gn[n].y};
          const cf w = cmul(c, qp[n][kT - j]);
          v[e] = (m & 1) ? -w.y : w.x;
          if (H16) v[e] *= 1.f / kPowScale;
        }
      }
      u32x4 hi, lo, third;
      if (WIDE && blk >= 12) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sm.aop[blk][0][ln][e] = __float_as_uint(v[e]);
          sm.aop[blk][1][ln][e] = __float_as_uint(v[4 + e]);
        }
        continue;
      }
      if (H16 && blk < 8) split8_f16<FINE>(v, hi, lo, third);
      else split8(v, hi, lo);
      if (FINE && !H16) third = split8_third(v, hi, lo);
      sm.aop[blk][0][ln] = hi;
      sm.aop[blk][1][ln] = lo;
      if constexpr (FINE)
        if (blk < 8) (blk < 4 ? sm.third[blk] : passed[blk - 4])[ln] = third;
    }
    if constexpr (FINE) fill_thirds<false>(sm.kthird, klocal, tid);
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) macc[t][i] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) wacc[i] = wdacc[i] = cf{0.f, 0.f};
    __syncthreads();
    if constexpr (FINE) {
#pragma unroll
      for (int s = 0; s < 4; ++s) third1[s] = passed[s][lane];
      __syncthreads();  // every wave has its pieces: the buffer takes the parked tiles
    }
    rp = fetch_params(group + static_cast<int>(gridDim.x));
  };

  // the row's reductions and its five gradient outputs
  auto finish_row = [&](int64_t row) {  // the group's outputs; with a carried state a group is one row
    MEGA_LANE_IDS;
    // W, W': over the 32 lanes (chunks) of a half wave, then over the waves.  A lane holds 32
    // partial sums (8 modes x (W, W') x (re, im)) and each half of the wave its own 8 modes: the
    // wave transposes them through its rows of the state buffer ([lane][value], pitch 33), and
    // lane (g, t) adds up value t of half g.
    wave_sync();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float* dst = myrows + lane * 33 + 4 * i;
      dst[0] = wacc[i].x;
      dst[1] = wacc[i].y;
      dst[2] = wdacc[i].x;
      dst[3] = wdacc[i].y;
    }
    wave_sync();
    {
      float part[32];
#pragma unroll
      for (int j = 0; j < 32; ++j) part[j] = myrows[(32 * g + j) * 33 + r];
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 32; ++j) acc += part[j];
      sums(wave).red[g][r] = acc;
    }
    // dkin[l] = sum_j M[j + l][j]: each wave sums the diagonals of its own M, one 32 x 32 tile
    // at a time through its own rows of the state buffer ([i][j], pitch 33).  Lane (g, t) walks
    // the wrapped diagonal tile[(j + t) mod 32][j] over its 16 columns j = 16 g .. 16 g + 15:
    // the part with j + t < 32 belongs to the diagonal d = t, the rest to d = t - 32.  The tiles
    // (0,0) and (1,1) hold the same lags d >= 0 (their d < 0 is not asked for) and are added
    // first; the tile (1,0) holds lag 32 + d for both signs of d.
    {
      float lo[2], hi[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        wave_sync();
#pragma unroll
        for (int i = 0; i < 16; ++i)
          myrows[(8 * (i >> 2) + 4 * g + (i & 3)) * 33 + r] = t == 0 ? macc[0][i] + macc[2][i] : macc[1][i];
        wave_sync();
        float v[16];
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
          const int j = 16 * g + jj;
          v[jj] = myrows[((j + r) & 31) * 33 + j];
        }
        lo[t] = hi[t] = 0.f;
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
          const bool below = 16 * g + jj + r < 32;
          lo[t] += below ? v[jj] : 0.f;
          hi[t] += below ? 0.f : v[jj];
        }
      }
      // the two halves of the wave took different columns
      const float same = lo[0] + __shfl_xor(lo[0], 32, 64);
      const float cross_lo = lo[1] + __shfl_xor(lo[1], 32, 64);
      const float cross_hi = hi[1] + __shfl_xor(hi[1], 32, 64);
      // lag l <= 31: same[d = l] + cross[d = l - 32]; lag l >= 32: cross[d = l - 32]
      sums(wave).dpart[lane] = g == 0 ? same + cross_hi : cross_lo;
    }
    __syncthreads();  // every wave is done with the state buffer: it takes the power table again
    if (tid < kT) sums(0).dkin[tid] = (sums(0).dpart[tid] + sums(1).dpart[tid]) + (sums(2).dpart[tid] + sums(3).dpart[tid]);
    {
      cf v = cmul(sm.pw[sa & 3][sn], sm.pw[4 + (sa >> 2)][sn]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qp[sn][4 * sa + e] = v;
        v = cmul(v, q1);
      }
    }
    __syncthreads();
    {
      // A_in = sum_l q^l dkin[l], B_in = sum_l l q^(l-1) dkin[l]: thread (n, a) takes l = 4 a .. 4 a + 3
      cf ain{0.f, 0.f}, bin{0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int l = 4 * sa + e;
        const float dk = sums(0).dkin[l];
        const cf v = qp[sn][l];
        ain.x = fmaf(dk, v.x, ain.x);
        ain.y = fmaf(dk, v.y, ain.y);
        if (l > 0) {
          const cf u = qp[sn][l - 1];
          const float dl = dk * static_cast<float>(l);
          bin.x = fmaf(dl, u.x, bin.x);
          bin.y = fmaf(dl, u.y, bin.y);
        }
      }
      ab[sa][0][sn] = ain;
      ab[sa][1][sn] = bin;
    }
    __syncthreads();
    if (tid < N) {
      const int n = tid;
      cf ain{0.f, 0.f}, bin{0.f, 0.f};
      for (int a = 0; a < 16; ++a) {
        ain = cadd(ain, ab[a][0][n]);
        bin = cadd(bin, ab[a][1][n]);
      }
      // mode n sits in half g = (n >> 1) & 1 at index 2 (n >> 2) + (n & 1)
      const int hg = (n >> 1) & 1, idx = 2 * (n >> 2) + (n & 1);
      cf w{0.f, 0.f}, wd{0.f, 0.f};
      for (int wv = 0; wv < kWaves; ++wv) {
        const float* part = sums(wv).red[hg] + 4 * idx;
        w.x += part[0];
        w.y += part[1];
        wd.x += part[2];
        wd.y += part[3];
      }
      if (H16) {  // (X and R each)
        constexpr float back = 1.f / (kPowScale * kPowScale);
        w = cf{back * w.x, back * w.y};
        wd = cf{back * wd.x, back * wd.y};
      }
      const cf qq = sm.pw[8][n];
      const cf A = cadd(ain, cmul(qq, w));
      const cf Bq{fmaf(kT, wd.x, bin.x + w.x), fmaf(kT, wd.y, bin.y + w.y)};
      const cf gm = sm.gn[n];
      const float pp = sm.pn[n];
      dp[row * N + n] = A.x * gm.x - A.y * gm.y;
      const cf t = cmul(Bq, cf{pp * gm.x, pp * gm.y});
      cf dqv{t.x, -t.y}, dgv{A.x * pp, -A.y * pp};
      if (!H16 && h0 != nullptr) {  // (float16 rows with a carried state go in pieces)
        // A carried state h0 adds b[t] = Re(gamma q^(t+1) h0) to the output (ema_parameters.cc:56-77).
        // With R0 = sum_t dy[t] q^t and R0' = dR0 / dq -- what the reverse scan has carried to the
        // start of the row -- its gradients are (ema_parameters.cc:158-188, PyTorch's convention)
        //   dgamma += conj(q h0 R0),  dq += conj(gamma h0 (R0 + q R0')),  dh0 = conj(gamma q R0)
        // (q R0' = 64 times what the scan has carried).
        const cf r0 = sm.carry[cur][0][n], r0d = sm.carry[cur][1][n];
        const cf h = h0[row * N + n];
        const cf e1 = cmul(cmul(qq, h), r0);
        dgv.x += e1.x;
        dgv.y -= e1.y;
        const cf e2 = cmul(cmul(gm, h), cf{fmaf(kT, r0d.x, r0.x), fmaf(kT, r0d.y, r0.y)});
        dqv.x += e2.x;
        dqv.y -= e2.y;
        if (dh0 != nullptr) {
          const cf e3 = cmul(cmul(gm, qq), r0);
          dh0[row * N + n] = cf{e3.x, -e3.y};
        }
      }
      dq[row * N + n] = dqv;
      dgamma[row * N + n] = dgv;
    }
    // the skip term sat on the diagonal of K, not in M: domega = sum dy x = dkin[0]
    if (tid == 0) domega[row] = sums(0).dkin[0];
  };

  Tile cur_tile = tile_at<ROWS>(ln, blockIdx.x, tail_of(blockIdx.x) + wave);  // this wave's tile of the item
  auto item = [&](int group, int t0, int tiles) {
    MEGA_LANE_IDS;
    // transposing read of the parked tile: row tile tt (32 time steps), k-step ks (16 chunks)
    const int tr_base = (8 * g + ((lane & 15) >> 2)) * kSP + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    auto read_tr = [&](int tt, int ks) {
      const uint16_t* q = stage + tr_base + 16 * ks * kSP + 32 * tt;
      const uint2 lo = lds_read_tr(q), hi = lds_read_tr(q + 4 * kSP);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    if (t0 + kWaves >= tiles) setup_row(group);
    const Tile w = cur_tile;
    using dx_t = typename std::conditional<DX32 != 0, float, uint16_t>::type;
    dx_t* dxrow = static_cast<dx_t*>(dx) + w.base;
    const bool on = w.nc > 0;
    u32x4 xr[4];  // time-reversed x as an operand: steps 63 - (16 s + 8 g + e)
    // the next item of this workgroup: its x tile is requested as soon as this item's has been
    // consumed, its dy tile at the end of the item
    Tile next = w;
    if (t0 > 0) {
      tile_backward<ROWS>(ln, next, tiles);
    } else {
      const int ng = group + static_cast<int>(gridDim.x);
      next = tile_at<ROWS>(ln, ng, tail_of(ng) + wave);
    }
    if (on) {
      // ---- the wave's private tile: X parked first (it arrived an item ago), read back with
      //      chunks along k and time-reversed; then DY, whose loads were issued last ------------
      uint16_t* mine = stage + r * kSP + 8 * g;
      if (ROWS == kShifted && w.cut())
#pragma unroll
        for (int s = 0; s < 4; ++s) xb[s].keep(r * kT + 16 * s + 8 * g, w.lo, w.hi);
#pragma unroll
      for (int s = 0; s < 4; ++s) *reinterpret_cast<u32x4*>(mine + 16 * s) = xb[s].pc[0];
      wave_sync();
      u32x4 xt[2][2];
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) xt[jt][ks] = read_tr(jt, ks);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(stage + r * kSP + 56 - 16 * s - 8 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) xr[s][e] = __builtin_amdgcn_alignbit(v[3 - e], v[3 - e], 16);
      }
      wave_sync();
      if (ROWS == kShifted && w.cut())
#pragma unroll
        for (int s = 0; s < 4; ++s) db[s].keep(r * kT + 16 * s + 8 * g, w.lo, w.hi);
#pragma unroll
      for (int s = 0; s < 4; ++s) *reinterpret_cast<u32x4*>(mine + 16 * s) = db[s].pc[0];
      wave_sync();
      // M += DY^T X over the tile's 32 chunks
#pragma unroll
      for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const u32x4 dyt = read_tr(it, ks);
          if (it == 0) macc[0] = mfma16<DT>(dyt, xt[0][ks], macc[0]);
          if (it == 1) {
            macc[1] = mfma16<DT>(dyt, xt[0][ks], macc[1]);
            macc[2] = mfma16<DT>(dyt, xt[1][ks], macc[2]);
          }
        }
      wave_sync();  // the tile has been read: its place takes the wave's rows of (G, G')
    }
    load_x(next);
    floatx16 xacc[2];  // (X, X') of the lane's chunk, until R is there
    if (on) {
      // ---- (G, G') = Pg DY, into this wave's own rows of the state buffer, and (X, X') = Pg XR with
      //      the same operands ---------------------------------------------------------------------
#pragma unroll
      for (int kind = 0; kind < 2; ++kind) {
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = xacc[kind][i] = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          u32x4 a[2];
          load_block(kind * 4 + s, a, lane);
          acc = mfma16<DT>(a[1], db[s].pc[0], mfma16<DT>(a[0], db[s].pc[0], acc));
          xacc[kind] = mfma16<DT>(a[1], xr[s], mfma16<DT>(a[0], xr[s], xacc[kind]));
          if constexpr (FINE) {
            const u32x4 third = kind ? third1[s] : sm.third[s][lane];
            acc = mfma16<DT>(third, db[s].pc[0], acc);
            xacc[kind] = mfma16<DT>(third, xr[s], xacc[kind]);
          }
        }
        float* dst = myrows + r * kRP + 32 * kind + 4 * g;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          *reinterpret_cast<float4*>(dst + 8 * qd) =
              make_float4(acc[4 * qd], acc[4 * qd + 1], acc[4 * qd + 2], acc[4 * qd + 3]);
      }
    }
    wave_sync();
    load_dy(next);
    // ---- reverse scan over the chunks of the segment; a wave's four sub-segments are its own
    //      chunks, one workgroup barrier hands over the waves' ends ---------------------------------
    //      (a wave whose tile has no steps passes on zeros: it may be its row's last, kShifted.  Chunks behind the
    //      row's end need no mask: their DY is zero, so their G is, and the scan starts from zero behind them)
    float* const col = sm.R + sa * CPS * kRP + 2 * sn;
    float2 gv[CPS], gd[CPS];
    const cf qS = sm.pw[10][sn], qW = sm.pw[11][sn];  // over a sub-segment, over a wave's chunks
    if (on) {
#pragma unroll
      for (int i = 0; i < CPS; ++i) {
        gv[i] = *reinterpret_cast<const float2*>(col + i * kRP);
        gd[i] = *reinterpret_cast<const float2*>(col + i * kRP + 32);
      }
      cf e{0.f, 0.f}, ed{0.f, 0.f};
#pragma unroll
      for (int i = CPS - 1; i >= 0; --i) rstep(e, ed, cf{gv[i].x, gv[i].y}, cf{gd[i].x, gd[i].y}, qT, 1.f);
      sm.sub_end[sa][0][sn] = e;
      sm.sub_end[sa][1][sn] = ed;
      wave_sync();
      if (sl == 0) {
        // the wave's chunks from zero: sub-segments 3, 2, 1, then this one
        cf h = sm.sub_end[sa + 3][0][sn], hd = sm.sub_end[sa + 3][1][sn];
        rstep(h, hd, sm.sub_end[sa + 2][0][sn], sm.sub_end[sa + 2][1][sn], qS, CPS);
        rstep(h, hd, sm.sub_end[sa + 1][0][sn], sm.sub_end[sa + 1][1][sn], qS, CPS);
        rstep(h, hd, e, ed, qS, CPS);
        sm.wave_end[par][wave][0][sn] = h;
        sm.wave_end[par][wave][1][sn] = hd;
      }
    } else if (sl == 0) {
      sm.wave_end[par][wave][0][sn] = cf{0.f, 0.f};
      sm.wave_end[par][wave][1][sn] = cf{0.f, 0.f};
    }
    lds_barrier();
    {
      cf h = sm.carry[cur][0][sn], hd = sm.carry[cur][1][sn];
      // through the tiles behind this wave's, from the last one of its row if that is among the four
      // (nothing comes from behind it)
      const int k = ln.tpr - 1 - w.chunk0 / 32, from = wave + k < kWaves ? wave + k : kWaves - 1;
      if (wave + k < kWaves) h = hd = cf{0.f, 0.f};
#pragma unroll
      for (int v = kWaves - 1; v >= 1; --v)
        if (v > wave && v <= from) rstep(h, hd, sm.wave_end[par][v][0][sn], sm.wave_end[par][v][1][sn], qW, 4.f * CPS);
      if (sa == 0) {
        // through wave 0's chunks too: the state at the start of the segment, the next item's carry
        cf ch = h, chd = hd;
        rstep(ch, chd, sm.wave_end[par][0][0][sn], sm.wave_end[par][0][1][sn], qW, 4.f * CPS);
        sm.carry[cur ^ 1][0][sn] = ch;
        sm.carry[cur ^ 1][1][sn] = chd;
      }
      if (sl == 3) {  // (R, R') behind the wave's last chunk
        *reinterpret_cast<float2*>(sm.wave_cin[wave] + 2 * sn) = make_float2(h.x, h.y);
        *reinterpret_cast<float2*>(sm.wave_cin[wave] + 32 + 2 * sn) = make_float2(hd.x, hd.y);
      }
      if (on) {
#pragma unroll
        for (int s = 3; s >= 1; --s) {
          const cf se = sm.sub_end[4 * wave + s][0][sn], sed = sm.sub_end[4 * wave + s][1][sn];
          if (s > sl) rstep(h, hd, se, sed, qS, CPS);
        }
#pragma unroll
        for (int i = CPS - 1; i >= 0; --i) {
          rstep(h, hd, cf{gv[i].x, gv[i].y}, cf{gd[i].x, gd[i].y}, qT, 1.f);
          *reinterpret_cast<float2*>(col + i * kRP) = make_float2(h.x, h.y);
          *reinterpret_cast<float2*>(col + i * kRP + 32) = make_float2(hd.x, hd.y);
        }
      }
    }
    wave_sync();
    if (on) {
      // (R, R')[c + 1]: the next row of the buffer, or, for the wave's last chunk, wave_cin;
      // behind the row's end R is zero
      const float* rnext = (r == 31) ? sm.wave_cin[wave] : myrows + (r + 1) * kRP;
      // the stores of dX go out first: they have the (X, X') products and the next item's
      // staging to retire under before the next loads are issued behind them
      // ---- DX = K^T DY + Qd R[c+1] (omega dy included: K carries omega on its diagonal) -------------
      if (DX32 != 1 || dx != nullptr) {
        u32x4 hb[WIDE ? 1 : 2][2];
        float hv[2][8];
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const float* src = rnext + 16 * s2 + 8 * g;
          const float4 u0 = *reinterpret_cast<const float4*>(src);
          const float4 u1 = *reinterpret_cast<const float4*>(src + 4);
          const float v[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
          if constexpr (WIDE) {
#pragma unroll
            for (int e = 0; e < 8; ++e) hv[s2][e] = v[e];
          } else {
            split8(v, hb[s2][0], hb[s2][1]);
          }
        }
#pragma unroll
        for (int jt = 0; jt < 2; ++jt) {
          floatx16 acc;
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
          for (int s = 2 * jt; s < 4; ++s) {
            u32x4 a[2];
            load_block(8 + s - 2 * jt, a, lane);
            const DyPieces<DT> d(db[s]);
            acc = mma_split<DyPieces<DT>::XP, true>(a, d.pc, acc);
            // (block b: lags 16 b - r + 8 g + e; of two-piece steps the third pieces' product with the second, 2^-26, is left out)
            if constexpr (FINE) acc = mfma_bf16(read_thirds(sm.kthird, 16 * (s - 2 * jt) - r + 8 * g + 31), d.pc[0], acc);
          }
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            u32x4 a[2];
            load_block(12 + 2 * jt + s2, a, lane);
            if constexpr (WIDE) acc = mma_f32(a, hv[s2], acc);
            else acc = mma_split<2, FINE>(a, hb[s2], acc);
          }
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            if constexpr (DX32) {
              // registers 8 pr + 4 h + e hold the steps 16 pr + 8 h + 4 g + e
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const int elem = r * kT + 16 * (2 * jt + pr) + 8 * h + 4 * g;
                if (dx != nullptr && ROWS != kAny && (ROWS == kWhole || elem >= w.lo) && elem + 4 <= w.hi) {
                  float4 v = make_float4(acc[8 * pr + 4 * h], acc[8 * pr + 4 * h + 1], acc[8 * pr + 4 * h + 2],
                                         acc[8 * pr + 4 * h + 3]);
                  if constexpr (DX32 == 2) {
                    const float4 o = *reinterpret_cast<const float4*>(dxrow + elem);
                    v = make_float4(v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w);
                  }
                  *reinterpret_cast<float4*>(dxrow + elem) = v;
                } else if (ROWS != kWhole && dx != nullptr) {
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    if (elem + e >= w.lo && elem + e < w.hi)
                      dxrow[elem + e] = acc[8 * pr + 4 * h + e] + (DX32 == 2 ? static_cast<float>(dxrow[elem + e]) : 0.f);
                }
              }
            } else {
              const uint4 oct = octet_of<DT>(acc, pr);
              store8_16<ROWS>(dxrow, r * kT + 16 * (2 * jt + pr) + 8 * g, w.lo, w.hi, oct);
            }
          }
        }
      }
      // ---- W += X R[c+1], W' += X' R[c+1] + X R'[c+1] -----------------------------------------------
      {
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const float4 rv = *reinterpret_cast<const float4*>(rnext + 4 * g + 8 * qd);
          const float4 rd = *reinterpret_cast<const float4*>(rnext + 32 + 4 * g + 8 * qd);
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const cf xv{xacc[0][4 * qd + 2 * b], xacc[0][4 * qd + 2 * b + 1]};
            const cf xd{xacc[1][4 * qd + 2 * b], xacc[1][4 * qd + 2 * b + 1]};
            const cf rr_ = b ? cf{rv.z, rv.w} : cf{rv.x, rv.y};
            const cf rdd = b ? cf{rd.z, rd.w} : cf{rd.x, rd.y};
            wacc[2 * qd + b] = cfma(xv, rr_, wacc[2 * qd + b]);
            wdacc[2 * qd + b] = cfma(xv, rdd, cfma(xd, rr_, wdacc[2 * qd + b]));
          }
        }
      }
    }
    cur ^= 1;
    par ^= 1;
    if (t0 == 0) finish_row(group);
#pragma unroll
    for (int s = 0; s < 4; ++s) db[s] = dn[s];
    cur_tile = next;
  };

  load_x(cur_tile);
  load_dy(cur_tile);
#pragma unroll
  for (int s = 0; s < 4; ++s) db[s] = dn[s];
  for (int group = blockIdx.x; group < ln.groups; group += static_cast<int>(gridDim.x)) {
    const int tiles = ln.tiles(group);
    for (int t0 = (tiles - 1) / kWaves * kWaves; t0 >= 0; t0 -= kWaves) item(group, t0, tiles);
  }
#undef MEGA_LANE_IDS
}

// Rows of a channel that the backward puts together (make_lines); a carried state's gradients are per row.
int bwd_lines(int64_t B, int64_t D, int64_t L, bool single, int rows, Lines* ln, int64_t* slots) {
  int cus = 0;
  const int rc = compute_units(&cus);
  if (rc != MEGA_OK) return rc;
  *slots = 2 * static_cast<int64_t>(cus);  // two workgroups fit a compute unit
  *ln = make_lines(B, D, L, *slots, single, rows);
  return MEGA_OK;
}

// single: gradients per row (B, D, N) as the operator returns them; else per group of rows
template <int DX32, int ROWS, int DT = MEGA_BF16>
int launch_bwd(const void* dy, const void* x, void* dx, const float* p, const cf* log_q,
               const cf* gamma, const float* omega, const cf* h0, float* dp, cf* dq, cf* dgamma, float* domega,
               cf* dh0, int64_t B, int64_t D, int64_t N, int64_t L, bool single, hipStream_t stream) {
  const int lds = static_cast<int>(kFine<ROWS> ? sizeof(BwdSmemFine) : sizeof(BwdSmem));
  MEGA_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&cema_scan_bwd_kernel<DT, DX32, ROWS>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  Lines ln;
  int64_t slots = 0;
  const int rc = bwd_lines(B, D, L, single || h0 != nullptr, ROWS, &ln, &slots);
  if (rc != MEGA_OK) return rc;
  const unsigned grid = static_cast<unsigned>(ln.groups < slots ? ln.groups : slots);
  cema_scan_bwd_kernel<DT, DX32, ROWS><<<dim3(grid), kThreads, lds, stream>>>(
      dy, x, dx, p, log_q, gamma, omega, h0, dp, dq, dgamma, domega, dh0, ln, static_cast<int>(N));
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

using BwdLaunch = decltype(&launch_bwd<0, kWhole>);
BwdLaunch bwd_for(int dx_mode, int rows) {
  static const BwdLaunch table[4][3] = {{launch_bwd<0, kWhole>, launch_bwd<0, kShifted>, launch_bwd<0, kAny>},
                                        {launch_bwd<1, kWhole>, launch_bwd<1, kShifted>, launch_bwd<1, kAny>},
                                        {launch_bwd<2, kWhole>, launch_bwd<2, kShifted>, launch_bwd<2, kAny>},
                                        {launch_bwd<0, kWhole, MEGA_F16>, launch_bwd<0, kShifted, MEGA_F16>, launch_bwd<0, kAny, MEGA_F16>}};
  return table[dx_mode][rows];
}

// the layout of rows of length L in these tensors
int rows_of(int64_t count, int64_t L, bool carried, std::initializer_list<const void*> tensors) {
  for (const void* t : tensors)
    if (reinterpret_cast<uintptr_t>(t) % 16 != 0) return kAny;
  // (a tensor whose end is off a boundary too: the last row's aligned piece would reach past it)
  return L % 8 == 0 ? kWhole : carried || count * L % 8 != 0 ? kAny : kShifted;
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_cema_scan_supported(int dtype, int64_t N, int64_t L) {
  // (float32 rows of other lengths: mega_cema_layer_scan_fwd)
  return valid_dtype(dtype) && N >= 1 && N <= 16 && L >= 1 && (dtype != MEGA_F32 || L % 8 == 0);
}

// any_length: float32 rows of every length, as the layer takes them
static int scan_fwd_entry(const char* who, const void* x, int dtype, const Coeffs& co, const float* h0, int64_t B, int64_t D,
                          int64_t N, int64_t L, void* y, float* h_last, bool any_length, void* stream) {
  MEGA_CHECK_ARG(B >= 0 && D >= 0 && L >= 0, "%s: negative size", who);
  MEGA_CHECK_ARG(B * D <= 0x7fffffff, "%s: too many rows", who);
  if (!mega_cema_scan_supported(any_length && dtype == MEGA_F32 ? MEGA_BF16 : dtype, N, L))
    return set_error(MEGA_ERR_UNSUPPORTED,
                     "%s: needs N <= 16 and, for float32 rows, L a multiple of 8 (dtype %d, N %lld, L %lld)",
                     who, dtype, (long long)N, (long long)L);
  const int rows = rows_of(B * D, L, h0 != nullptr, {x, y});
  for (const void* t : {x, static_cast<const void*>(y)})
    MEGA_CHECK_ARG(dtype != MEGA_F32 || reinterpret_cast<uintptr_t>(t) % 16 == 0, "%s: float32 rows must be 16-byte aligned", who);
  if (B == 0 || D == 0) return MEGA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const cf* h0c = reinterpret_cast<const cf*>(h0);
  cf* hl = reinterpret_cast<cf*>(h_last);
  auto go = dtype == MEGA_F32    ? (rows == kWhole     ? launch_fwd<MEGA_F32, kWhole>
                                    : rows == kShifted ? launch_fwd<MEGA_F32, kShifted>
                                                       : launch_fwd<MEGA_F32, kAny>)
            : dtype == MEGA_BF16 ? (rows == kWhole     ? launch_fwd<MEGA_BF16, kWhole>
                                    : rows == kShifted ? launch_fwd<MEGA_BF16, kShifted>
                                                       : launch_fwd<MEGA_BF16, kAny>)
                                 : (rows == kWhole     ? launch_fwd<MEGA_F16, kWhole>
                                    : rows == kShifted ? launch_fwd<MEGA_F16, kShifted>
                                                       : launch_fwd<MEGA_F16, kAny>);
  return go(x, y, co, h0c, hl, B, D, N, L, s);
}

static int scan_fwd(const char* who, bool any_length, const void* x, int dtype, const float* p, const float* log_q, const float* gamma,
                    const float* omega, const float* h0, int64_t B, int64_t D, int64_t N, int64_t L, void* y, float* h_last,
                    void* stream) {
  MEGA_CHECK_ARG(x && p && log_q && gamma && y, "%s: null pointer", who);
  Coeffs co{};
  co.p = p;
  co.log_q = reinterpret_cast<const cf*>(log_q);
  co.gamma = reinterpret_cast<const cf*>(gamma);
  co.omega = omega;
  return scan_fwd_entry(who, x, dtype, co, h0, B, D, N, L, y, h_last, any_length, stream);
}

extern "C" int mega_cema_scan_fwd(const void* x, int dtype, const float* p, const float* log_q,
                                  const float* gamma, const float* omega, const float* h0, int64_t B,
                                  int64_t D, int64_t N, int64_t L, void* y, float* h_last,
                                  void* stream) {
  return scan_fwd("mega_cema_scan_fwd", false, x, dtype, p, log_q, gamma, omega, h0, B, D, N, L, y, h_last, stream);
}

extern "C" int mega_cema_layer_scan_fwd(const void* x, int dtype, const float* p, const float* log_q,
                                        const float* gamma, const float* omega, const float* h0, int64_t B,
                                        int64_t D, int64_t N, int64_t L, void* y, float* h_last,
                                        void* stream) {
  return scan_fwd("mega_cema_layer_scan_fwd", true, x, dtype, p, log_q, gamma, omega, h0, B, D, N, L, y, h_last, stream);
}

extern "C" int mega_cema_layer_fwd(const void* x, int dtype, int param_dtype, const void* alpha, const void* delta, const void* theta,
                                   const void* gamma, const void* omega, int64_t B, int64_t D, int64_t N, int64_t L, void* y,
                                   void* workspace, void* stream) {
  const char* who = "mega_cema_layer_fwd";
  MEGA_CHECK_ARG(x && alpha && delta && theta && gamma && omega && y && workspace, "%s: null pointer", who);
  MEGA_CHECK_ARG(valid_dtype(param_dtype), "%s: unknown parameter dtype %d", who, param_dtype);
  MEGA_CHECK_ARG(B >= 1 && D >= 1 && N >= 1 && N <= 16 && L >= 1 && B * D <= 0x7fffffff, "%s: bad sizes", who);
  Coeffs co{};
  co.dtype = param_dtype;
  co.raw_omega = omega;
  Lines ln;
  int64_t slots = 0;
  bool one = false;
  if (const int rc = lines_of(B, D, L, rows_of(B * D, L, false, {x, y}), &ln, &slots, &one); rc != MEGA_OK) return rc;
  if (one) {
    co.alpha = alpha; co.delta = delta; co.theta = theta; co.raw_gamma = gamma;
  } else {
    float* w = static_cast<float*>(workspace);
    const int rc = mega_cema_layer_coeffs_fwd(param_dtype, alpha, delta, theta, gamma, D, N, w, w + D * N, w + 3 * D * N, stream);
    if (rc != MEGA_OK) return rc;
    co.p = w;
    co.log_q = reinterpret_cast<const cf*>(w + D * N);
    co.gamma = reinterpret_cast<const cf*>(w + 3 * D * N);
  }
  return scan_fwd_entry(who, x, dtype, co, nullptr, B, D, N, L, y, nullptr, true, stream);
}

extern "C" int mega_cema_scan_bwd_supported(int dtype, int64_t N, int64_t L) {
  return dtype == MEGA_BF16 && N >= 1 && N <= 16 && L >= 1;
}

extern "C" int mega_cema_scan_bwd_state(const void* dy, const void* x, int dtype, const float* p,
                                        const float* log_q, const float* gamma, const float* omega,
                                        const float* h0, int64_t B, int64_t D, int64_t N, int64_t L, void* dx,
                                        float* dp, float* dq, float* dgamma, float* domega, float* dh0,
                                        void* stream) {
  const char* who = "mega_cema_scan_bwd";
  MEGA_CHECK_ARG(dy && x && p && log_q && gamma && dx && dp && dq && dgamma && domega, "%s: null pointer", who);
  MEGA_CHECK_ARG(B >= 0 && D >= 0 && L >= 0, "%s: negative size", who);
  MEGA_CHECK_ARG(B * D <= 0x7fffffff, "%s: too many rows", who);
  if (!mega_cema_scan_bwd_supported(dtype, N, L))
    return set_error(MEGA_ERR_UNSUPPORTED,
                     "%s: needs bfloat16 rows and N <= 16 (dtype %d, N %lld, L %lld)", who,
                     dtype, (long long)N, (long long)L);
  if (B == 0 || D == 0) return MEGA_OK;
  MEGA_CHECK_ARG(dh0 == nullptr || h0 != nullptr, "%s: dh0 without h0", who);
  return bwd_for(0, rows_of(B * D, L, h0 != nullptr, {dy, x, dx}))(dy, x, dx, p, reinterpret_cast<const cf*>(log_q), reinterpret_cast<const cf*>(gamma),
                           omega, reinterpret_cast<const cf*>(h0), dp, reinterpret_cast<cf*>(dq),
                           reinterpret_cast<cf*>(dgamma), domega, reinterpret_cast<cf*>(dh0), B, D, N, L, true,
                           static_cast<hipStream_t>(stream));
}

extern "C" int mega_cema_scan_bwd(const void* dy, const void* x, int dtype, const float* p,
                                  const float* log_q, const float* gamma, const float* omega,
                                  int64_t B, int64_t D, int64_t N, int64_t L, void* dx, float* dp,
                                  float* dq, float* dgamma, float* domega, void* stream) {
  return mega_cema_scan_bwd_state(dy, x, dtype, p, log_q, gamma, omega, nullptr, B, D, N, L, dx, dp, dq, dgamma,
                                  domega, nullptr, stream);
}

extern "C" int mega_cema_scan_bwd_wide(const void* dy, const void* x, const float* p, const float* log_q,
                                       const float* gamma, const float* omega, const float* h0, int64_t B,
                                       int64_t D, int64_t N, int64_t L, float* dx, int accumulate_dx, float* dp,
                                       float* dq, float* dgamma, float* domega, float* dh0, void* stream) {
  const char* who = "mega_cema_scan_bwd_wide";
  MEGA_CHECK_ARG(dy && x && p && log_q && gamma && dp && dq && dgamma && domega, "%s: null pointer", who);
  MEGA_CHECK_ARG(B >= 0 && D >= 0 && L >= 0, "%s: negative size", who);
  MEGA_CHECK_ARG(B * D <= 0x7fffffff, "%s: too many rows", who);
  if (!mega_cema_scan_bwd_supported(MEGA_BF16, N, L))
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: needs N <= 16 (N %lld, L %lld)", who,
                     (long long)N, (long long)L);
  if (B == 0 || D == 0) return MEGA_OK;
  MEGA_CHECK_ARG(dh0 == nullptr || h0 != nullptr, "%s: dh0 without h0", who);
  if (accumulate_dx && dx != nullptr)
    return bwd_for(2, rows_of(B * D, L, h0 != nullptr, {dy, x, dx}))(dy, x, dx, p, reinterpret_cast<const cf*>(log_q), reinterpret_cast<const cf*>(gamma),
                         omega, reinterpret_cast<const cf*>(h0), dp, reinterpret_cast<cf*>(dq),
                         reinterpret_cast<cf*>(dgamma), domega, reinterpret_cast<cf*>(dh0), B, D, N, L, true,
                         static_cast<hipStream_t>(stream));
  return bwd_for(1, rows_of(B * D, L, h0 != nullptr, {dy, x, dx}))(dy, x, dx, p, reinterpret_cast<const cf*>(log_q), reinterpret_cast<const cf*>(gamma),
                       omega, reinterpret_cast<const cf*>(h0), dp, reinterpret_cast<cf*>(dq),
                       reinterpret_cast<cf*>(dgamma), domega, reinterpret_cast<cf*>(dh0), B, D, N, L, true,
                       static_cast<hipStream_t>(stream));
}

extern "C" int64_t mega_cema_layer_scan_sets(int64_t B, int64_t D, int64_t L) {
  Lines ln;
  int64_t slots = 0;
  if (B < 1 || D < 1 || L < 1 || bwd_lines(B, D, L, false, kWhole, &ln, &slots) != MEGA_OK) return 0;
  return ln.groups / ln.D;
}

extern "C" int mega_cema_layer_scan_bwd(const void* dy, const void* x, const float* p, const float* log_q,
                                        const float* gamma, const float* omega, int64_t B, int64_t D, int64_t N,
                                        int64_t L, void* dx, int dx_mode, float* dp, float* dq, float* dgamma,
                                        float* domega, void* stream) {
  const char* who = "mega_cema_layer_scan_bwd";
  MEGA_CHECK_ARG(dy && x && p && log_q && gamma && dp && dq && dgamma && domega, "%s: null pointer", who);
  MEGA_CHECK_ARG(B >= 1 && D >= 1 && B * D <= 0x7fffffff, "%s: bad sizes", who);
  MEGA_CHECK_ARG(dx_mode >= 0 && dx_mode <= 3 && (dx != nullptr || dx_mode == 1), "%s: bad dx", who);
  if (!mega_cema_scan_bwd_supported(MEGA_BF16, N, L))
    return set_error(MEGA_ERR_UNSUPPORTED, "%s: needs N <= 16 (N %lld, L %lld)", who, (long long)N, (long long)L);
  return bwd_for(dx_mode, rows_of(B * D, L, false, {dy, x, dx}))(dy, x, dx, p, reinterpret_cast<const cf*>(log_q), reinterpret_cast<const cf*>(gamma), omega, nullptr, dp,
            reinterpret_cast<cf*>(dq), reinterpret_cast<cf*>(dgamma), domega, nullptr, B, D, N, L, false,
            static_cast<hipStream_t>(stream));
}
