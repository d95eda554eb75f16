// Register-resident FFT engine for the causal convolution (gfx950).
//
// Plain C++17 with no HIP dependency in the algorithmic part, so the same
// phases run under g++ in a CPU harness (threads emulated one after another,
// LDS as an ordinary array) and under hipcc inside the kernel.
//
// Problem.  y = irfft(rfft(a, 2N) * rfft(b, 2N))[:L] with N = 2^n >= L
// (megalodon/modules/fused_ops/fftconv.py:30-50).  Both real sequences are
// split into even/odd samples, z[n] = s[2n] + i s[2n+1], n < M = N/2 (the
// upper half of the N-point z sequence is the zero padding).  The N-point
// spectrum Z[r] then splits by parity of r into two independent M-point
// transforms that never need the zeros:
//     Z[2a]   = FFT_M(z[n])[a]            ("even half", H = 0)
//     Z[2a+1] = FFT_M(z[n] W_N^n)[a]      ("odd half",  H = 1)
// With E = (Z[r] + conj Z[N-r])/2 (spectrum of the even samples) and
// O = -i (Z[r] - conj Z[N-r])/2 (odd samples) the product is the polyphase
// identity   Ey = Ea Eb + W_N^r Oa Ob,   Oy = Ea Ob + Oa Eb,   Zy = Ey + i Oy,
// and only the first M outputs of the inverse are needed (the [:L] crop):
//     zy[n] = IFFT_M(Zy[2a])[n] + W_N^-n IFFT_M(Zy[2a+1])[n].
//
// Engine.  One workgroup of T = M/32 lanes transforms one M-point half with 32
// complex points per lane in registers: M = 32 * 32 * R3 (R3 = M/1024 in
// {2,4,8,16}); pass 1 radix-32 over the top digit, LDS exchange, pass 2
// radix-32, LDS exchange, pass 3 radix-R3 (32/R3 butterflies per lane).  All are
// decimation in time: a pass takes its inputs' twiddles into its butterflies, six
// fused operations each, where twiddles of its own between the passes had to be
// formed (136 operations) and multiplied in (124) beside butterflies of four to eight.  The
// residues handled by one lane in pass 3 are chosen in conjugate pairs
// (c, 1024-c) / (c, 1023-c), so both Z[r] and Z[N-r] of every bin sit in the
// same lane and the pointwise stage needs no further exchange.  The inverse is
// the mirror image, the same transforms on swapped re/im.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define MEGA_HD __host__ __device__ __forceinline__
#else
#define MEGA_HD inline
#endif

namespace mega {
namespace fftc {

struct c32 {
  float x, y;
};
template <int V>
struct alignas(4 * V) fvec {
  float v[V];
};

// cos/sin of 2*pi*k/64
constexpr float kC64[64] = {
    1.f, 0.99518472667219693f, 0.98078528040323043f, 0.95694033573220882f, 0.92387953251128674f, 0.88192126434835505f, 0.83146961230254524f, 0.77301045336273699f, 0.70710678118654757f, 0.63439328416364549f, 0.55557023301960229f, 0.47139673682599781f, 0.38268343236508984f, 0.29028467725446233f, 0.19509032201612833f, 0.09801714032956077f,
    0.f, -0.098017140329560645f, -0.19509032201612819f, -0.29028467725446216f, -0.38268343236508973f, -0.4713967368259977f, -0.55557023301960196f, -0.63439328416364538f, -0.70710678118654746f, -0.77301045336273699f, -0.83146961230254535f, -0.88192126434835494f, -0.92387953251128674f, -0.95694033573220882f, -0.98078528040323043f, -0.99518472667219682f,
    -1.f, -0.99518472667219693f, -0.98078528040323043f, -0.95694033573220894f, -0.92387953251128685f, -0.88192126434835505f, -0.83146961230254546f, -0.7730104533627371f, -0.70710678118654768f, -0.63439328416364593f, -0.55557023301960218f, -0.47139673682599786f, -0.38268343236509034f, -0.29028467725446244f, -0.19509032201612866f, -0.098017140329560451f,
    0.f, 0.09801714032956009f, 0.1950903220161283f, 0.29028467725446205f, 0.38268343236509f, 0.47139673682599759f, 0.55557023301960184f, 0.6343932841636456f, 0.70710678118654735f, 0.77301045336273666f, 0.83146961230254524f, 0.88192126434835483f, 0.92387953251128652f, 0.95694033573220882f, 0.98078528040323032f, 0.99518472667219693f};
constexpr float kS64[64] = {
    0.f, 0.098017140329560604f, 0.19509032201612825f, 0.29028467725446233f, 0.38268343236508978f, 0.47139673682599764f, 0.55557023301960218f, 0.63439328416364549f, 0.70710678118654746f, 0.77301045336273699f, 0.83146961230254524f, 0.88192126434835494f, 0.92387953251128674f, 0.95694033573220894f, 0.98078528040323043f, 0.99518472667219682f,
    1.f, 0.99518472667219693f, 0.98078528040323043f, 0.95694033573220894f, 0.92387953251128674f, 0.88192126434835505f, 0.83146961230254546f, 0.7730104533627371f, 0.70710678118654757f, 0.63439328416364549f, 0.55557023301960218f, 0.47139673682599786f, 0.38268343236508989f, 0.29028467725446239f, 0.19509032201612861f, 0.098017140329560826f,
    0.f, -0.09801714032956059f, -0.19509032201612836f, -0.29028467725446211f, -0.38268343236508967f, -0.47139673682599764f, -0.55557023301960196f, -0.63439328416364527f, -0.70710678118654746f, -0.77301045336273666f, -0.83146961230254524f, -0.88192126434835494f, -0.92387953251128652f, -0.95694033573220882f, -0.98078528040323032f, -0.99518472667219693f,
    -1.f, -0.99518472667219693f, -0.98078528040323043f, -0.95694033573220894f, -0.92387953251128663f, -0.88192126434835505f, -0.83146961230254546f, -0.77301045336273688f, -0.70710678118654768f, -0.63439328416364593f, -0.55557023301960218f, -0.47139673682599792f, -0.38268343236509039f, -0.2902846772544625f, -0.19509032201612872f, -0.098017140329560506f};

constexpr float kRsqrt2 = 0.70710678118654752f;

template <int BITS>
constexpr int bitrev(int x) {
  int r = 0;
  for (int i = 0; i < BITS; ++i) r |= ((x >> i) & 1) << (BITS - 1 - i);
  return r;
}
constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x >> 1); }

// v *= W_R^k with W_R = exp(-2 pi i / R), k in [0, R) known at compile time after unrolling
template <int R>
MEGA_HD void mul_w(float& xr, float& xi, int k) {
  const int q = (k * (64 / R)) & 63;
  const float c = kC64[q], s = kS64[q];  // W = c - i s
  const float r = xr * c + xi * s;
  const float i = xi * c - xr * s;
  xr = r;
  xi = i;
}

MEGA_HD float fma1(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
MEGA_HD c32 cmulv(c32 a, c32 b) { return c32{fma1(-a.y, b.y, a.x * b.x), fma1(a.y, b.x, a.x * b.y)}; }
MEGA_HD c32 csqv(c32 a) { return c32{fma1(-a.y, a.y, a.x * a.x), (a.x + a.x) * a.y}; }

// (a, b) <- (a + w b, a - w b): the sum in four fused operations, the difference as 2 a - sum in two.  With the
// twiddle in front of the butterfly its product costs no instruction of its own; behind it (decimation in
// frequency) a butterfly and its twiddle are eight.
MEGA_HD void butterfly(float& ar, float& ai, float& br, float& bi, c32 w) {
  const float tr = fma1(-bi, w.y, fma1(br, w.x, ar)), ti = fma1(bi, w.x, fma1(br, w.y, ai));
  br = fma1(2.f, ar, -tr);
  bi = fma1(2.f, ai, -ti);
  ar = tr;
  ai = ti;
}
// the same with w = 1 and w = -i
MEGA_HD void butterfly1(float& ar, float& ai, float& br, float& bi) {
  const float r = br, i = bi;
  br = ar - r;
  bi = ai - i;
  ar += r;
  ai += i;
}
MEGA_HD void butterfly_mi(float& ar, float& ai, float& br, float& bi) {
  const float r = br, i = bi;
  br = ar - i;
  bi = ai + r;
  ar += i;
  ai -= r;
}

// Stage R of a transform of N natural-order inputs v[j] with a twiddle of its own on each, v[j] w^j: butterflies of blocks
// of R outputs, w here the power N / R of that twiddle.  After the last stage, R = N, output k stands at position
// bitrev(k).  The twiddles of a stage are w times roots of unity, two butterflies to a product (its quarter turn is free).
template <int N, int R>
MEGA_HD void stage_w(float* re, float* im, c32 w) {
  constexpr int S = N / R, B = ilog2(R) - 1, Q = R >= 4 ? R / 4 : 1;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    c32 t = w;
    if (i > 0) mul_w<R>(t.x, t.y, i);
#pragma unroll
    for (int b = 0; b < S; ++b) {
      const int p = b + 2 * S * bitrev<B>(i);
      butterfly(re[p], im[p], re[p + S], im[p + S], t);
      if (R >= 4) {
        const int q = b + 2 * S * bitrev<B>(i + R / 4);
        butterfly(re[q], im[q], re[q + S], im[q + S], c32{t.y, -t.x});
      }
    }
  }
}
// ... with w = W_X^(N / R), known at compile time (X = 0: w = 1)
template <int N, int R, int X = 0>
MEGA_HD void stage(float* re, float* im) {
  constexpr int S = N / R, B = ilog2(R) - 1;
#pragma unroll
  for (int i = 0; i < R / 2; ++i) {
    const int turn = i * (64 / R) + (X ? S * (64 / (X ? X : 64)) : 0);  // in 64ths, below 32
#pragma unroll
    for (int b = 0; b < S; ++b) {
      const int p = b + 2 * S * bitrev<B>(i);
      if (turn == 0) butterfly1(re[p], im[p], re[p + S], im[p + S]);
      else if (turn == 16) butterfly_mi(re[p], im[p], re[p + S], im[p + S]);
      else butterfly(re[p], im[p], re[p + S], im[p + S], c32{kC64[turn], -kS64[turn]});
    }
  }
}
// sum_j v[j] W_N^(j k), or with X sum_j v[j] W_X^j W_N^(j k): output k at position bitrev(k)
template <int N, int X = 0>
MEGA_HD void transform(float* re, float* im) {
  stage<N, 2, X>(re, im);
  if constexpr (N >= 4) stage<N, 4, X>(re, im);
  if constexpr (N >= 8) stage<N, 8, X>(re, im);
  if constexpr (N >= 16) stage<N, 16, X>(re, im);
  if constexpr (N >= 32) stage<N, 32, X>(re, im);
}
// sum_j v[j] w^j W_N^(j k), N <= 16, from w alone
template <int N>
MEGA_HD void transform_w(float* re, float* im, c32 w) {
  const c32 w2 = csqv(w), w4 = csqv(w2), w8 = csqv(w4);
  if constexpr (N == 2) {
    stage_w<N, 2>(re, im, w);
  } else if constexpr (N == 4) {
    stage_w<N, 2>(re, im, w2);
    stage_w<N, 4>(re, im, w);
  } else if constexpr (N == 8) {
    stage_w<N, 2>(re, im, w4);
    stage_w<N, 4>(re, im, w2);
    stage_w<N, 8>(re, im, w);
  } else {
    stage_w<N, 2>(re, im, w8);
    stage_w<N, 4>(re, im, w4);
    stage_w<N, 8>(re, im, w2);
    stage_w<N, 16>(re, im, w);
  }
}

// The same sums for inputs that stand at bitrev(j) * S: output k at position k * S.
template <int R, int S>
MEGA_HD void dit(float* re, float* im) {
  if constexpr (R > 1) {
    constexpr int H = R / 2;
    dit<H, S>(re, im);
    dit<H, S>(re + H * S, im + H * S);
#pragma unroll
    for (int i = 0; i < H; ++i) {
      float *ar = re + i * S, *ai = im + i * S, *br = ar + H * S, *bi = ai + H * S;
      if (i == 0) butterfly1(*ar, *ai, *br, *bi);
      else if (4 * i == R) butterfly_mi(*ar, *ai, *br, *bi);
      else butterfly(*ar, *ai, *br, *bi, c32{kC64[i * (64 / R)], -kS64[i * (64 / R)]});
    }
  }
}

// The transform of 32 with a lane's own twiddle, sum_j v[j] w^j W_32^(j k), from w, w^4 and w^16.
struct Powers {
  c32 w1, w4, w16;
};
MEGA_HD void transform32_w(float* re, float* im, const Powers& w) {
  stage_w<32, 2>(re, im, w.w16);
  stage_w<32, 4>(re, im, csqv(w.w4));
  stage_w<32, 8>(re, im, w.w4);
  stage_w<32, 16>(re, im, csqv(w.w1));
  stage_w<32, 32>(re, im, w.w1);
}
// ... and over odd frequencies, P[n] = sum_a u[a] z_n^(2a+1) with z_n = z W_64^n and w = z^2: even and odd a apart, P[n] = z_n E +
// z_n^3 O and P[n + 16] = -i (z_n E - z_n^3 O).  P[n] ends at position 2*bitrev4(n) for n < 16 and 1 + 2*bitrev4(n-16)
// otherwise.
MEGA_HD void odd_last(float& er, float& ei, float& orr, float& oi, c32 z1, c32 z3) {
  const float pr = fma1(-ei, z1.y, er * z1.x), pi = fma1(ei, z1.x, er * z1.y);
  const float tr = fma1(-oi, z3.y, fma1(orr, z3.x, pr)), ti = fma1(oi, z3.x, fma1(orr, z3.y, pi));
  orr = fma1(2.f, pi, -ti);
  oi = fma1(-2.f, pr, tr);
  er = tr;
  ei = ti;
}
MEGA_HD void odd_transform32_w(float* re, float* im, const Powers& w, c32 z) {
  stage_w<32, 2>(re, im, w.w16);
  stage_w<32, 4>(re, im, csqv(w.w4));
  stage_w<32, 8>(re, im, w.w4);
  stage_w<32, 16>(re, im, csqv(w.w1));
  const c32 z3 = cmulv(z, w.w1);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int p = 2 * bitrev<4>(i);
    c32 a = z, b = z3;
    if (i > 0) {
      mul_w<64>(a.x, a.y, i);
      mul_w<64>(b.x, b.y, 3 * i);
    }
    odd_last(re[p], im[p], re[p + 1], im[p + 1], a, b);
  }
}
MEGA_HD constexpr int shifted_dit32_pos(int n) {
  return n < 16 ? 2 * bitrev<4>(n) : 1 + 2 * bitrev<4>(n - 16);
}

// ---------------------------------------------------------------------------
template <int LOGM>
struct Cfg {
  static constexpr int M = 1 << LOGM;       // complex points of one half
  static constexpr int T = M / 32;          // lanes per workgroup
  static constexpr int R3 = M / 1024;       // radix of the third pass
  static constexpr int NSLOT = 16 / R3;     // residue pairs per lane
  static constexpr int LD1 = T + R3;        // row pitch of exchange 1 (floats)
  // Exchange 2: pitch of a residue's R3 values and how many of them one access moves.  Four at once
  // need no padding (both directions then run over consecutive banks), which is also what lets four
  // workgroups of M = 4096 share a compute unit's LDS; six apart in pairs, only three fit.
  static constexpr int LD2 = R3 + (R3 >= 8 ? 2 : 0);
  static constexpr int V2 = R3 == 4 ? 4 : 2;
  static constexpr int PLANE = (32 * LD1 > 1024 * LD2) ? 32 * LD1 : 1024 * LD2;
  static constexpr int TABLE = 4 * T + 3 * R3 + 192 + 2048;  // c32 entries
  static_assert(LOGM >= 11 && LOGM <= 14, "M must be 2048..16384");
};

// Per-lane twiddles for one M (device memory, W_X^k = exp(-2 pi i k / X)).
// The inputs of a pass have the twiddles w^j of one w that depends only on the lane; a transform of 32 takes
// its first, fourth and sixteenth power.
//   k1[t]       = W_M^t                      inverse pass 1 (t = lane)
//   kz[t]       = W_N^t                      inverse pass 1, odd half
//   k2e[a2]     = W_M^(R3 a2)                forward pass 2, even half
//   k2o[a2]     = W_N^(R3 (2 a2 + 1))        forward pass 2, odd half
//   ki2[n0]     = W_T^n0                     inverse pass 2
//   pw[h*1024 + c] = W_N^(2c + h)            forward pass 3 (residue c), pointwise twiddle
struct Tables {
  const Powers *k1, *k2e, *k2o, *ki2;
  const c32 *kz, *pw;
};

template <int LOGM>
MEGA_HD Tables make_tables(const c32* base) {
  using C = Cfg<LOGM>;
  Tables tb;
  tb.k1 = reinterpret_cast<const Powers*>(base);
  tb.k2e = tb.k1 + C::T;
  tb.k2o = tb.k2e + 32;
  tb.ki2 = tb.k2o + 32;
  tb.kz = reinterpret_cast<const c32*>(tb.ki2 + C::R3);
  tb.pw = tb.kz + C::T;
  return tb;
}

// Host-side fill of the table (float64 trigonometry, exact argument reduction).
template <int LOGM>
inline void fill_tables(c32* out) {
  using C = Cfg<LOGM>;
  const double N = 2.0 * C::M;
  auto w = [](double num, double den) {
    const double fr = __builtin_fmod(num, den) / den;
    const double a = -6.283185307179586476925286766559 * fr;
    return c32{static_cast<float>(__builtin_cos(a)), static_cast<float>(__builtin_sin(a))};
  };
  c32* p = out;
  auto powers = [&](double num, double den) {
    for (int e = 1; e <= 16; e *= 4) *p++ = w(e * num, den);
  };
  for (int t = 0; t < C::T; ++t) powers(t, C::M);
  for (int a2 = 0; a2 < 32; ++a2) powers(static_cast<double>(C::R3) * a2, C::M);
  for (int a2 = 0; a2 < 32; ++a2) powers(static_cast<double>(C::R3) * (2 * a2 + 1), N);
  for (int n0 = 0; n0 < C::R3; ++n0) powers(n0, C::T);
  for (int t = 0; t < C::T; ++t) *p++ = w(t, N);
  for (int h = 0; h < 2; ++h)
    for (int c = 0; c < 1024; ++c) *p++ = w(2.0 * c + h, N);
}

// table[idx] addressed as uniform base + 32-bit unsigned byte offset (lets the
// compiler use the scalar-base addressing form instead of a 64-bit lane address)
#if defined(__HIP_DEVICE_COMPILE__)
// (said to be global memory: of a base that came through `launder` the compiler does not know it, and a flat load counts
// among the LDS operations too, so that every wait for one waits for the other)
#define MEGA_FFT_GLOBAL __attribute__((address_space(1)))
#else
#define MEGA_FFT_GLOBAL
#endif
MEGA_HD c32 ldc(const c32* base, unsigned idx) {
  const auto* const p = (const MEGA_FFT_GLOBAL char*)(base) + idx * 8u;
  const auto* const f = (const MEGA_FFT_GLOBAL float*)(p);
  return c32{f[0], f[1]};
}
MEGA_HD Powers ldc(const Powers* base, unsigned idx) {
  const auto* const p = (const MEGA_FFT_GLOBAL char*)(base) + idx * 24u;
  const auto* const f = (const MEGA_FFT_GLOBAL float*)(p);
  return Powers{c32{f[0], f[1]}, c32{f[2], f[3]}, c32{f[4], f[5]}};
}

// residues of slot s for half H
template <int H>
MEGA_HD void slot_residues(int s, int& c0, int& c1) {
  if (H == 0) {
    c0 = s;
    c1 = s == 0 ? 512 : 1024 - s;
  } else {
    c0 = s;
    c1 = 1023 - s;
  }
}

// ------------------------------ forward ------------------------------------
// Every pass takes its inputs' twiddles with it (transform32_w); pass 1's are known at compile time.
// Pass 1 on natural-order input v[j] = z[t + T j]; output a2 at position bitrev5(a2).
template <int H>
MEGA_HD void fwd_first(float* re, float* im) {
  transform<32, H == 0 ? 0 : 64>(re, im);
}
template <int LOGM>
MEGA_HD void x1_write(const float* re, const float* im, int t, float* lre, float* lim) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int a2 = 0; a2 < 32; ++a2) {
    const int pos = bitrev<5>(a2);
    lre[a2 * C::LD1 + t] = re[pos];
    lim[a2 * C::LD1 + t] = im[pos];
  }
}
// lane (a2', n0') = (t / R3, t % R3) gathers n1 = 0..31
template <int LOGM>
MEGA_HD void x1_read(float* re, float* im, int t, const float* lre, const float* lim) {
  using C = Cfg<LOGM>;
  const int a2p = t / C::R3, n0p = t % C::R3;
#pragma unroll
  for (int n1 = 0; n1 < 32; ++n1) {
    re[n1] = lre[a2p * C::LD1 + n1 * C::R3 + n0p];
    im[n1] = lim[a2p * C::LD1 + n1 * C::R3 + n0p];
  }
}
// Pass 2 behind the twiddles W_M^(R3 n1 a2') (even) or W_N^(R3 n1 (2 a2' + 1)); what their share of n0' is goes to pass 3.
// A pass needs its twiddles with its first butterfly, so the kernels ask for them a pass ahead.
template <int LOGM, int H>
MEGA_HD Powers second_twiddles(int t, const Tables& tb) {
  return ldc(H == 0 ? tb.k2e : tb.k2o, t / Cfg<LOGM>::R3);
}
MEGA_HD void fwd_second(float* re, float* im, const Powers& w) { transform32_w(re, im, w); }
// element (a2', a1, n0') goes to residue c = a2' + 32 a1
template <int LOGM>
MEGA_HD void x2_write(const float* re, const float* im, int t, float* lre, float* lim) {
  using C = Cfg<LOGM>;
  const int a2p = t / C::R3, n0p = t % C::R3;
#pragma unroll
  for (int a1 = 0; a1 < 32; ++a1) {
    const int pos = bitrev<5>(a1);
    const int c = a2p + 32 * a1;
    lre[c * C::LD2 + n0p] = re[pos];
    lim[c * C::LD2 + n0p] = im[pos];
  }
}
// register index of (slot u, member w, element e)
template <int LOGM>
MEGA_HD constexpr int sidx(int u, int w, int e) {
  return (u * 2 + w) * Cfg<LOGM>::R3 + e;
}
template <int LOGM, int H>
MEGA_HD void x2_read(float* re, float* im, int t, const float* lre, const float* lim) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int u = 0; u < C::NSLOT; ++u) {
    int c[2];
    slot_residues<H>(t + C::T * u, c[0], c[1]);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      using V = fvec<C::V2>;
      const V* pr = reinterpret_cast<const V*>(lre + c[w] * C::LD2);
      const V* pi = reinterpret_cast<const V*>(lim + c[w] * C::LD2);
#pragma unroll
      for (int e = 0; e < C::R3 / C::V2; ++e) {
        const V a = pr[e], b = pi[e];
#pragma unroll
        for (int i = 0; i < C::V2; ++i) {
          re[sidx<LOGM>(u, w, C::V2 * e + i)] = a.v[i];
          im[sidx<LOGM>(u, w, C::V2 * e + i)] = b.v[i];
        }
      }
    }
  }
}
// pass 3: bin a0 of (u, w) ends at register sidx(u, w, bitrev(a0)); the twiddles of residue c are W_M^(n0 c) (even) or
// W_N^(n0 (2 c + 1))
template <int LOGM>
struct Thirds {
  c32 w[Cfg<LOGM>::NSLOT];  // of c0 of the lane's slots
};
template <int LOGM, int H>
MEGA_HD Thirds<LOGM> third_twiddles(int t, const Tables& tb) {
  Thirds<LOGM> th;
#pragma unroll
  for (int u = 0; u < Cfg<LOGM>::NSLOT; ++u) th.w[u] = ldc(tb.pw, H * 1024 + t + Cfg<LOGM>::T * u);
  return th;
}
template <int LOGM, int H>
MEGA_HD void fwd_third(float* re, float* im, int t, const Thirds<LOGM>& th) {
  constexpr int R3 = Cfg<LOGM>::R3, q = 64 / R3;
#pragma unroll
  for (int u = 0; u < Cfg<LOGM>::NSLOT; ++u) {
    const c32 w0 = th.w[u];
    // the partner's: c1 = 1024 - c0 or (2 c1 + 1) = 2048 - (2 c0 + 1), W_M^1024 = W_R3; 512 beside 0
    c32 w1{fma1(-kS64[q], w0.y, kC64[q] * w0.x), fma1(-kC64[q], w0.y, -kS64[q] * w0.x)};
    if (H == 0 && u == 0) {
      const bool self = t == 0;
      w1.x = self ? kC64[q / 2] : w1.x;
      w1.y = self ? -kS64[q / 2] : w1.y;
    }
    transform_w<R3>(re + sidx<LOGM>(u, 0, 0), im + sidx<LOGM>(u, 0, 0), w0);
    transform_w<R3>(re + sidx<LOGM>(u, 1, 0), im + sidx<LOGM>(u, 1, 0), w1);
  }
}

// ------------------------------ pointwise ----------------------------------
// One conjugate pair of bins (r, r' = N - r).  (ar, ai) = Za[r], (apr, api) =
// Za[r'], same for b; w = W_N^r.  Returns Zy[r] in (ar, ai), Zy[r'] in (apr, api).
MEGA_HD void pair_product(float& ar, float& ai, float& apr, float& api, float br, float bi,
                          float bpr, float bpi, float wr, float wi) {
  // 2E = Z[r] + conj Z[r'];  2O = -i (Z[r] - conj Z[r'])
  const float ear = ar + apr, eai = ai - api;
  const float oar = ai + api, oai = apr - ar;
  const float ebr = br + bpr, ebi = bi - bpi;
  const float obr = bi + bpi, obi = bpr - br;
  // t = Oa Ob
  const float tr = oar * obr - oai * obi, ti = oar * obi + oai * obr;
  // Ey = Ea Eb + w t
  float eyr = ear * ebr - eai * ebi, eyi = ear * ebi + eai * ebr;
  eyr += wr * tr - wi * ti;
  eyi += wr * ti + wi * tr;
  // Oy = Ea Ob + Oa Eb
  const float oyr = ear * obr - eai * obi + oar * ebr - oai * ebi;
  const float oyi = ear * obi + eai * obr + oar * ebi + oai * ebr;
  ar = eyr - oyi;
  ai = eyi + oyr;
  apr = eyr + oyi;
  api = oyr - eyi;
}

// a (in flight) times parked b, both in pass-3 register layout; result Zy in a.
template <int LOGM, int H>
MEGA_HD void pointwise(float* re, float* im, const float* bre, const float* bim, int t,
                       const Tables& tb) {
  using C = Cfg<LOGM>;
  constexpr int R3 = C::R3;
  constexpr int LR = ilog2(R3);
#pragma unroll
  for (int u = 0; u < C::NSLOT; ++u) {
    const int s = t + C::T * u;
    const bool self = (H == 0) && (u == 0) && (s == 0);
    if (!self) {
      const c32 pw = ldc(tb.pw, H * 1024 + s);  // W_N^(2 c0 + H)
#pragma unroll
      for (int a0 = 0; a0 < R3; ++a0) {
        const int i0 = sidx<LOGM>(u, 0, bitrev<LR>(a0));
        const int i1 = sidx<LOGM>(u, 1, bitrev<LR>(R3 - 1 - a0));
        float wr = pw.x, wi = pw.y;
        if (a0 != 0) mul_w<R3>(wr, wi, a0);
        pair_product(re[i0], im[i0], re[i1], im[i1], bre[i0], bim[i0], bre[i1], bim[i1], wr, wi);
      }
    } else if (u == 0) {
      // slot 0 of the even half: residues 0 and 512 pair with themselves
      float nr[2 * R3], ni[2 * R3];
      const c32 pw512 = ldc(tb.pw, 512);  // W_N^1024
#pragma unroll
      for (int w = 0; w < 2; ++w) {
#pragma unroll
        for (int a0 = 0; a0 < R3; ++a0) {
          const int pa = w == 0 ? (R3 - a0) % R3 : R3 - 1 - a0;
          const int i0 = sidx<LOGM>(0, w, bitrev<LR>(a0));
          const int i1 = sidx<LOGM>(0, w, bitrev<LR>(pa));
          float wr = w == 0 ? 1.f : pw512.x, wi = w == 0 ? 0.f : pw512.y;
          if (a0 != 0) mul_w<R3>(wr, wi, a0);
          float ar = re[i0], ai = im[i0], apr = re[i1], api = im[i1];
          pair_product(ar, ai, apr, api, bre[i0], bim[i0], bre[i1], bim[i1], wr, wi);
          nr[w * R3 + a0] = ar;
          ni[w * R3 + a0] = ai;
        }
      }
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int a0 = 0; a0 < R3; ++a0) {
          re[sidx<LOGM>(0, w, bitrev<LR>(a0))] = nr[w * R3 + a0];
          im[sidx<LOGM>(0, w, bitrev<LR>(a0))] = ni[w * R3 + a0];
        }
    }
  }
}

// ------------------------------ inverse ------------------------------------
// pass 3': inverse radix-R3 over a0 (swapped re/im: a conjugated twiddle is a plain one there)
template <int LOGM>
MEGA_HD void inv_third(float* re, float* im) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int g = 0; g < 2 * C::NSLOT; ++g) dit<C::R3, 1>(im + g * C::R3, re + g * C::R3);
}
template <int LOGM, int H>
MEGA_HD void ix2_write(const float* re, const float* im, int t, float* lre, float* lim) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int u = 0; u < C::NSLOT; ++u) {
    int c[2];
    slot_residues<H>(t + C::T * u, c[0], c[1]);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      using V = fvec<C::V2>;
      V* pr = reinterpret_cast<V*>(lre + c[w] * C::LD2);
      V* pi = reinterpret_cast<V*>(lim + c[w] * C::LD2);
#pragma unroll
      for (int e = 0; e < C::R3 / C::V2; ++e) {
        V a, b;
#pragma unroll
        for (int i = 0; i < C::V2; ++i) {
          a.v[i] = re[sidx<LOGM>(u, w, C::V2 * e + i)];
          b.v[i] = im[sidx<LOGM>(u, w, C::V2 * e + i)];
        }
        pr[e] = a;
        pi[e] = b;
      }
    }
  }
}
template <int LOGM>
MEGA_HD void ix2_read(float* re, float* im, int t, const float* lre, const float* lim) {
  using C = Cfg<LOGM>;
  const int a2p = t / C::R3, n0p = t % C::R3;
#pragma unroll
  for (int a1 = 0; a1 < 32; ++a1) {
    const int c = a2p + 32 * a1;
    re[a1] = lre[c * C::LD2 + n0p];
    im[a1] = lim[c * C::LD2 + n0p];
  }
}
// pass 2': inverse radix-32 over a1 -> n1 at bitrev5(n1), behind the twiddles conj W_T^(n0' a1)
template <int LOGM>
MEGA_HD Powers inv_second_twiddles(int t, const Tables& tb) {
  return ldc(tb.ki2, t % Cfg<LOGM>::R3);
}
MEGA_HD void inv_second(float* re, float* im, const Powers& w) { transform32_w(im, re, w); }
template <int LOGM>
MEGA_HD void ix1_write(const float* re, const float* im, int t, float* lre, float* lim) {
  using C = Cfg<LOGM>;
  const int a2p = t / C::R3, n0p = t % C::R3;
#pragma unroll
  for (int n1 = 0; n1 < 32; ++n1) {
    const int pos = bitrev<5>(n1);
    lre[a2p * C::LD1 + n1 * C::R3 + n0p] = re[pos];
    lim[a2p * C::LD1 + n1 * C::R3 + n0p] = im[pos];
  }
}
template <int LOGM>
MEGA_HD void ix1_read(float* re, float* im, int t, const float* lre, const float* lim) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int a2 = 0; a2 < 32; ++a2) {
    re[a2] = lre[a2 * C::LD1 + t];
    im[a2] = lim[a2 * C::LD1 + t];
  }
}
// pass 1': inverse radix-32 over a2, behind the twiddles conj W_M^(t a2) or conj W_N^(t (2 a2 + 1)); zy[t + T n2] ends at
// register out_pos<H>(n2)
struct Firsts {
  Powers w;
  c32 z;
};
template <int H>
MEGA_HD Firsts inv_first_twiddles(int t, const Tables& tb) {
  return Firsts{ldc(tb.k1, t), H == 0 ? c32{1.f, 0.f} : ldc(tb.kz, t)};
}
template <int H>
MEGA_HD void inv_first(float* re, float* im, const Firsts& f) {
  if (H == 0) transform32_w(im, re, f.w);
  else odd_transform32_w(im, re, f.w, f.z);
}
template <int H>
MEGA_HD constexpr int out_pos(int n2) {
  return H == 0 ? bitrev<5>(n2) : shifted_dit32_pos(n2);
}

// How a launch shares out its rows: how many rows of a channel a group takes, chosen for the shortest line of
// transforms, in halves of one, that a workgroup slot gets (5 for a pair of rows, 3 for a row alone).  `bound`: a channel's sum
// stands in its groups' slots, so that there may be no more groups than slots, unless a group has the channel to itself.
// Of the sizes that leave as many groups to a channel the smallest is the shortest, so only these are looked at, 2 sqrt(B)
// at most: for the three launches of a step on 10^6 rows of one channel, 24 ms of the host's time size by size, 0.08 so.
inline int64_t group_rows(int64_t B, int64_t D, int64_t slots, int pair, bool bound) {
  int64_t best = B, least = -1;
  for (int64_t nb = 1;;) {
    const int64_t shares = (B + nb - 1) / nb, groups = D * shares;
    if (!bound || shares == 1 || groups <= slots) {
      const int64_t cost = (groups + slots - 1) / slots * (pair == 2 ? nb / 2 * 5 + nb % 2 * 3 : nb * 3);
      if (least < 0 || cost < least) best = nb, least = cost;
    }
    if (shares == 1) return best;
    nb = (B + shares - 2) / (shares - 1);  // the smallest that leaves fewer
  }
}

}  // namespace fftc
}  // namespace mega
