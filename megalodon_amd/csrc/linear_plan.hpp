// Which tiles the linear layers' products run in (attention.hip): sizes in, a laid-out launch out.  Plain C++.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/megalodon_hip.h"
#include "gemm_params.hpp"

namespace mega {

enum { kForward, kInputGrad, kWeightGrad };

// The tiles of the `count` problems of a launch (sizes along the axis they lie side by side on), in tiles of T.
inline void lay_out(GemmParams& q, int kind, int count, const int64_t* sizes, int T) {
  const auto tiles = [&](int64_t n) { return static_cast<int>((n + T - 1) / T); };
  q.start[0] = q.start[1] = 0x7fffffff;
  if (kind != kInputGrad || q.op_b[0] == nullptr) q.seg_start[0] = 0x7fffffff;
  if (kind != kInputGrad || q.op_b[1] == nullptr) q.seg_start[1] = 0x7fffffff;
  int along = tiles(sizes[0]);
  for (int i = 1; i < count; ++i) {
    q.start[i - 1] = along;
    q.size[i - 1] = static_cast<int>(sizes[i]);
    along += tiles(sizes[i]);
  }
  q.mt_count = kind == kWeightGrad ? along : tiles(q.M);
  q.nt_count = kind == kForward ? along : tiles(q.N);
  q.per_batch = q.items = q.mt_count * q.nt_count;
  q.full = q.items, q.cut = 0;
}

// Time of a launch in us by what was measured (1000 to 32768 tokens, layers of 1024 to 11008).  A tile of 256 takes longer
// for 32 k the more of the chip works (the clock falls: forward 0.45 us alone, 0.80 with every CU busy); tiles of 128 run
// two to a CU, each pair as long as two one after the other; every round of tiles starts and ends in a few us.
//
// Where the last round holds few tiles, they are cut along k, a part for a workgroup, and another launch adds up the parts (0.12
// us for each part of 256 KB written and read, 14 us for two launches).  2 x 11008 x 4096, us whole / cut: 1531 tokens (516 tiles)
// 278 / 235, 2100 (774) 351 / 332, 3000 (1032) 477 / 435, 9000 (3096) 1345 / 1288; the parts of few tiles are read by 32
// workgroups of a wave each (eight of four waves: 19.6 us for 32 parts, so under 10).  Tiles that fill more than half a round stay
// whole: there is no second workgroup for each.
inline double estimate_cut(GemmParams& q, double slabs, int cus) {
  const int grid = std::max(cus / kXcds, 1) * kXcds, left = q.items % grid, full = q.items - left;
  const auto round = [&](double tiles, double k) { return k * (0.45 + 0.35 * tiles / grid) + 5; };
  const double whole = full / grid * round(grid, slabs) + 3;
  double best = whole + (left > 0 ? round(left, slabs) : 0);
  for (int cut = 2; cut <= 8 && left > 0 && left * cut <= grid && slabs >= 16 * cut; ++cut) {
    const double t = whole + round(left * cut, slabs / cut) + 0.12 * left * cut + 14;
    if (t < best) best = t, q.full = full, q.cut = cut;
  }
  return best;
}
inline double estimate(GemmParams& q, int kind, int T, int cus) {
  const double slabs = (q.K + kSlab - 1) / kSlab, rounds = (q.items + cus - 1) / cus, load = q.items / (rounds * cus);
  if (T == kTile) {
    if (kind == kForward && q.split_ok) return estimate_cut(q, slabs, cus);
    if (kind == kWeightGrad) return rounds * (slabs * (0.40 + 0.36 * load) + 1) + 2;
    if (kind == kForward) return rounds * (slabs * (0.45 + 0.35 * load) + 5) + 3;
    return rounds * (slabs * (0.42 + 0.37 * load) + 5) + 2;
  }
  if (kind == kWeightGrad) {
    // Tiles for half of the CUs or fewer are cut along the tokens, as forward products are.  us, whole / cut: 4096 tokens, 2048 x
    // 1024 (128 tiles) 28.5 / 26.8, 1024 x 1024 28.4 / 23.9, 512 x 512 22.4 / 20.5; 8192 tokens 51 / 40 and (512 x 512)
    // 50 / 26; 32768 tokens 187 / 127, 191 / 72, 186 / 41.
    double best = rounds * slabs * 0.23 + 3;
    for (int cut = 2; q.split_ok && cut <= 16 && q.items * cut <= cus && slabs >= 16 * cut; ++cut) {
      const double t = slabs / cut * 0.23 + 0.03 * q.items * cut + 7;
      if (t < best) best = t, q.full = 0, q.cut = cut;
    }
    return best;
  }
  if (kind == kForward) {
    // A row or two of tiles read their weights from memory, not from an L2 that others have filled: 0.40 us a slab.  As many as
    // leave half of the CUs idle are cut along k as well, down to what streaming the weights takes.  us, library / whole / cut: 16
    // tokens, 1024 + 8192 + 4096 x 4096 60 / 45 / 33; 100 tokens 61 / 53 / 38, 512 + 4096 + 2048 x 2048 64 / 28 / 21.
    const double slab = q.mt_count <= 2 ? 0.40 : 0.255, stream = 2.0 * q.nt_count * T * q.K / 4.0e6;
    double best = rounds * (slabs * slab + 1.3) + 3;
    for (int cut = 2; q.split_ok && cut <= 8 && q.items * cut <= cus && slabs >= 16 * cut; ++cut) {
      const double t = std::max(slabs / cut * slab, stream) + 0.03 * q.items * cut * std::min(q.M, T) / T + 9;
      if (t < best) best = t, q.full = 0, q.cut = cut;
    }
    return best;
  }
  return rounds * (slabs * 0.27 + 1) + 3;
}

// Lays the tiles out in the size that is expected to be faster; its time.
inline double plan(GemmParams& q, int kind, int count, const int64_t* sizes, int cus, bool* small) {
  GemmParams l = q;
  lay_out(l, kind, count, sizes, kTile);
  lay_out(q, kind, count, sizes, kSmall);
  const double tl = estimate(l, kind, kTile, cus), ts = estimate(q, kind, kSmall, cus);
  *small = ts <= tl;
  if (!*small) q = l;
  return std::min(ts, tl);
}

// The part of a launch's problems that is problem i alone.
inline GemmParams one_of(const GemmParams& q, int kind, int i, int64_t size) {
  GemmParams o = q;
  if (kind == kForward) {
    if (i > 0) o.B = q.op[i - 1], o.C = q.out[i - 1], o.bias = q.bias_of[i - 1];
    o.N = (int)size;
    o.ldc = size;
  } else {
    if (i > 0) o.A = q.op[i - 1], o.C = q.out[i - 1];
    o.M = (int)size;
    o.lda = size;
  }
  return o;
}
// The time of `count` problems in one launch, or one launch after the other where that is shorter (*apart).
inline double plan_group(const GemmParams& q, int kind, int count, const int64_t* sizes, int cus, bool* apart) {
  GemmParams g = q;
  bool small;
  const double together = plan(g, kind, count, sizes, cus, &small);
  *apart = false;
  if (count == 1) return together;
  double sum = 0;
  for (int i = 0; i < count; ++i) {
    GemmParams o = one_of(q, kind, i, sizes[i]);
    sum += plan(o, kind, 1, sizes + i, cus, &small);
  }
  *apart = sum < 1.05 * together;  // (at equal rounds of tiles: 2 x 11008 x 4096, 32768 tokens, 4280 us apart, 4384 together)
  return std::min(sum, together);
}

// A call's products as the planning functions take them: sizes, no operands.
inline GemmParams linear_sizes(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out) {
  GemmParams q{};
  q.M = static_cast<int>(kind == kWeightGrad ? n_out[0] : tokens);
  q.N = static_cast<int>(kind == kForward ? n_out[0] : n_in);
  q.K = static_cast<int>(kind == kForward ? n_in : kind == kWeightGrad ? tokens : 0);
  for (int i = 0; kind == kInputGrad && i < count; ++i) q.K += static_cast<int>(n_out[i]);
  q.split_ok = 1;
  return q;
}
// Whether the layers of an input gradient lie behind each other along k of one product, in tiles of 128: one rounding, and dx
// is neither read again nor launched for again.  us, one after the other / so: 4096 tokens, 256 + 2048 + 1024 x 1024 50 / 32,
// 2 x 2752 x 1024 59 / 50; 4084 tokens, 512 + 4096 + 2048 x 2048 140 / 114; 500 tokens of the first 41 / 26.  Where tiles of
// 256 are the faster ones, one after the other, each onto the sum so far.
inline bool joined_along_k(int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  GemmParams all = linear_sizes(kInputGrad, tokens, n_in, count, n_out);
  bool small;
  plan(all, kInputGrad, 1, &n_in, cus, &small);
  return small;
}
// The time of a call, of all of its launches: the estimate that its tiles were chosen by, put right where that is known to be off.
// - Forward, up to 128 tokens, weights of 64 MB and more: they are read at 5.4 TB/s, 0.65 of the estimate's time in the mean; above 200
//   MB, which the memory-side cache no longer holds, only by tiles that are cut along k (three layers of 284 MB, uncut, 99 us).
// - Forward, a layer alone that fills one round with tiles of 128: 0.30 us a slab where the estimate has 0.255 (1344 tokens, 2560 ->
//   2752 31 us for 25).
// - Input gradients one after the other: each onto the sum so far, read and written again (two layers of 512: 1226 tokens, 8192
//   inputs, 46 us for 35; 19663 tokens, 512 inputs, 45 for 35).
inline double linear_time(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  bool apart, small;
  double time = 0;
  if (kind != kInputGrad) {
    GemmParams q = linear_sizes(kind, tokens, n_in, count, n_out);
    time = plan_group(q, kind, count, n_out, cus, &apart);
    if (kind == kForward && tokens <= 128) {
      double weights = 0;
      for (int i = 0; i < count; ++i) weights += 2.0 * n_in * n_out[i];
      if (weights > 200e6) plan(q, kind, count, n_out, cus, &small);
      return weights >= 64e6 && (weights <= 200e6 || (!apart && q.cut > 0)) ? std::min(time, weights / 5.4e6 + 5) : time;
    }
    if (kind == kForward && count == 1) {
      plan(q, kind, 1, n_out, cus, &small);
      if (small && q.cut == 0 && q.mt_count > 2 && q.items <= cus) time *= 1.13;
    }
    return time;
  }
  const int n = joined_along_k(tokens, n_in, count, n_out, cus) ? count : 1;
  for (int i = 0; i < count; i += n)
    time += plan_group(linear_sizes(kind, tokens, n_in, n, n_out + i), kind, 1, &n_in, cus, &apart) + (i > 0 ? 2.0 * tokens * n_in / 2.2e6 : 0);
  return time;
}

// What a product's launch refuses, or null.  (The contiguous reduction axis of forward and input gradient comes in slabs of 64.)
inline const char* linear_refuses(int kind, int dtype, int64_t tokens, int64_t n_in, int count, const int64_t* n_out) {
  if (dtype != MEGA_BF16 && dtype != MEGA_F16) return "bfloat16 or float16 tensors";
  if (count < 1 || count > 3 || n_out == nullptr) return "one to three layers";
  const int64_t in = kind == kForward ? 64 : 8, out = kind == kInputGrad ? 64 : 8;
  if (tokens < 1 || n_in < in || n_in % in != 0 || tokens >= (1 << 30) / n_in) return "bad sizes";
  for (int i = 0; i < count; ++i)
    if (n_out[i] < out || n_out[i] % out != 0 || tokens >= (1 << 30) / n_out[i] || n_in >= (1 << 30) / n_out[i]) return "bad sizes";
  return nullptr;
}

// The time in us of a general library's product of x (tokens, n_in) and a layer (n_out, n_in), forward or the input gradient: the
// smaller of two estimates, and no less than its host path (`host`) or than reading the weights for few tokens takes.
// One is the mean rate of products of so many terms, in PFLOP/s; widths off the multiples of 1024 cost it a quarter up to some 2^39.
// The other is what the tiles allow.  The library's are up to 256 x 256, in as many rounds as they need, by as many workgroups as
// divide them evenly; where none does, tiles are cut along k between workgroups, which costs about 1.3 tiles.  PFLOP/s of 4096
// -> 11008: 2500 tokens (430 tiles, two rounds of 215) 1.42, 5000 (four of 215) 1.46, 4096 (688) 0.92, 3500 (602) 0.90; 6912 -> 2560:
// 12000 (two of 235) 1.58, 16384 (640) 1.02.  For up to two rounds it looks for a tile that fits, then takes 256 x 256.  Widths off
// 256 cost up to two rounds 20 % and more rounds 10.
inline double library_time(int kind, int64_t tokens, int64_t n_in, int64_t n_out, int cus, double host) {
  const double products = static_cast<double>(tokens) * n_in * n_out;
  const double rate = kind == kInputGrad ? 1.1 : products > 0x1p39 ? 1.5 : products < 0x1p33 ? 1.0 : n_out % 1024 == 0 ? 1.4 : 1.1;
  const double mean = 2e-9 * products / rate + (kind == kInputGrad ? 10 : 8);
  const int rows = static_cast<int>(tokens), cols = static_cast<int>(kind == kInputGrad ? n_in : n_out);
  const double k = static_cast<double>(kind == kInputGrad ? n_out : n_in);
  const auto in_tiles = [&](int m, int n) {
    const double root = std::sqrt(m * n / 65536.0), tile = 1.2 / 64 * k * root * std::sqrt(root) + 6;  // (area to 3/4)
    const int tiles = (rows + m - 1) / m * ((cols + n - 1) / n), rounds = (tiles + cus - 1) / cus;
    return (tiles % rounds == 0 ? static_cast<double>(rounds) : static_cast<double>(tiles) / cus + 1.3) * tile + 3;
  };
  double even = in_tiles(256, 256);
  const bool fitted = (rows + 255) / 256 * ((cols + 255) / 256) <= 2 * cus;
  constexpr int kShapes[][2] = {{256, 192}, {256, 160}, {256, 128}, {192, 128}, {160, 128}, {128, 128}, {128, 64}, {64, 64}};
  for (int i = 0; fitted && i < 8; ++i) even = std::min({even, in_tiles(kShapes[i][0], kShapes[i][1]), in_tiles(kShapes[i][1], kShapes[i][0])});
  if (cols % 256 != 0) even *= fitted ? 1.2 : 1.1;
  const double stream = kind == kForward && tokens <= 256 ? 2.0 * n_in * n_out / 5.9e6 + 1 : 0;  // (64 to 380 MB, 1 to 64 tokens)
  return std::max({host, stream, std::min(mean, even)});
}

// Whether the launch is expected to be faster than the library's products, one call a layer (sizes that linear_refuses lets pass).
inline bool linear_takes(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  if (kind == kWeightGrad) {
    // Both operands run across the reduction axis, the library's slowest layout: this kernel is ahead at nearly every size (us,
    // library / here): 4096 tokens, 256 + 2048 + 1024 x 1024 91 / 30, 2 x 2752 x 1024 85 / 58, 2 x 5504 x 2048 174 / 166, 11008 x 4096
    // 380 / 281; 4084 tokens, 2048 x 5504 106 / 82; 1531, 4096 x 11008 174 / 122; 32768, 3328 x 1024 595 / 280, 1024 x 1024 198 / 72,
    // 512 x 512 152 / 41, 64 x 64 169 / 31.  Of 640 measured (300 to 32768 tokens, layers and groups of 768 to 13824) four are 3 to 16 %
    // slower, all of 24000 tokens and more: 32768, 2560 x 6912 1290 / 1490.  Of 88 of 1 to 300 tokens (512 x 512 to 13824 x 5120; from
    // 19 / 6, the library's host path, to 92 / 70) three are 4 to 15 % slower, matrices of 64 MB and more from 64 or 128 tokens: 64,
    // 8192 x 4096 20 / 23.
    return true;
  }
  for (int i = 0; kind == kInputGrad && i < count; ++i)
    if (static_cast<double>(tokens) * n_in * n_out[i] > 0x1p35) return false;  // goes through a transposed copy of W there
  const double here = linear_time(kind, tokens, n_in, count, n_out, cus);
  // Of 3128 forward products and input gradients, alone and in groups (300 to 32768 tokens, layers of 512 to 13824, widths on and
  // off 256), this takes 806: 24 of them are more than 3 % slower than the library's calls (1.10 in the mean, the worst 1.35), the
  // others 1.39 times as fast in the mean.  By the mean rate alone it took 1059, 193 of them slower (1.13 in the mean).  us, library /
  // here: 4096 tokens, 256 + 2048 + 1024 x 1024 60 / 33, 2 x 2752 x 1024 71 / 61, 2 x 5504 x 2048 181 / 165, 2 x 11008 x 4096 800 / 585;
  // left to the library: 2 x 11008 x 4096 of 1250 tokens 167 / 204, of 2500 317 / 374, of 5000 616 / 666.
  // (After what linear_time puts right, of 11556 that it takes of 44454 drawn, 1 to 32768 tokens, 146 are more than 3 % slower, 1.09 in
  // the mean, the worst 1.26; the time of all 0.52 of the library's in the mean.  Before, 1296 of 28872 were, the worst 1.62.)
  // Its host path is 18 us a call, more than many small products take.  A single layer of few tokens is up to 3 us above its
  // estimate here, so it has to be ahead by as much (us, library / here: 16 tokens, 5504 -> 2048 18.5 / 21.1, 512 tokens, 2752 ->
  // 1024 18.4 / 20.1; 16 tokens, 1024 -> 1024 18.3 / 9.7); several take less (384 tokens, 2 x 5504 x 2048 39.3 / 29.7, estimate 38).
  const double host = count == 1 ? 17 : 20;
  if (here <= 1.02 * host * count) return true;  // (nothing takes it less: spares the host its estimate, up to 1 us a call)
  double library = 0;
  for (int i = 0; i < count; ++i) library += library_time(kind, tokens, n_in, n_out[i], cus, host);
  return here <= 1.02 * library;  // (large tiles here take 2 to 5 % less than their estimate)
}

// The memory for the parts of cut tiles.
inline int64_t linear_workspace_bytes(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  const GemmParams q = linear_sizes(kind, tokens, n_in, count, n_out);
  bool apart, small;
  plan_group(q, kind, count, n_out, cus, &apart);
  int64_t values = 0;
  for (int i = 0; i < (apart ? count : 1); ++i) {
    GemmParams o = apart ? one_of(q, kind, i, n_out[i]) : q;
    plan(o, kind, apart ? 1 : count, apart ? n_out + i : n_out, cus, &small);
    const int64_t tile = small ? kSmall : kTile;
    values = std::max(values, static_cast<int64_t>(o.items - o.full) * o.cut * tile * tile);
  }
  return values * static_cast<int64_t>(sizeof(float));
}

}  // namespace mega
