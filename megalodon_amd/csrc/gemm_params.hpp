// One launch of the product kernels (attention.hip), as its host side lays it out.
#pragma once

#include <cstdint>

namespace mega {

constexpr int kTile = 256;     // workgroup tile (M and N)
constexpr int kSmall = 128;    // the same where 256 leaves compute units idle
constexpr int kSlab = 32;      // k elements staged per iteration
constexpr int kXcds = 8;       // accelerator dies, each with a private L2

// C[m][n] = alpha * sum_k A(m, k) B(n, k); element (m, k) of an operand sits at
// [m * ld + k], or at [k * ld + m] when the operand is flagged k-major
struct GemmParams {
  const uint16_t* A;
  const uint16_t* B;
  uint16_t* C;
  int M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sa0, sa1, sb0, sb1, sc0, sc1;  // batch z = z0 * nh + z1 -> offset z0*s0 + z1*s1
  int nh;
  float alpha;
  // Causal structure with rows = queries r, columns = keys c, c <= r + off
  // (off = L2 - L1 >= 0, the length of a key/value prefix):
  int tri_out;  // 1: tiles wholly above that diagonal are skipped (left unwritten)
  int k_mode;   // 0: all k; 1: m = queries, k = keys: k < (mt+1)*256 + off, rounded up to a slab;
                // 2: m = keys, k = queries: k >= mt*256 - off, rounded down to a slab
  int off;
  // persistent schedule (filled in by the launcher): work items of equal weight,
  // walked by gridDim.x workgroups
  int mt_count, nt_count;  // tiles along m and n
  int per_batch;           // work items per batch index
  int items;               // per_batch * batch
  int snake;               // 128-wide tiles of unequal length: all of them run at once
  int ta, tb;   // operand is k-major: element (m, k) at [k * ld + m]
  int kvb;      // rows of k that a k-major B holds when K has been rounded up behind them (0: all K); A holds
                // zeros there, and zeros stand in for those rows of B (0 times an infinity would be NaN)
  int ms;       // rows of C to store when M has been rounded up (0: all M)
  // Linear layers (LIN): C = A B^T + bias + add, with up to three problems in one launch.  Side by side along n (two
  // k-contiguous operands: layers of one input) they differ in B, C, ldc, bias and N; along m (two k-major operands: their
  // weight gradients) in A, lda, C and M.  Tiles mt (nt) >= start[i] belong to problem i + 1.
  const uint16_t* bias;    // N values or null
  const uint16_t* add;     // summand of C's layout or null
  const uint16_t* op[2];
  uint16_t* out[2];
  const uint16_t* bias_of[2];
  int size[2], start[2];
  // ... and an input gradient whose layers lie behind each other along k: k slabs >= seg_start[i] (of kSlab) are those of
  // op[i] and op_b[i], rows of A size[i] apart there
  const uint16_t* op_b[2];
  int seg_start[2];
  int kva;      // as kvb, for a k-major A (LIN: rows behind it are not there; else they hold zeros)
  // CUT: items full .. items - 1, fewer than there are CUs, are cut along k into `cut` parts; float32 sums of part i
  // of item full + r at parts + (r cut + i) T T, as the waves hold them (linear_parts_kernel adds them up).
  int full, cut;
  float* parts;
  int split_ok;  // (the launcher's: there is memory for the parts)
  int n_group;  // plain schedule: tiles numbered n fastest inside bands of n_group column tiles, then m,
                // then band (0: one band) -- the 32 tiles an XCD works on at a time then share fewer
                // distinct operand blocks (4 x 8 instead of 2 x 16 of a 16-column problem)
};

}  // namespace mega
