// The tiles and the choice of the linear layers' products (linear_plan.hpp), for the CPU.  Built by
// tests/test_linear_plan_cpu.py with g++.
#include "../../megalodon_amd/csrc/linear_plan.hpp"

using namespace mega;

extern "C" int emu_linear_takes(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  return linear_takes(kind, tokens, n_in, count, n_out, cus);
}

extern "C" double emu_linear_time(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  return linear_time(kind, tokens, n_in, count, n_out, cus);
}

// the tile of a call's products: 128 or 256, 0 where its layers run in tiles of either
extern "C" int emu_linear_tile(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  const GemmParams q = linear_sizes(kind, tokens, n_in, count, n_out);
  bool apart = false, small = false;
  int tile = -1;
  const auto with = [&](GemmParams o, int n, const int64_t* sizes) {
    plan(o, kind, n, sizes, cus, &small);
    const int t = small ? kSmall : kTile;
    tile = tile < 0 || tile == t ? t : 0;
  };
  if (kind == kInputGrad) {
    const int n = joined_along_k(tokens, n_in, count, n_out, cus) ? count : 1;
    for (int i = 0; i < count; i += n) with(linear_sizes(kind, tokens, n_in, n, n_out + i), 1, &n_in);
    return tile;
  }
  plan_group(q, kind, count, n_out, cus, &apart);
  for (int i = 0; i < (apart ? count : 1); ++i) with(apart ? one_of(q, kind, i, n_out[i]) : q, apart ? 1 : count, apart ? n_out + i : n_out);
  return tile;
}

extern "C" int emu_linear_joined(int, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  return joined_along_k(tokens, n_in, count, n_out, cus);
}

extern "C" double emu_linear_library(int kind, int64_t tokens, int64_t n_in, int count, const int64_t* n_out, int cus) {
  double time = 0;
  for (int i = 0; i < count; ++i) time += library_time(kind, tokens, n_in, n_out[i], cus, 20);
  return time;
}
