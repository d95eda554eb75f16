// The transform path of the causal convolution: row kernels, their tables and scratch, one transform size to a
// translation unit (fftconv_m11.hip .. fftconv_m14.hip: M = 2^11 .. 2^14 complex points).
#pragma once

#include "common.hpp"
#include "fftconv_core.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace mega {

// ------------------------------ tables --------------------------------------
constexpr int kFftDevices = 16;
constexpr int kFftScratch = 4;  // scratch blocks per device and size before streams start taking turns
constexpr int kSlotParts = 3;   // parts of a workgroup's scratch slot, 2 M floats each; a part of all slots is one allocation
struct Scratch {
  float* part[kSlotParts];  // null behind the parts that a block has
};
struct StreamScratch {
  hipStream_t stream;  // the stream whose launches used the block last
  Scratch parts;
  hipEvent_t done;     // recorded behind the last launch that used the block
  uint64_t tick;       // when that was
  bool pinned;         // used under stream capture: the graph's replays own the block from then on
};
struct TableCache {
  fftc::c32* ptr[kFftDevices][4] = {};
  int slots[kFftDevices][4] = {};
  // Launches on different streams of a device may overlap, and a workgroup's
  // slot is picked by its index alone, so a stream gets a block of its own --
  // up to kFftScratch of them per device and size.  A further stream takes
  // over the block that has been idle longest and first waits (on the device,
  // through the block's event) for the last launch that used it.  Blocks used
  // under stream capture are never handed on.
  std::vector<StreamScratch> scratch[kFftDevices][4];
  uint64_t tick = 0;
  std::mutex mu;
};
extern TableCache fft_tables;  // fftconv.hip

// Rows of a size, by the unit that has it: mode 0 and 1 as fftconv_kernel has them.
template <int LOGM>
int fftconv_rows(int dtype, int mode, const void* a, const void* b, void* out, int64_t B, int64_t D, int64_t L, int flip,
                 const float* omega, hipStream_t stream);
// Makes a size's tables and the stream's scratch block.
template <int LOGM>
int fftconv_tables(hipStream_t stream);

namespace {
// ------------------------------ row I/O --------------------------------------
template <int DT>
__device__ __forceinline__ float ld(const void* base, int64_t i) {
  return Elem<DT>::load(static_cast<const typename Elem<DT>::type*>(base) + i);
}
template <int DT>
__device__ __forceinline__ void st(void* base, int64_t i, float v) {
  Elem<DT>::store(static_cast<typename Elem<DT>::type*>(base) + i, v);
}
// uniform base + 32-bit unsigned byte offset (scalar-base addressing form)
template <typename V>
__device__ __forceinline__ V gld(const void* base, unsigned byte_off) {
  return *reinterpret_cast<const V*>(static_cast<const char*>(base) + byte_off);
}
template <typename V>
__device__ __forceinline__ void gst(void* base, unsigned byte_off, V v) {
  *reinterpret_cast<V*>(static_cast<char*>(base) + byte_off) = v;
}

// A pair of adjacent elements as one 32/64-bit access.
template <int DT> struct Pair;
typedef float float2_any __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32_any __attribute__((aligned(2)));
// at any element (by a cast to the typedef itself: as a template's argument, of gld, it would lose its alignment)
__device__ __forceinline__ uint32_t load_u32_any(const void* base, unsigned off) {
  return *reinterpret_cast<const u32_any*>(static_cast<const char*>(base) + off);
}
__device__ __forceinline__ void store_u32_any(void* base, unsigned off, uint32_t v) {
  *reinterpret_cast<u32_any*>(static_cast<char*>(base) + off) = v;
}
template <> struct Pair<MEGA_F32> {
  using type = float2;
  static __device__ __forceinline__ type load_any(const void* base, unsigned off) {
    const float2_any v = *reinterpret_cast<const float2_any*>(static_cast<const char*>(base) + off);
    return make_float2(v.x, v.y);
  }
  static __device__ __forceinline__ void store_any(void* base, unsigned off, type v) {
    *reinterpret_cast<float2_any*>(static_cast<char*>(base) + off) = float2_any{v.x, v.y};
  }
  static __device__ __forceinline__ void unpack(type v, float& lo, float& hi) { lo = v.x; hi = v.y; }
  static __device__ __forceinline__ type pack(float lo, float hi) { return make_float2(lo, hi); }
};
template <> struct Pair<MEGA_BF16> {
  using type = uint32_t;
  static __device__ __forceinline__ type load_any(const void* base, unsigned off) { return load_u32_any(base, off); }
  static __device__ __forceinline__ void store_any(void* base, unsigned off, type v) { store_u32_any(base, off, v); }
  static __device__ __forceinline__ void unpack(type v, float& lo, float& hi) {
    lo = __uint_as_float(v << 16);
    hi = __uint_as_float(v & 0xffff0000u);
  }
  static __device__ __forceinline__ type pack(float lo, float hi) { return pack_bf16x2(lo, hi); }
};
template <> struct Pair<MEGA_F16> {
  using type = uint32_t;
  static __device__ __forceinline__ type load_any(const void* base, unsigned off) { return load_u32_any(base, off); }
  static __device__ __forceinline__ void store_any(void* base, unsigned off, type v) { store_u32_any(base, off, v); }
  static __device__ __forceinline__ void unpack(type v, float& lo, float& hi) {
    lo = f16_bits_to_float(static_cast<uint16_t>(v & 0xffffu));
    hi = f16_bits_to_float(static_cast<uint16_t>(v >> 16));
  }
  static __device__ __forceinline__ type pack(float lo, float hi) {
    return static_cast<uint32_t>(float_to_f16_bits(lo)) |
           (static_cast<uint32_t>(float_to_f16_bits(hi)) << 16);
  }
};

}  // namespace

#ifdef MEGA_FFTCONV_LOGM
namespace {

using namespace fftc;

// Workgroups of a transform size that share a compute unit: the kernel's time is the latency of its
// exchanges and barriers, so two waves per SIMD at every size, which is what the registers (32 complex
// points per lane and operand: 229-256 of 256) and the planes in LDS allow.  With one wave
// per SIMD below M = 16384 (and 330 registers) and the loads in branches, forward / backward in
// bfloat16 took 2 x 1024 rows of 3000: 152 / 348 us, now 51 / 138; of 8192: 226 / 479, now 95 / 198;
// 1024 rows of 16384: 236 / 485, now 115 / 219; of 32768: 440 / 891, now 246 / 502 (the last by the loads alone).
template <int LOGM>
constexpr int kPerCu = 1 << (14 - LOGM);

bool stream_is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return st != hipStreamCaptureStatusNone;
}

// Twiddle tables (one per device and transform size) and the per-workgroup
// scratch slots live for the life of the process.  They are made on first use,
// or ahead of time by mega_fftconv_prepare; making them allocates and, for the
// tables, synchronises the stream once, so that call cannot be captured into a
// graph.  A part of scratch is 2*M floats per resident workgroup (kPerCu of
// them per CU: 34 MB at every size); a block gets as many of the three as its launches have needed.
template <int LOGM>
int get_tables(hipStream_t stream, const c32** out, int* slots) {
  using C = Cfg<LOGM>;
  int dev = 0;
  MEGA_CHECK_HIP(hipGetDevice(&dev));
  MEGA_CHECK_ARG(dev >= 0 && dev < kFftDevices, "device index %d not supported", dev);
  std::lock_guard<std::mutex> lock(fft_tables.mu);
  c32*& slot = fft_tables.ptr[dev][LOGM - 11];
  if (slot == nullptr) {
    hipDeviceProp_t prop;
    MEGA_CHECK_HIP(hipGetDeviceProperties(&prop, dev));
    fft_tables.slots[dev][LOGM - 11] = prop.multiProcessorCount * kPerCu<LOGM>;
    c32* p = nullptr;
    MEGA_CHECK_HIP(hipMalloc(reinterpret_cast<void**>(&p), sizeof(c32) * C::TABLE));
    std::vector<c32> host(C::TABLE);
    fill_tables<LOGM>(host.data());
    hipError_t e = hipMemcpyAsync(p, host.data(), sizeof(c32) * C::TABLE, hipMemcpyHostToDevice, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) {
      (void)hipFree(p);
      return set_error(MEGA_ERR_HIP, "fftconv table init failed: %s", hipGetErrorString(e));
    }
    slot = p;
  }
  *out = slot;
  *slots = fft_tables.slots[dev][LOGM - 11];
  return MEGA_OK;
}

// The stream's scratch block, with `need` parts or more; under capture, where nothing can be allocated, with those that
// it has (*have).
template <int LOGM>
int get_scratch(hipStream_t stream, int need, Scratch* scratch, int* have) {
  using C = Cfg<LOGM>;
  int dev = 0;
  MEGA_CHECK_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(fft_tables.mu);
  std::vector<StreamScratch>& blocks = fft_tables.scratch[dev][LOGM - 11];
  StreamScratch* mine = nullptr;
  int open_blocks = 0;
  for (StreamScratch& s : blocks) {
    if (s.stream == stream) mine = &s;
    open_blocks += s.pinned ? 0 : 1;
  }
  const bool capturing = stream_is_capturing(stream);
  if (mine == nullptr && open_blocks >= kFftScratch && !capturing) {
    // take over the block that has been idle longest, behind its last launch
    for (StreamScratch& s : blocks)
      if (!s.pinned && (mine == nullptr || s.tick < mine->tick)) mine = &s;
    MEGA_CHECK_HIP(hipStreamWaitEvent(stream, mine->done, 0));
    mine->stream = stream;
  }
  const bool fresh = mine == nullptr;
  StreamScratch made{stream, {}, nullptr, 0, false};
  if (fresh) mine = &made;
  *have = 0;
  while (*have < kSlotParts && mine->parts.part[*have] != nullptr) ++*have;
  while (*have < need && (fresh || !capturing)) {
    const hipError_t e = hipMalloc(reinterpret_cast<void**>(&mine->parts.part[*have]), sizeof(float) * 2 * C::M * fft_tables.slots[dev][LOGM - 11]);
    if (e != hipSuccess) {
      mine->parts.part[*have] = nullptr;
      if (fresh)
        for (float* p : made.parts.part) (void)hipFree(p);
      return set_error(MEGA_ERR_HIP, "fftconv scratch: %s", hipGetErrorString(e));
    }
    ++*have;
  }
  if (fresh) {
    const hipError_t e = hipEventCreateWithFlags(&made.done, hipEventDisableTiming);
    if (e != hipSuccess) {
      for (float* p : made.parts.part) (void)hipFree(p);
      return set_error(MEGA_ERR_HIP, "fftconv scratch event: %s", hipGetErrorString(e));
    }
    blocks.push_back(made);
    mine = &blocks.back();
  }
  mine->tick = ++fft_tables.tick;
  if (capturing) mine->pinned = true;
  *scratch = mine->parts;
  return MEGA_OK;
}

// Marks the end of the launches that used `stream`'s scratch block, so that a
// later take-over can order itself behind them.  Not recorded under capture
// (the block is pinned there).
template <int LOGM>
int scratch_used(hipStream_t stream) {
  int dev = 0;
  MEGA_CHECK_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(fft_tables.mu);
  for (StreamScratch& s : fft_tables.scratch[dev][LOGM - 11])
    if (s.stream == stream && !s.pinned) MEGA_CHECK_HIP(hipEventRecord(s.done, stream));
  return MEGA_OK;
}

// The lane id, hidden from the optimiser: left alone it keeps the offsets of a row's 32 accesses in
// registers from its load to its store, across both halves (with two waves per SIMD: 74 spilled).
__device__ __forceinline__ int own_lane(int t) {
  asm volatile("" : "+v"(t));
  return t;
}

// z[n] = s[2n] + i s[2n+1] of the zero-padded (optionally reversed) row.  Every lane reads inside the
// row and takes zero for what lies behind it, so that the 32 loads stand in one piece without branches.
// A pair (s[2n], s[2n+1]) is one access addressed with a 32-bit offset from the wave-uniform row base.
// VEC: L is even and the row is pair-aligned.  Otherwise the pairs lie at any element, and of an odd L the last value is
// taken with the one in front of it (L >= 2).  (Element by element the loads had no registers to stand in together and were
// waited for one by one: 2 x 512 rows of 10001 bfloat16 forward and backward 403 us, 8 x 1024 of 2049 691.)
template <int LOGM, int DT, bool VEC>
__device__ __forceinline__ void load_row(float* re, float* im, const void* row, int L, bool flip,
                                         int lane) {
  using C = Cfg<LOGM>;
  const unsigned t = static_cast<unsigned>(own_lane(lane));
  const unsigned count = VEC ? static_cast<unsigned>(L) >> 1 : static_cast<unsigned>(L), last = count - 1u;
  const unsigned turn = flip ? ~0u : 0u, from = flip ? count : 0u;  // i or count - 1 - i
  if (VEC) {
    using P = typename Pair<DT>::type;
    P raw[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const unsigned n = t + C::T * j;
      raw[j] = gld<P>(row, (((n < last ? n : last) ^ turn) + from) * static_cast<unsigned>(sizeof(P)));
    }
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const bool in = t + C::T * j < count;
      float lo, hi;
      Pair<DT>::unpack(raw[j], lo, hi);
      re[j] = in ? (flip ? hi : lo) : 0.f;
      im[j] = in ? (flip ? lo : hi) : 0.f;
    }
  } else {
    using P = typename Pair<DT>::type;
    constexpr int kSize = sizeof(P) / 2;
    P raw[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int m = 2 * static_cast<int>(t + C::T * j), at = flip ? L - 2 - m : m;
      raw[j] = Pair<DT>::load_any(row, static_cast<unsigned>(max(0, min(at, L - 2)) * kSize));
    }
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int m = 2 * static_cast<int>(t + C::T * j);
      float lo, hi;
      Pair<DT>::unpack(raw[j], lo, hi);
      const bool alone = m + 1 == L;
      re[j] = m < L ? (flip != alone ? hi : lo) : 0.f;
      im[j] = m + 1 < L ? (flip ? lo : hi) : 0.f;
    }
  }
}

// out[2n] = re[j], out[2n+1] = im[j] for n = t + T j (reversed when flip);
// ACC adds to what is there (fp32 rows only).  With `res` non-null the stored
// value is out[m] + w * res[m] (res has the dtype and layout of the output row).
template <int LOGM, int DT, bool VEC, bool ACC>
__device__ __forceinline__ void store_row(const float* re, const float* im, void* row, int L,
                                          bool flip, int lane, const void* res = nullptr,
                                          float w = 0.f) {
  using C = Cfg<LOGM>;
  const int t = own_lane(lane);
  if (VEC) {
    using P = typename Pair<DT>::type;
    const unsigned half = static_cast<unsigned>(L) >> 1;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const unsigned n = static_cast<unsigned>(t) + C::T * j;
      if (n < half) {
        float lo = flip ? im[j] : re[j], hi = flip ? re[j] : im[j];
        const unsigned off = (flip ? half - 1u - n : n) * static_cast<unsigned>(sizeof(P));
        if (ACC) {
          float plo, phi;
          Pair<DT>::unpack(gld<P>(row, off), plo, phi);
          lo += plo;
          hi += phi;
        }
        if (res != nullptr) {
          float rlo, rhi;
          Pair<DT>::unpack(gld<P>(res, off), rlo, rhi);
          lo = fmaf(w, rlo, lo);
          hi = fmaf(w, rhi, hi);
        }
        gst<P>(row, off, Pair<DT>::pack(lo, hi));
      }
    }
  } else {
    using P = typename Pair<DT>::type;
    constexpr int kSize = sizeof(P) / 2;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int m = 2 * (t + C::T * j);
      if (m + 1 < L) {
        const unsigned off = static_cast<unsigned>(flip ? L - 2 - m : m) * kSize;
        float lo = flip ? im[j] : re[j], hi = flip ? re[j] : im[j];
        if (ACC) {
          float plo, phi;
          Pair<DT>::unpack(Pair<DT>::load_any(row, off), plo, phi);
          lo += plo;
          hi += phi;
        }
        if (res != nullptr) {
          float rlo, rhi;
          Pair<DT>::unpack(Pair<DT>::load_any(res, off), rlo, rhi);
          lo = fmaf(w, rlo, lo);
          hi = fmaf(w, rhi, hi);
        }
        Pair<DT>::store_any(row, off, Pair<DT>::pack(lo, hi));
      } else if (m < L) {
        const int o = flip ? 0 : m;
        const float r = ACC ? ld<DT>(row, o) + re[j] : re[j];
        st<DT>(row, o, res != nullptr ? fmaf(w, ld<DT>(res, o), r) : r);
      }
    }
  }
}

// Hides the table base from common-subexpression elimination / loop hoisting:
// twiddles are re-read from L1/L2 at each use instead of being kept live in
// registers across transforms (which would spill).
__device__ __forceinline__ Tables launder(Tables tb) {
  asm volatile("" : "+s"(tb.k1), "+s"(tb.k2e), "+s"(tb.k2o), "+s"(tb.ki2), "+s"(tb.kz), "+s"(tb.pw));
  return tb;
}

template <int LOGM, int H>
__device__ __forceinline__ void forward_half(float* re, float* im, int t, const Tables& tb0,
                                             float* lre, float* lim) {
  const Tables tb = launder(tb0);
  const Powers second = second_twiddles<LOGM, H>(t, tb);
  fwd_first<H>(re, im);
  __syncthreads();
  x1_write<LOGM>(re, im, t, lre, lim);
  __syncthreads();
  x1_read<LOGM>(re, im, t, lre, lim);
  const Thirds<LOGM> third = third_twiddles<LOGM, H>(t, tb);
  fwd_second(re, im, second);
  __syncthreads();
  x2_write<LOGM>(re, im, t, lre, lim);
  __syncthreads();
  x2_read<LOGM, H>(re, im, t, lre, lim);
  fwd_third<LOGM, H>(re, im, t, third);
}

template <int LOGM, int H>
__device__ __forceinline__ void inverse_half(float* re, float* im, int t, const Tables& tb0,
                                             float* lre, float* lim) {
  const Tables tb = launder(tb0);
  const Powers second = inv_second_twiddles<LOGM>(t, tb);
  inv_third<LOGM>(re, im);
  __syncthreads();
  ix2_write<LOGM, H>(re, im, t, lre, lim);
  __syncthreads();
  ix2_read<LOGM>(re, im, t, lre, lim);
  const Firsts first = inv_first_twiddles<H>(t, tb);
  inv_second(re, im, second);
  __syncthreads();
  ix1_write<LOGM>(re, im, t, lre, lim);
  __syncthreads();
  ix1_read<LOGM>(re, im, t, lre, lim);
  inv_first<H>(re, im, first);
}

// The lane's 32 values as they stand in its registers, to and from a part of the workgroup's scratch slot (2 M floats a part).
template <int LOGM>
__device__ __forceinline__ void keep(float* part, const float* re, const float* im, int t) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    gst<float>(part, (j * C::T + t) * 4u, re[j]);
    gst<float>(part, (C::M + j * C::T + t) * 4u, im[j]);
  }
}
template <int LOGM, bool ADD>
__device__ __forceinline__ void fetch(const float* part, float* re, float* im, int t) {
  using C = Cfg<LOGM>;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    const float a = gld<float>(part, (j * C::T + t) * 4u), b = gld<float>(part, (C::M + j * C::T + t) * 4u);
    re[j] = ADD ? re[j] + a : a;
    im[j] = ADD ? im[j] + b : b;
  }
}

// Has the lane's values worked out here.  Where branches follow (the product of spectra with its lane of self-paired residues, the
// stores at a row's end) the last butterflies are otherwise sunk into them, and both their operands stay in registers until then: pairs
// of rows spilled 15 to 49 beside k's spectrum (80 bytes a lane: 40 MiB that the runtime took at a first launch).  Forward, us, before / now: bfloat16
// 3 x 1024 rows of 4095 86 / 73, 4 x 1024 of 5001 166 / 145, 2 x 1024 of 8192 89 / 84, of 10001 190 / 169, of 12000 173 / 163, 2 x 512 of 16384 97 / 92;
// float32 86 / 72, 163 / 138, 94 / 81, 192 / 169, 179 / 175, 101 / 97.
__device__ __forceinline__ void settle(float* re, float* im) {
#pragma unroll
  for (int j = 0; j < 32; ++j) asm volatile("" : "+v"(re[j]), "+v"(im[j]));
}

// Back from a product of spectra.  Half 0 leaves its M outputs zy[t + T j] in `part`; half 1 adds them and has the
// sum in (re, im), zy[t + T j] at register j.  FULL: the registers hold k's spectrum too.
template <int LOGM, int H, bool FULL>
__device__ __forceinline__ void outputs(float* re, float* im, int t, const Tables& tb, float* lre, float* lim, float* part) {
  inverse_half<LOGM, H>(re, im, t, tb, lre, lim);
  float ore[32], oim[32];
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    ore[j] = re[out_pos<H>(j)];
    oim[j] = im[out_pos<H>(j)];
  }
  if (H == 1 && FULL) settle(ore, oim);
  if (H == 0) keep<LOGM>(part, ore, oim, t);
  else fetch<LOGM, true>(part, ore, oim, t);
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    re[j] = ore[j];
    im[j] = oim[j];
  }
}

// The rows of a channel that a workgroup takes: two at a time, which then share the transform of k (MODE 0) or the
// inverse transform of dk, whose spectrum is summed over them (MODE 1).  The kernels' time is mostly the transforms'
// arithmetic (75 to 77 % of the vector issue slots at M = 4096), so what counts is their number: 2.5 per row instead of 3.  In MODE 0
// k's spectrum then has to stay in registers to the row's end, which none of them leaves (one, of odd rows at M = 8192) since `settle`; at M = 16384 67
// to 76 would, and the rows go one by one (PAIR 1), as a channel's only row does.  One kernel for dx and dk, with dy's spectrum formed once (4
// transforms per row), spills 54 to 139 registers and takes 269 us where these two take 168.
// bfloat16, forward / backward in us: 2 x 1024 rows of 8192 97 / 194 -> 86 / 168, 4 x 1024 of 8190 181 / 385 -> 158 / 325; of
// channels whose rows now share out the chip for dk too: 8 x 256 of 8192 89 / 377 -> 82 / 169, 8 x 512 of 3001 120 / 541 -> 119 / 271
// (since, with twiddles inside the butterflies and odd rows' loads in pairs: forward alone 88, 148, 76, 80).
struct Rows {
  int B, D, L;
  int nb, groups;  // group g: channel g % D, rows g / D nb ..
};

// spectrum of a row's half H; SCALED: times 1 / (4 N) (E, O halves and the inverse), as one factor of every product is
template <int LOGM, int DT, bool VEC, int H, bool SCALED>
__device__ __forceinline__ void spectrum(float* re, float* im, const void* row, int L, bool flip, int t, const Tables& tb,
                                         float* lre, float* lim) {
  load_row<LOGM, DT, VEC>(re, im, row, L, flip, t);
  forward_half<LOGM, H>(re, im, t, tb, lre, lim);
  if (SCALED) {
    constexpr float scale = 1.0f / (8.0f * Cfg<LOGM>::M);
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      re[j] *= scale;
      im[j] *= scale;
    }
  }
}

// MODE 0: out[b,d,:] = conv(a[b,d,:], k[d,:]) (+ omega[d] a[b,d,:] when omega is given); `flip` reverses a on load and the
//         result on store (backward dx).  a, out have dtype DT; b is k, fp32.
// MODE 1: out[d,:] = sum_b reverse(conv(reverse(a[b,d,:]), x[b,d,:])), fp32 (backward dk); b is x.  `flip`: a channel's rows are
//         shared by several workgroups, whose sums stand in their slots.
template <int LOGM, int DT, int MODE, bool VEC, int H, int PAIR>
__device__ __forceinline__ void conv_half(const void* a, const void* b, void* out, const Rows& rows, int d, int b0, int n, bool add,
                                          int flip, const Tables& tb, float* lre, float* lim, const Scratch& scratch, const float* omega) {
  using C = Cfg<LOGM>;
  const int64_t pitch = static_cast<int64_t>(rows.L) * (DT == MEGA_F32 ? 4 : 2);
  float pre[32], pim[32];
  const int count = PAIR == 1 ? 1 : n;
  constexpr bool FULL = MODE == 0 && PAIR > 1;
  if (MODE == 0) {
    const int t = own_lane(threadIdx.x) & (C::T - 1);  // (restores the range so that offsets stay 32-bit)
    spectrum<LOGM, MEGA_F32, VEC, H, true>(pre, pim, static_cast<const float*>(b) + static_cast<int64_t>(d) * rows.L, rows.L, false, t, tb, lre, lim);
  }
#pragma unroll 1
  for (int i = 0; i < count; ++i) {
    const int t = own_lane(threadIdx.x) & (C::T - 1);
    const int64_t row = static_cast<int64_t>(b0 + i) * rows.D + d;
    const char* arow = static_cast<const char*>(a) + row * pitch;
    float re[32], im[32];
    if (MODE == 1) spectrum<LOGM, DT, VEC, H, true>(pre, pim, static_cast<const char*>(b) + row * pitch, rows.L, false, t, tb, lre, lim);
    spectrum<LOGM, DT, VEC, H, false>(re, im, arow, rows.L, MODE == 1 || flip != 0, t, tb, lre, lim);
    if (H == 0 && FULL) settle(re, im);
    pointwise<LOGM, H>(re, im, pre, pim, t, launder(tb));
    // the slot's parts: half 0's outputs; with pairs those of the second row, or (MODE 1) the spectrum so far; last a
    // shared channel's sum
    if (MODE == 1 && PAIR > 1) {
      if (i > 0) fetch<LOGM, true>(scratch.part[1], re, im, t);
      if (i + 1 < count) {
        keep<LOGM>(scratch.part[1], re, im, t);
        continue;
      }
    }
    outputs<LOGM, H, FULL>(re, im, t, tb, lre, lim, MODE == 0 && PAIR > 1 && i > 0 ? scratch.part[1] : scratch.part[0]);
    if (H == 1 && MODE == 0)
      store_row<LOGM, DT, VEC, false>(re, im, static_cast<char*>(out) + row * pitch, rows.L, flip != 0, t,
                                      omega != nullptr ? arow : nullptr, omega != nullptr ? omega[d] : 0.f);
    if (H == 1 && MODE == 1) {
      float* sum = flip ? scratch.part[PAIR] : static_cast<float*>(out) + static_cast<int64_t>(d) * rows.L;
      if (add) store_row<LOGM, MEGA_F32, VEC, true>(re, im, sum, rows.L, true, t);
      else store_row<LOGM, MEGA_F32, VEC, false>(re, im, sum, rows.L, true, t);
    }
  }
}
template <int LOGM, int DT, int MODE, bool VEC, int PAIR>
__global__ __launch_bounds__(Cfg<LOGM>::T, 2) void fftconv_kernel(
    const void* __restrict__ a, const void* __restrict__ b, void* __restrict__ out, const Rows rows, int flip,
    const c32* __restrict__ tab, const Scratch all, const float* __restrict__ omega) {
  extern __shared__ __align__(16) float lds[];
  float *lre = lds, *lim = lds + Cfg<LOGM>::PLANE;
  const Tables tb = make_tables<LOGM>(tab);
  const size_t slot = blockIdx.x * 2 * Cfg<LOGM>::M;  // (within a part; parts that the launch does not use are never touched)
  const Scratch scratch{{all.part[0] + slot, all.part[1] + slot, all.part[2] + slot}};
  for (int g = blockIdx.x; g < rows.groups; g += gridDim.x) {
    const int d = g % rows.D, first = g / rows.D * rows.nb, end = min(rows.B, first + rows.nb);
    for (int b0 = first; b0 < end; b0 += PAIR) {
      const int n = min(PAIR, end - b0);
      conv_half<LOGM, DT, MODE, VEC, 0, PAIR>(a, b, out, rows, d, b0, n, b0 > first, flip, tb, lre, lim, scratch, omega);
      conv_half<LOGM, DT, MODE, VEC, 1, PAIR>(a, b, out, rows, d, b0, n, b0 > first, flip, tb, lre, lim, scratch, omega);
    }
  }
}
// dk of channels whose rows several workgroups took, from their slots in order
__global__ __launch_bounds__(256) void split_sum_kernel(const float* __restrict__ sums, float* __restrict__ dk, const Rows rows, int slot) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(rows.D) * rows.L) return;
  const int d = static_cast<int>(i / rows.L), m = static_cast<int>(i % rows.L);
  float sum = 0.f;
  for (int g = d; g < rows.groups; g += rows.D) sum += sums[static_cast<int64_t>(g) * slot + m];
  dk[i] = sum;
}

Rows make_rows(int64_t B, int64_t D, int64_t L, int64_t nb) {
  return Rows{static_cast<int>(B), static_cast<int>(D), static_cast<int>(L), static_cast<int>(nb), static_cast<int>(D * ((B + nb - 1) / nb))};
}

template <int LOGM, int DT, int MODE, bool VEC, int PAIR>
int launch_rows(const void* a, const void* b, void* out, const Rows& rows, int flip, const float* omega, const c32* tab, const Scratch& scratch,
                int slots, hipStream_t stream) {
  const size_t lds_bytes = sizeof(float) * 2 * Cfg<LOGM>::PLANE;
  MEGA_CHECK_HIP(hipFuncSetAttribute(
      reinterpret_cast<const void*>(&fftconv_kernel<LOGM, DT, MODE, VEC, PAIR>),
      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
  fftconv_kernel<LOGM, DT, MODE, VEC, PAIR><<<dim3(static_cast<unsigned>(std::min(rows.groups, slots))), Cfg<LOGM>::T, lds_bytes, stream>>>(
      a, b, out, rows, flip, tab, scratch, omega);
  MEGA_CHECK_LAUNCH();
  return MEGA_OK;
}

template <int LOGM, int DT, int MODE, bool VEC>
int launch_fft_v(const void* a, const void* b, void* out, int64_t B, int64_t D, int64_t L, int flip, const float* omega, hipStream_t stream) {
  using C = Cfg<LOGM>;
  const c32* tab = nullptr;
  Scratch scratch{};
  int slots = 0, have = 0;
  int rc = get_tables<LOGM>(stream, &tab, &slots);
  if (rc != MEGA_OK) return rc;
  MEGA_CHECK_ARG(B * D <= 0x7fffffff, "fftconv: too many rows");
  constexpr int kMost = MODE == 0 && LOGM == 14 ? 1 : 2;
  int64_t nb = group_rows(B, D, slots, kMost, MODE == 1);
  int pair = nb == 1 ? 1 : kMost;
  const auto parts = [&] { return pair + (MODE == 1 && nb < B ? 1 : 0); };
  rc = get_scratch<LOGM>(stream, parts(), &scratch, &have);
  if (rc != MEGA_OK) return rc;
  // (fewer under capture, in a block of other launches: rows one by one then, and no channel's dk shared out)
  if (have < parts()) pair = 1, nb = MODE == 1 ? B : group_rows(B, D, slots, 1, false);
  const Rows rows = make_rows(B, D, L, nb);
  const bool split = MODE == 1 && nb < B;
  const int how = MODE == 1 ? split : flip;
  if (kMost == 1 || pair == 1) rc = launch_rows<LOGM, DT, MODE, VEC, 1>(a, b, out, rows, how, omega, tab, scratch, slots, stream);
  else rc = launch_rows<LOGM, DT, MODE, VEC, kMost>(a, b, out, rows, how, omega, tab, scratch, slots, stream);
  if (rc != MEGA_OK) return rc;
  if (split) {
    split_sum_kernel<<<dim3(static_cast<unsigned>((D * L + 255) / 256)), 256, 0, stream>>>(scratch.part[pair], static_cast<float*>(out), rows, 2 * C::M);
    MEGA_CHECK_LAUNCH();
  }
  return scratch_used<LOGM>(stream);
}

template <int LOGM, int DT, int MODE>
int launch_fft(const void* a, const void* b, void* out, int64_t B, int64_t D, int64_t L, int flip,
               const float* omega, hipStream_t stream) {
  const auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 8 == 0; };
  const bool vec = (L % 2 == 0) && al(a) && al(b) && al(out);
  return vec ? launch_fft_v<LOGM, DT, MODE, true>(a, b, out, B, D, L, flip, omega, stream)
             : launch_fft_v<LOGM, DT, MODE, false>(a, b, out, B, D, L, flip, omega, stream);
}

}  // namespace

template <int LOGM>
int fftconv_rows(int dtype, int mode, const void* a, const void* b, void* out, int64_t B, int64_t D, int64_t L, int flip,
                 const float* omega, hipStream_t stream) {
  switch (2 * dtype + mode) {
    case 2 * MEGA_F32: return launch_fft<LOGM, MEGA_F32, 0>(a, b, out, B, D, L, flip, omega, stream);
    case 2 * MEGA_F32 + 1: return launch_fft<LOGM, MEGA_F32, 1>(a, b, out, B, D, L, flip, omega, stream);
    case 2 * MEGA_BF16: return launch_fft<LOGM, MEGA_BF16, 0>(a, b, out, B, D, L, flip, omega, stream);
    case 2 * MEGA_BF16 + 1: return launch_fft<LOGM, MEGA_BF16, 1>(a, b, out, B, D, L, flip, omega, stream);
    case 2 * MEGA_F16: return launch_fft<LOGM, MEGA_F16, 0>(a, b, out, B, D, L, flip, omega, stream);
    default: return launch_fft<LOGM, MEGA_F16, 1>(a, b, out, B, D, L, flip, omega, stream);
  }
}
template <int LOGM>
int fftconv_tables(hipStream_t stream) {
  const c32* tab = nullptr;
  Scratch scratch{};
  int slots = 0, have = 0;
  if (const int rc = get_tables<LOGM>(stream, &tab, &slots); rc != MEGA_OK) return rc;
  return get_scratch<LOGM>(stream, kSlotParts, &scratch, &have);
}
template int fftconv_rows<MEGA_FFTCONV_LOGM>(int, int, const void*, const void*, void*, int64_t, int64_t, int64_t, int, const float*, hipStream_t);
template int fftconv_tables<MEGA_FFTCONV_LOGM>(hipStream_t);
#endif  // MEGA_FFTCONV_LOGM

}  // namespace mega
