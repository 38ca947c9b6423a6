// conv_nchwc, f32 only as in the reference:
//
//   * conv_nchwc_mfma_*, for k0 = 16 and c0 a multiple of 16 (the reference's own
//     tuned tile shape is 16 x 16 x 16,
//     runtime/src/iree/builtins/ukernel/arch/x86_64/conv_nchwc_x86_64_avx512_base.c:17-28):
//     an output panel of 16 pixels x 16 channels is a 16x16 MFMA block whose K
//     runs over (ic_outer, fh, fw, ci). A wave owns TW panels of consecutive
//     output pixels times TO blocks of OC_outer and feeds
//     v_mfma_f32_16x16x4_f32: a lane's 16-byte piece of one input pixel (four
//     ci, straight from global memory) is the operand of four instructions,
//     one per word, against four filter words of the same four ci (staged
//     through LDS by the workgroup, or loaded by each wave: the direct and the
//     split kernel). Sums are in MFMA order, so results equal the
//     reference's to rounding, and exactly where every partial sum is exact
//     (the reference's own test data, tools/conv_nchwc_test.c:174-178).
//   * conv_nchwc_generic, for every other shape: one thread per output
//     element, accumulating in the order of the CPU generic tile function
//     (runtime/src/iree/builtins/ukernel/conv_nchwc_tile_generic.c:34-57) with
//     a separate multiply and add, so that results equal the reference's
//     generic path bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "uk_device_common.h"
#include "uk_hip_abi.h"
#include "uk_launch.h"

namespace uk_mfma {
// mmt4d_mfma.hip: partial sums and zeroed counters the library keeps per host thread
// and stream (0 and the pointers, 1 when there are none to be had, or a status).
struct KSplitWorkspace {
  char* partials;
  uint32_t* counters;
};
int acquire_ksplit_workspace(size_t partial_bytes, uint32_t n_counters, hipStream_t stream, KSplitWorkspace* ws);
}  // namespace uk_mfma

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

struct ConvArgs {
  const float* in;
  const float* flt;
  float* out;
  int64_t in_sn, in_sic, in_sh;
  int64_t f_soc, f_sic, f_sfh;
  int64_t out_sn, out_soc, out_soh;
  int64_t OC, OH, OW, IC, FH, FW;
  int32_t k0, c0, stride_h, stride_w;
  uint32_t accumulate;
  int64_t total;
  int64_t N;
  // Direct kernel: floats from an image's first element down to the lowest one that
  // the pixels of a step start at, and that the steps of a pixel start at (negative
  // strides, else 0); the same of the filters of a few channel blocks.
  int64_t in_low_px, in_low_step, f_low_oc, f_low_step;
  int32_t steps;    // 16-channel products a sum has (the matrix-core kernels)
  // Split kernel: workgroups a tile's steps are divided over, and where those meet
  // (blocks of partial sums; one counter per tile, zero between launches).
  int32_t slices;
  uint32_t* partials;
  uint32_t* counters;
};

__global__ __launch_bounds__(kThreads) void conv_nchwc_generic_kernel(ConvArgs a) {
  for (int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x; idx < a.total;
       idx += (int64_t)gridDim.x * kThreads) {
    int64_t t = idx;
    const int32_t ko = (int32_t)(t % a.k0); t /= a.k0;
    const int64_t ow = t % a.OW; t /= a.OW;
    const int64_t oh = t % a.OH; t /= a.OH;
    const int64_t oc = t % a.OC;
    const int64_t n = t / a.OC;
    float* o = a.out + n * a.out_sn + oc * a.out_soc + oh * a.out_soh + ow * a.k0 + ko;
    float acc = a.accumulate ? *o : 0.f;
    const float* in_n = a.in + n * a.in_sn + (oh * a.stride_h) * a.in_sh + (ow * a.stride_w) * a.c0;
    const float* f_oc = a.flt + oc * a.f_soc + ko;
    for (int64_t ic = 0; ic < a.IC; ++ic) {
      for (int64_t fh = 0; fh < a.FH; ++fh) {
        const float* in_row = in_n + ic * a.in_sic + fh * a.in_sh;
        const float* f_row = f_oc + ic * a.f_sic + fh * a.f_sfh;
        for (int64_t fw = 0; fw < a.FW; ++fw) {
          for (int32_t ci = 0; ci < a.c0; ++ci) {
            acc += in_row[fw * a.c0 + ci] * f_row[(fw * a.c0 + ci) * (int64_t)a.k0];
          }
        }
      }
    }
    *o = acc;
  }
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_a4 __attribute__((aligned(4)));  // dword-aligned wide accesses are legal here

// A workgroup of four waves owns (n, TO output-channel blocks, 4 x TW panels of
// 16 output pixels); each wave computes TW panels against all TO blocks.
// Pixels are counted through (oh, ow) together, so rows shorter than a panel
// waste nothing. A step is one (ic_outer, fh, fw, 16 channels): 16 input
// floats per pixel against a [16 ci][16 ko] filter tile per channel block.
//
// Lane (q, r) = (lane / 16, lane % 16) supplies input pixel r, channels
// 4q..4q+3 of the step's 16 (one 16-byte global load, a step ahead, two
// register buffers) and filter words [ci = 4q + w][ko = r], w = 0..3. Those
// four words are 64 bytes apart in memory, so the filter tiles go through LDS:
// the first TO waves copy a step's tiles with one 16-byte load per lane
// (global memory a step ahead, LDS double-buffered, rows padded to 20 floats so
// that the 64 lanes of a read hit 64 different banks), one barrier per step.
// With the filter as the first MFMA operand a lane ends up holding output
// pixel r, channels 4q..4q+3: one 16-byte store. Pixels, panels and channel
// blocks past the end read the last valid one instead and are not stored; a
// prefetch past the last step reloads the last step. The launch bound keeps the
// accumulators in the vector registers the MFMAs name, without a copy to and
// from the accumulation registers around the loop (3x3, stride 2, 288 -> 96
// channels at 81x81, batch 5: 217 -> 214 us).
//
// For sums of up to ten steps (1x1 filters on few channels), which are loads and
// stores: there the waves of a workgroup share the filter loads. Longer sums take
// the kernels below (batch 16, 256 -> 256 channels, 3x3 at 56x56: 569 us here, 437).
constexpr int kFilterRow = 20;                 // floats per padded ci row in LDS
constexpr int kFilterTile = 16 * kFilterRow;   // floats per [16][16] tile in LDS

template <int TW, int TO>
__global__ __launch_bounds__(kThreads, 2) void conv_nchwc_mfma_lds_kernel(ConvArgs a, int64_t px_chunks,
                                                                   int64_t px_groups,
                                                                   int64_t oc_chunks) {
  static_assert(TO * 64 <= kThreads, "one loader lane per 16 bytes of the step's filter tiles");
  __shared__ __attribute__((aligned(16))) float filt[2][TO * kFilterTile];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Consecutive workgroup ids go round-robin to the 8 XCDs, each with its own
  // L2. Give every XCD a contiguous range of the work instead, so that one L2
  // sees one image and one filter slice at a time, not a slice of all.
  const uint32_t nb = gridDim.x, xcd = blockIdx.x & 7u;
  int64_t t = (int64_t)(xcd * (nb / 8u) + min(xcd, nb % 8u) + (blockIdx.x >> 3));
  const int64_t pxg = t % px_groups; t /= px_groups;
  const int64_t occ = t % oc_chunks; t /= oc_chunks;
  const int64_t n = t;
  const int64_t pxc_raw = pxg * 4 + wave;
  const bool wave_ok = pxc_raw < px_chunks;
  const int64_t pxc = wave_ok ? pxc_raw : px_chunks - 1;
  const int r = lane & 15, q = lane >> 4;
  const int64_t pixels = a.OH * a.OW;

  const float* pa[TW];
  float* po[TW][TO];
  bool ok[TW][TO];
#pragma unroll
  for (int tw = 0; tw < TW; ++tw) {
    const int64_t px = pxc * (16 * TW) + tw * 16 + r;
    const int64_t px_in = px < pixels ? px : pixels - 1;
    const int64_t oh = px_in / a.OW, ow = px_in - oh * a.OW;
    pa[tw] = a.in + n * a.in_sn + (oh * a.stride_h) * a.in_sh + (ow * a.stride_w) * a.c0 + 4 * q;
#pragma unroll
    for (int to = 0; to < TO; ++to) {
      const int64_t oc = occ * TO + to;
      const int64_t oc_in = oc < a.OC ? oc : a.OC - 1;
      ok[tw][to] = wave_ok && px < pixels && oc < a.OC;
      po[tw][to] = a.out + n * a.out_sn + oc_in * a.out_soc + oh * a.out_soh + ow * 16 + 4 * q;
    }
  }
  // Loader lanes (waves 0..TO-1): wave `wave` copies channel block occ*TO+wave,
  // lane l the 16 bytes [ci = l / 4][ko = 4 * (l % 4) ..].
  const bool loader = wave < TO;
  const int64_t oc_ld = min(occ * TO + (loader ? wave : 0), a.OC - 1);
  const float* pf = a.flt + oc_ld * a.f_soc + lane * 4;
  const int f_dst = (loader ? wave : 0) * kFilterTile + (lane >> 2) * kFilterRow + (lane & 3) * 4;
  const int f_src = (4 * q) * kFilterRow + r;   // + to * kFilterTile + w * kFilterRow

  v4f acc[TW][TO];
#pragma unroll
  for (int tw = 0; tw < TW; ++tw)
#pragma unroll
    for (int to = 0; to < TO; ++to) {
      acc[tw][to] = v4f{0.f, 0.f, 0.f, 0.f};
      if (a.accumulate && ok[tw][to]) acc[tw][to] = *reinterpret_cast<const v4f_a4*>(po[tw][to]);
    }

  // Within one (ic_outer, fh) consecutive steps follow each other at 16 input
  // floats and 256 filter floats.
  const int64_t taps = a.FW * (a.c0 / 16);
  const int64_t steps = a.IC * a.FH * taps;
  if (steps > 0) {
    int64_t ic = 0, fh = 0, tap = 0;  // the step the next prefetch loads
    v4f av[2][TW];
    v4f fv = v4f{0.f, 0.f, 0.f, 0.f};
    auto prefetch = [&](auto buf) {
      constexpr int B = decltype(buf)::value;
      const int64_t ao = ic * a.in_sic + fh * a.in_sh + tap * 16;
      const int64_t bo = ic * a.f_sic + fh * a.f_sfh + tap * 256;
      // Every wave issues the filter load (the waves that do not stage it read
      // the first block's tile and drop it): one issue order on all paths
      // keeps the compiler's wait counts from covering the loads just issued.
      fv = *reinterpret_cast<const v4f_a4*>(pf + bo);
#pragma unroll
      for (int tw = 0; tw < TW; ++tw) av[B][tw] = *reinterpret_cast<const v4f_a4*>(pa[tw] + ao);
      // Advance, staying on the last step once it is reached.
      if (!(ic == a.IC - 1 && fh == a.FH - 1 && tap == taps - 1)) {
        if (++tap == taps) {
          tap = 0;
          if (++fh == a.FH) {
            fh = 0;
            ++ic;
          }
        }
      }
    };
    auto stage_filter = [&](int b) {
      if (loader) *reinterpret_cast<v4f*>(&filt[b][f_dst]) = fv;
    };
    // Computes the step held in av[B] and filt[B]; meanwhile fetches the next
    // step into av[1 - B] and, through fv, filt[1 - B].
    auto iteration = [&](auto buf) {
      constexpr int B = decltype(buf)::value;
      prefetch(std::integral_constant<int, 1 - B>{});
      float bv[TO][4];
#pragma unroll
      for (int to = 0; to < TO; ++to)
#pragma unroll
        for (int w = 0; w < 4; ++w) bv[to][w] = filt[B][to * kFilterTile + w * kFilterRow + f_src];
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int tw = 0; tw < TW; ++tw)
#pragma unroll
          for (int to = 0; to < TO; ++to)
            acc[tw][to] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[to][w], av[B][tw][w],
                                                               acc[tw][to], 0, 0, 0);
      stage_filter(1 - B);
      __syncthreads();
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    prefetch(B0{});
    stage_filter(0);
    __syncthreads();
    int64_t s = 0;
    for (; s + 1 < steps; s += 2) {
      iteration(B0{});
      iteration(B1{});
    }
    if (s < steps) iteration(B0{});
  }
#pragma unroll
  for (int tw = 0; tw < TW; ++tw)
#pragma unroll
    for (int to = 0; to < TO; ++to)
      if (ok[tw][to]) *reinterpret_cast<v4f_a4*>(po[tw][to]) = acc[tw][to];
}

// The same division of the work without LDS: each wave loads the filter from
// global memory in the order in which the matrix instructions can take it, and
// waves share nothing. Lane (q, r) loads, of the filter rows ci = 4q + w, w =
// 0..3, TO consecutive floats each (one 4 * TO byte load a row), so that the 16
// lanes of a row cover all 16 * TO output channels. MFMA (w, i) multiplies word w
// of the pixel with float i of row 4q + w: its 16 output rows are the channels i,
// TO + i, 2 TO + i, ... of the 16 * TO, and the accumulators of i = 0..TO-1 together
// hold, in each lane, 4 * TO consecutive channels of output pixel r. Sums are the
// same, in the same order, as with the filter in LDS, but in tiles of one panel and
// one block, which are summed in four chains (conv_add_steps).
//
// Bound by the rate of the f32 MFMAs, which is easily lost: vector instructions
// take the same pipe, and beside a few 64-bit address additions per load two and
// more waves on a matrix core ran their MFMAs at 0.70 of it. So a load here is a
// buffer load, whose address is a scalar offset that moves along and a 32-bit lane
// offset that does not: no vector instruction but loads and MFMAs in the loop.
// They are issued one between several MFMAs (the groups below), D - 1 steps ahead
// in D register sets. 3x3, 256 -> 256 channels, batch 16 at 48x64 (369 us of MFMAs),
// tiles of 4x4: 64-bit addresses 520 us, filters through LDS with a barrier a step
// 474, this 399; 2x4 579 / 495 / 402; 1x4 - / 523 / 416; batch 4 at 64x64 (123 us)
// 155 / 175 / 140.
template <int... I, typename F>
__device__ __forceinline__ void for_each_index(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// The resource of buffer loads from `base` + 32-bit offsets, without bounds of its own.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_at(const float* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, -1, 0x00027000);
}

template <int TO>
__device__ __forceinline__ auto load_floats(__amdgpu_buffer_rsrc_t from, uint32_t lane_bytes, uint32_t bytes) {
  typedef float vTOf __attribute__((ext_vector_type(TO)));
  if constexpr (TO == 4) {
    return __builtin_bit_cast(vTOf, __builtin_amdgcn_raw_buffer_load_b128(from, lane_bytes, bytes, 0));
  } else if constexpr (TO == 2) {
    return __builtin_bit_cast(vTOf, __builtin_amdgcn_raw_buffer_load_b64(from, lane_bytes, bytes, 0));
  } else {
    return vTOf(__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, lane_bytes, bytes, 0)));
  }
}

// Where the loads of a sum come from: `base` + a lane's bytes + the step's bytes, 32-bit
// ones through a buffer resource or (WIDE: images and filters that span more) 64-bit ones.
template <bool WIDE>
struct LoadFrom {
  using Bytes = uint32_t;   // a step back is an addition that wraps
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ explicit LoadFrom(const float* base) : rsrc(buffer_at(base)) {}
  template <int TO>
  __device__ __forceinline__ auto load(Bytes lane, Bytes step) const { return load_floats<TO>(rsrc, lane, step); }
};
template <>
struct LoadFrom<true> {
  using Bytes = int64_t;
  const char* base;
  __device__ explicit LoadFrom(const float* b) : base((const char*)b) {}
  template <int TO>
  __device__ __forceinline__ auto load(Bytes lane, Bytes step) const {
    typedef float vTOf __attribute__((ext_vector_type(TO)));
    typedef vTOf vTOf_a4 __attribute__((aligned(4)));
    return (vTOf)*reinterpret_cast<const vTOf_a4*>(base + lane + step);
  }
};

// One of two values that are both there: a select, where ?: would choose between two
// places to load from.
template <typename T>
__device__ __forceinline__ T pick(bool first, T a, T b) { return first ? a : b; }

// Where a lane's results of panel tw go: 4 * TO consecutive channels of one pixel
// (nullptr: past the end). Channel c of them is word c / TO of the accumulator of i =
// c % TO.
template <int TW, int TO>
__device__ __forceinline__ float* conv_out_of(const ConvArgs& a, int32_t pxc, int32_t occ, int32_t n, int tw) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int32_t px = (pxc * TW + tw) * 16 + r, OW = (int32_t)a.OW;
  const int32_t oh = px / OW, ow = px - oh * OW;
  const int32_t oc = occ * TO + q * TO / 4;
  if (px >= (int32_t)(a.OH * a.OW) || oc >= (int32_t)a.OC) return nullptr;
  return a.out + n * a.out_sn + oc * a.out_soc + oh * a.out_soh + ow * 16 + q * 4 * TO % 16;
}

// What the sums of a tile start from: the output under ACCUMULATE, else zero.
template <int TW, int TO>
__device__ __forceinline__ void conv_begin(const ConvArgs& a, int32_t pxc, int32_t occ, int32_t n, v4f (&acc)[TW][TO]) {
#pragma unroll
  for (int tw = 0; tw < TW; ++tw) {
#pragma unroll
    for (int to = 0; to < TO; ++to) acc[tw][to] = v4f{0.f, 0.f, 0.f, 0.f};
    if (!a.accumulate) continue;
    if (const float* po = conv_out_of<TW, TO>(a, pxc, occ, n, tw)) {
#pragma unroll
      for (int v = 0; v < TO; ++v) {
        const v4f o = *reinterpret_cast<const v4f_a4*>(po + 4 * v);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[tw][(4 * v + e) % TO][(4 * v + e) / TO] = o[e];
      }
    }
  }
}

template <int TW, int TO>
__device__ __forceinline__ void conv_store(const ConvArgs& a, int32_t pxc, int32_t occ, int32_t n,
                                           const v4f (&acc)[TW][TO]) {
#pragma unroll
  for (int tw = 0; tw < TW; ++tw) {
    float* po = conv_out_of<TW, TO>(a, pxc, occ, n, tw);
    if (!po) continue;
#pragma unroll
    for (int v = 0; v < TO; ++v) {
      v4f o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = acc[tw][(4 * v + e) % TO][(4 * v + e) / TO];
      *reinterpret_cast<v4f_a4*>(po + 4 * v) = o;
    }
  }
}

// Adds steps [begin, begin + steps) of the sums to `sum`. CHAINS > 1: words w, w + CHAINS,
// .. of the pixels' pieces add up apart and meet at the end: shorter chains of roundings
// (the split kernel's parts of a sum are fewer than the slices of input channels that it
// took the place of: 3x3, 256 -> 32 channels at 10x10, batch 8, relative error 4.3e-7 with
// one chain, 2.2e-7 with four), and MFMAs that do not wait for each other in small tiles.
template <int TW, int TO, int D, int CHAINS, bool WIDE = false>
__device__ __forceinline__ void conv_add_steps(const ConvArgs& a, int32_t pxc, int32_t occ, int32_t n, int32_t begin,
                                               int32_t steps, v4f (&sum)[TW][TO]) {
  typedef float vTOf __attribute__((ext_vector_type(TO)));
  if (steps <= 0) return;
  v4f acc[CHAINS][TW][TO];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int tw = 0; tw < TW; ++tw)
#pragma unroll
      for (int to = 0; to < TO; ++to) acc[c][tw][to] = c == 0 ? sum[tw][to] : v4f{0.f, 0.f, 0.f, 0.f};
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  const int32_t last_px = (int32_t)(a.OH * a.OW) - 1, OW = (int32_t)a.OW;
  using Bytes = typename LoadFrom<WIDE>::Bytes;
  Bytes pa[TW];
#pragma unroll
  for (int tw = 0; tw < TW; ++tw) {
    const int32_t px = min((pxc * TW + tw) * 16 + r, last_px);
    const int32_t oh = px / OW, ow = px - oh * OW;
    pa[tw] = (Bytes)(((int64_t)oh * a.stride_h * a.in_sh + (int64_t)ow * a.stride_w * a.c0 + 4 * q -
                         a.in_low_px) * 4);
  }
  constexpr int kLanesPerBlock = 16 / TO;
  const int32_t oc_ld = min(r / kLanesPerBlock, (int32_t)a.OC - 1 - occ * TO);
  const Bytes pf = (Bytes)((oc_ld * a.f_soc + (4 * q) * 16 + r % kLanesPerBlock * TO - a.f_low_oc) * 4);

  // Within one (ic_outer, fh) consecutive steps follow each other at 16 input
  // floats and 256 filter floats.
  const int32_t IC = (int32_t)a.IC, FH = (int32_t)a.FH, taps = (int32_t)(a.FW * (a.c0 / 16));
  const Bytes in_next_fh = (Bytes)((a.in_sh - (taps - 1) * 16) * 4);
  const Bytes f_next_fh = (Bytes)((a.f_sfh - (taps - 1) * 256) * 4);
  const Bytes in_next_ic = (Bytes)((a.in_sic - (FH - 1) * a.in_sh - (taps - 1) * 16) * 4);
  const Bytes f_next_ic = (Bytes)((a.f_sic - (FH - 1) * a.f_sfh - (taps - 1) * 256) * 4);
  // From the last step of all back to the first, for the prefetches past the end.
  const Bytes in_again = (Bytes)(-((IC - 1) * a.in_sic + (FH - 1) * a.in_sh + (taps - 1) * 16) * 4);
  const Bytes f_again = (Bytes)(-((IC - 1) * a.f_sic + (FH - 1) * a.f_sfh + (taps - 1) * 256) * 4);
  const LoadFrom<WIDE> in(a.in + n * a.in_sn + a.in_low_px + a.in_low_step);
  const LoadFrom<WIDE> flt(a.flt + occ * TO * a.f_soc + a.f_low_oc + a.f_low_step);
  // The step the next prefetch loads: its offsets and its distance from the ends of
  // its (ic_outer, fh), its ic_outer and the sum.
  const int32_t row0 = begin / taps, tap0 = begin - row0 * taps;
  const int32_t ic0 = row0 / FH, fh0 = row0 - ic0 * FH;
  Bytes ao = (Bytes)((ic0 * a.in_sic + fh0 * a.in_sh + tap0 * 16 - a.in_low_step) * 4);
  Bytes bo = (Bytes)((ic0 * a.f_sic + fh0 * a.f_sfh + tap0 * 256 - a.f_low_step) * 4);
  int32_t tap = taps - 1 - tap0, fh = FH - 1 - fh0, ic = IC - 1 - ic0;
  constexpr int kProducts = 4 * TW * TO, kLoads = TW + 4;
  v4f av[D][TW];
  vTOf fv[D][4];
  auto prefetch = [&](auto buf) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int w = 0; w < 4; ++w) fv[B][w] = flt.template load<TO>(pf + w * 64, bo);
#pragma unroll
    for (int tw = 0; tw < TW; ++tw) av[B][tw] = in.template load<4>(pa[tw], ao);
    if constexpr (kProducts >= 16) {
      // All scalar selects: there are MFMAs enough to hide them, which a branch
      // between them would keep apart.
      const bool next_tap = tap != 0, next_fh = fh != 0, next_ic = ic != 0;
      ao += pick(next_tap, (Bytes)64, pick(next_fh, in_next_fh, pick(next_ic, in_next_ic, in_again)));
      bo += pick(next_tap, (Bytes)1024, pick(next_fh, f_next_fh, pick(next_ic, f_next_ic, f_again)));
      ic = pick(next_tap | next_fh, ic, pick(next_ic, ic - 1, IC - 1));
      fh = pick(next_tap, fh, pick(next_fh, fh - 1, FH - 1));
      tap = pick(next_tap, tap - 1, taps - 1);
    } else {
      ao += 64;
      bo += 1024;
      if (tap-- == 0) {
        ao += pick(fh != 0, in_next_fh, pick(ic != 0, in_next_ic, in_again)) - 64;
        bo += pick(fh != 0, f_next_fh, pick(ic != 0, f_next_ic, f_again)) - 1024;
        ic = pick(fh != 0, ic, pick(ic != 0, ic - 1, IC - 1));
        fh = pick(fh != 0, fh - 1, FH - 1);
        tap = taps - 1;
      }
    }
  };
  auto compute = [&](auto buf) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int tw = 0; tw < TW; ++tw)
#pragma unroll
        for (int to = 0; to < TO; ++to)
          acc[w % CHAINS][tw][to] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(fv[B][w][to], av[B][tw][w], acc[w % CHAINS][tw][to], 0, 0, 0);
  };
  for_each_index(std::make_integer_sequence<int, D - 1>{}, prefetch);
  auto iteration = [&](auto buf) {
    constexpr int B = decltype(buf)::value;
    __builtin_amdgcn_sched_barrier(0);
    prefetch(std::integral_constant<int, (B + D - 1) % D>{});
    compute(buf);
    // One load and a few scalar instructions between every `apart` MFMAs: they
    // are issued while the MFMA before them runs.
    if constexpr (kProducts >= 16) {
      constexpr int apart = kProducts / kLoads;
#pragma unroll
      for (int l = 0; l < kLoads; ++l) {
        __builtin_amdgcn_sched_group_barrier(0x008 /* MFMA */, apart / 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x020 /* loads */, 1, 0);
        if constexpr (apart > 2) __builtin_amdgcn_sched_group_barrier(0x008, apart - apart / 2 - 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x006 /* VALU, SALU */, 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int32_t s = steps;
  const std::make_integer_sequence<int, D> sets{};
  for (; s >= D; s -= D) for_each_index(sets, iteration);
  // The last steps % D are in the first register sets.
  for_each_index(sets, [&](auto buf) {
    if (decltype(buf)::value < s) compute(buf);
  });
#pragma unroll
  for (int tw = 0; tw < TW; ++tw)
#pragma unroll
    for (int to = 0; to < TO; ++to) {
      sum[tw][to] = acc[0][tw][to];
#pragma unroll
      for (int c = 1; c < CHAINS; ++c) sum[tw][to] += acc[c][tw][to];
    }
}

template <int TW, int TO, int D, bool WIDE>
__device__ __forceinline__ void conv_wave_tile(const ConvArgs& a, int32_t pxc, int32_t occ, int32_t n) {
  v4f acc[TW][TO];
  conv_begin<TW, TO>(a, pxc, occ, n, acc);
  conv_add_steps<TW, TO, D, TW * TO == 1 ? 4 : 1, WIDE>(a, pxc, occ, n, 0, a.steps, acc);
  conv_store<TW, TO>(a, pxc, occ, n, acc);
}

// Consecutive workgroup ids go round-robin to the 8 XCDs, each with its own L2.
// Gives every XCD a contiguous range of the work instead, so that one L2 sees one
// image and one filter slice at a time, not a slice of all.
__device__ __forceinline__ uint32_t xcd_contiguous(uint32_t id, uint32_t count) {
  const uint32_t xcd = id & 7u;
  return xcd * (count / 8u) + min(xcd, count % 8u) + (id >> 3);
}

// A workgroup of four waves owns (n, TO channel blocks, 4 x TW panels).
template <int TW, int TO, int D, bool WIDE = false>
__global__ __launch_bounds__(kThreads, 1) void conv_nchwc_mfma_direct_kernel(ConvArgs a, uint32_t px_chunks,
                                                                             uint32_t px_groups, uint32_t oc_chunks) {
  uint32_t t = xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t pxg = t % px_groups; t /= px_groups;
  const uint32_t pxc = pxg * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (pxc >= px_chunks) return;
  conv_wave_tile<TW, TO, D, WIDE>(a, (int32_t)pxc, (int32_t)(t % oc_chunks), (int32_t)(t / oc_chunks));
}

// Layers with too few tiles for the chip: the four waves of a workgroup own one tile and
// divide its steps, each a run of consecutive ones. Their sums meet in LDS and are added
// up in wave order. With `a.slices` > 1, the steps are divided over that many
// workgroups first, whose sums meet in memory: each stores its block with device-scope
// stores (the slices run on different XCDs), counts itself in when they have been
// acknowledged, and the one that is last adds the slices up in order and stores the
// result; see mmt4d_thin_kernel for why no fence is needed. Results are the same on
// every run.
template <int TW, int TO, int D, bool WIDE = false>
__global__ __launch_bounds__(kThreads) void conv_nchwc_mfma_split_kernel(ConvArgs a, uint32_t px_chunks,
                                                                         uint32_t oc_chunks) {
  __shared__ v4f partial[kWaves - 1][TW * TO][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t id = xcd_contiguous(blockIdx.x, gridDim.x), slices = (uint32_t)a.slices;
  const uint32_t tile = id / slices, slice = id - tile * slices;
  uint32_t t = tile;
  const int32_t pxc = (int32_t)(t % px_chunks); t /= px_chunks;
  const int32_t occ = (int32_t)(t % oc_chunks), n = (int32_t)(t / oc_chunks);
  const uint32_t share = slice * kWaves + wave, shares = slices * kWaves, steps = (uint32_t)a.steps;
  const uint32_t begin = (uint32_t)((uint64_t)share * steps / shares);
  const uint32_t end = (uint32_t)((uint64_t)(share + 1) * steps / shares);
  v4f acc[TW][TO];
#pragma unroll
  for (int tw = 0; tw < TW; ++tw)
#pragma unroll
    for (int to = 0; to < TO; ++to) acc[tw][to] = v4f{0.f, 0.f, 0.f, 0.f};
  if (share == 0) conv_begin<TW, TO>(a, pxc, occ, n, acc);
  conv_add_steps<TW, TO, D, TW * TO == 1 ? 4 : 2, WIDE>(a, pxc, occ, n, (int32_t)begin, (int32_t)(end - begin), acc);
  if (wave > 0) {
#pragma unroll
    for (int tw = 0; tw < TW; ++tw)
#pragma unroll
      for (int to = 0; to < TO; ++to) partial[wave - 1][tw * TO + to][lane] = acc[tw][to];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < kWaves - 1; ++w)
#pragma unroll
    for (int tw = 0; tw < TW; ++tw)
#pragma unroll
      for (int to = 0; to < TO; ++to) acc[tw][to] += partial[w][tw * TO + to][lane];
  if (slices > 1) {
    uint32_t* mine = a.partials + ((size_t)id * (TW * TO * 64) + lane) * 4;
#pragma unroll
    for (int tw = 0; tw < TW; ++tw)
#pragma unroll
      for (int to = 0; to < TO; ++to)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          __hip_atomic_store(mine + (tw * TO + to) * 256 + e, __builtin_bit_cast(uint32_t, (float)acc[tw][to][e]),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // All of the wave's stores above have been acknowledged before the count.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    uint32_t arrived = 0;
    if (lane == 0) {
      arrived = __hip_atomic_fetch_add(a.counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if ((uint32_t)__builtin_amdgcn_readfirstlane((int)arrived) != slices - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");   // no load below moves above the test
    if (lane == 0) __hip_atomic_store(a.counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t* all = a.partials + ((size_t)tile * slices * (TW * TO * 64) + lane) * 4;
#pragma unroll
    for (int tw = 0; tw < TW; ++tw)
#pragma unroll
      for (int to = 0; to < TO; ++to) acc[tw][to] = v4f{0.f, 0.f, 0.f, 0.f};
    for (uint32_t sl = 0; sl < slices; ++sl) {
#pragma unroll
      for (int tw = 0; tw < TW; ++tw)
#pragma unroll
        for (int to = 0; to < TO; ++to)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[tw][to][e] += __builtin_bit_cast(
                float, __hip_atomic_load(all + ((size_t)sl * (TW * TO) + tw * TO + to) * 256 + e, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT));
    }
  }
  conv_store<TW, TO>(a, pxc, occ, n, acc);
}

// D = 0: the filter through LDS, else the direct kernel with D register sets.
template <int TW, int TO, int D, bool WIDE = false>
int launch_mfma(const ConvArgs& a, hipStream_t stream) {
  const int64_t px_chunks = uk::ceil_div(a.OH * a.OW, (int64_t)16 * TW);
  const int64_t px_groups = uk::ceil_div(px_chunks, (int64_t)(kThreads / 64));
  const int64_t oc_chunks = uk::ceil_div(a.OC, (int64_t)TO);
  const int64_t blocks = a.N * oc_chunks * px_groups;
  if (blocks >= (1ll << 31)) return -1;
  if constexpr (D == 0) {
    uk::launch(3, conv_nchwc_mfma_lds_kernel<TW, TO>, dim3((uint32_t)blocks), dim3(kThreads), 0, stream,
               a, px_chunks, px_groups, oc_chunks);
  } else {
    uk::launch(3, conv_nchwc_mfma_direct_kernel<TW, TO, D, WIDE>, dim3((uint32_t)blocks), dim3(kThreads), 0, stream, a,
               (uint32_t)px_chunks, (uint32_t)px_groups, (uint32_t)oc_chunks);
  }
  return (int)hipGetLastError();
}

// The split kernel with up to `slices` workgroups a tile (fewer when no workspace is to
// be had: calls under capture).
template <int TW, int TO, int D, bool WIDE = false>
int launch_split(ConvArgs a, int32_t slices, hipStream_t stream) {
  const int64_t px_chunks = uk::ceil_div(a.OH * a.OW, (int64_t)16 * TW);
  const int64_t oc_chunks = uk::ceil_div(a.OC, (int64_t)TO);
  const int64_t tiles = px_chunks * oc_chunks * a.N;
  if (tiles * slices >= (1ll << 31)) return -1;
  if (slices > 1) {
    uk_mfma::KSplitWorkspace ws{};
    const int got = uk_mfma::acquire_ksplit_workspace((size_t)(tiles * slices) * TW * TO * 1024, (uint32_t)tiles,
                                                      stream, &ws);
    if (got > 1) return got;
    if (got == 0) {
      a.slices = slices;
      a.partials = (uint32_t*)ws.partials;
      a.counters = ws.counters;
    }
  }
  uk::launch(3, conv_nchwc_mfma_split_kernel<TW, TO, D, WIDE>, dim3((uint32_t)(tiles * a.slices)), dim3(kThreads), 0,
             stream, a, (uint32_t)px_chunks, (uint32_t)oc_chunks);
  return (int)hipGetLastError();
}

// Sums of up to ten steps. A kernel and its share of the output: TW panels of pixels
// and TO output-channel blocks per wave. `cost` is the measured time of one step per
// panel and block of a wave in 0.1 ns (the four MFMAs alone take 533), with the rounds
// of workgroups on the compute units that `rounds` names; the direct kernel's are from
// before its buffer loads, with which 70 such layers took 0.94 of the time in the mean and
// none more than 0.2 us longer. `short_cost`, on the same
// scale, is for fewer than eight steps (1x1 filters on few channels), which are loads
// and stores rather than products and want several small waves on a matrix core; 0:
// not taken for them (16 -> 224
// channels, 1x1, 107x107, batch 7: 23.8 us on 4x4 through LDS, 18.4 on 2x2; 64
// -> 64, stride 2, 62x62, batch 5: 8.6 on 1x2 direct, 7.3 on 1x4 through LDS).
struct MfmaTile {
  int tw, to;
  enum { kOne, kMore, kAny } rounds;
  int cost, short_cost;
  int (*launch)(const ConvArgs&, hipStream_t);
  const char* name;
};
constexpr MfmaTile kMfmaTiles[] = {
    {4, 4, MfmaTile::kOne, 645, 0, launch_mfma<4, 4, 3>, "conv_nchwc_mfma_direct_4x4"},
    {2, 4, MfmaTile::kOne, 710, 0, launch_mfma<2, 4, 3>, "conv_nchwc_mfma_direct_2x4"},
    {2, 2, MfmaTile::kOne, 870, 0, launch_mfma<2, 2, 4>, "conv_nchwc_mfma_direct_2x2"},
    {1, 4, MfmaTile::kOne, 905, 0, launch_mfma<1, 4, 4>, "conv_nchwc_mfma_direct_1x4"},
    {1, 2, MfmaTile::kAny, 1050, 1370, launch_mfma<1, 2, 4>, "conv_nchwc_mfma_direct_1x2"},
    {1, 1, MfmaTile::kAny, 1220, 1220, launch_mfma<1, 1, 4>, "conv_nchwc_mfma_direct_1x1"},
    {4, 4, MfmaTile::kMore, 700, 0, launch_mfma<4, 4, 0>, "conv_nchwc_mfma_lds_4x4"},
    {2, 4, MfmaTile::kMore, 730, 800, launch_mfma<2, 4, 0>, "conv_nchwc_mfma_lds_2x4"},
    {1, 4, MfmaTile::kMore, 790, 750, launch_mfma<1, 4, 0>, "conv_nchwc_mfma_lds_1x4"},
    {2, 2, MfmaTile::kMore, 830, 830, launch_mfma<2, 2, 0>, "conv_nchwc_mfma_lds_2x2"},
    {2, 1, MfmaTile::kMore, 1000, 1000, launch_mfma<2, 1, 0>, "conv_nchwc_mfma_lds_2x1"},
};

// Longer sums: the direct kernel (four waves, four tiles) and the split kernel (four waves
// a tile, one to four workgroups). A call takes the one it is estimated to be done first
// with: what the fullest compute unit's matrix cores walk through, `cost` a step, panel
// and block, plus `per_tile` for the ends of a wave's tile, plus kSlicesMeet where
// workgroups meet; all in 0.1 ns, fitted to 158 layers of 16 to 512 channels at 7x7 to
// 111x111, batch 1 to 16. On those it picks a kernel 1.9 % slower than the fastest one in
// the geometric mean, 19 % at worst, and 1.40 times as fast as what was before (tiles with
// 64-bit addresses, through LDS, or with slices of the input channels that a second launch
// added up), 0.99 at worst.
struct LongTile {
  int tw, to, cost, per_tile;
  int (*direct)(const ConvArgs&, hipStream_t);
  int (*split)(ConvArgs, int32_t slices, hipStream_t);
  const char* name;
};
constexpr LongTile kLongTiles[] = {
    {1, 4, 620, 3000, launch_mfma<1, 4, 4>, nullptr, "conv_nchwc_mfma_direct_1x4"},
    {2, 2, 680, 3000, launch_mfma<2, 2, 4>, nullptr, "conv_nchwc_mfma_direct_2x2"},
    {2, 4, 590, 3000, launch_mfma<2, 4, 3>, nullptr, "conv_nchwc_mfma_direct_2x4"},
    {1, 4, 706, 4200, nullptr, launch_split<1, 4, 4>, "conv_nchwc_mfma_split_1x4"},
    {2, 2, 800, 4200, nullptr, launch_split<2, 2, 4>, "conv_nchwc_mfma_split_2x2"},
    {1, 1, 1170, 4200, nullptr, launch_split<1, 1, 8>, "conv_nchwc_mfma_split_1x1"},
};
constexpr int64_t kSlicesMeet = 27000;
// The same for layers beyond 32-bit offsets, with 64-bit ones, from five steps a wave of
// the split kernel on. The direct kernel then runs its MFMAs at 0.7 of the rate where a
// matrix core has several waves: one round of it. us through LDS / here, planes of input
// channels 64 MB and more apart: 3x3, 512 -> 512 at 7x7 91.6 / 13.1, 256 -> 256 at 14x14
// 47.0 / 10.7, 128 -> 128 at 56x56 25.5 / 15.3, 256 -> 256 at 28x28, batch 4 62.1 / 45.5,
// batch 8 98.4 / 79.7.
constexpr LongTile kWideTiles[] = {
    {2, 2, 870, 3000, launch_mfma<2, 2, 4, true>, nullptr, "conv_nchwc_mfma_direct_wide_2x2"},
    {2, 4, 710, 3000, launch_mfma<2, 4, 3, true>, nullptr, "conv_nchwc_mfma_direct_wide_2x4"},
    {1, 4, 1050, 4200, nullptr, launch_split<1, 4, 4, true>, "conv_nchwc_mfma_split_wide_1x4"},
};

// For sums of `a.steps` > 10 steps: the tile and slices of `tiles` that are estimated to
// be done first, if that is before `least`; the direct kernel in up to `most_direct`
// workgroups. Returns a HIP status, or -1 when not served.
template <size_t TILES>
int launch_long(const ConvArgs& a, const LongTile (&tiles)[TILES], int64_t most_direct, int64_t least, int64_t cus,
                hipStream_t stream, const char** name) {
  const int64_t pixels = a.OH * a.OW, steps = a.steps;
  const LongTile* best = nullptr;
  int best_slices = 1;
  for (const LongTile& t : tiles) {
    const int64_t px = 16 * t.tw * (t.direct ? kWaves : 1);
    const int64_t groups = a.N * uk::ceil_div(pixels, px) * uk::ceil_div(a.OC, (int64_t)t.to);
    if (t.direct && groups > most_direct) continue;
    for (int slices = 1; slices <= (t.direct ? 1 : 4); slices *= 2) {
      // (16 MB of partial sums at most.)
      if (slices > 1 && groups * slices * t.tw * t.to > 16384) break;
      const int64_t wave_steps = t.direct ? steps : uk::ceil_div(steps, (int64_t)kWaves * slices);
      const int64_t cost = uk::ceil_div(groups * slices, cus) * (wave_steps * t.tw * t.to * t.cost + t.per_tile) +
                           (slices > 1 ? kSlicesMeet : 0);
      if (cost < least) {
        least = cost;
        best = &t;
        best_slices = slices;
      }
    }
  }
  if (!best) return -1;
  *name = best->name;
  return best->direct ? best->direct(a, stream) : best->split(a, best_slices, stream);
}

// Workgroups a launch of `tile` has. tw and to are powers of
// two, so that going through the table costs shifts and not divisions: at 5 us
// a launch the host is what small layers wait for.
int64_t mfma_blocks(const ConvArgs& a, const MfmaTile& tile) {
  const int px_shift = 4 + 2 + __builtin_ctz((unsigned)tile.tw);   // 16 pixels, four waves
  const int to_shift = __builtin_ctz((unsigned)tile.to);
  const int64_t px_groups = (a.OH * a.OW + (1ll << px_shift) - 1) >> px_shift;
  return a.N * ((a.OC + tile.to - 1) >> to_shift) * px_groups;
}

}  // namespace

extern "C" int iree_uk_amd_hip_conv_nchwc_has_mfma_kernel(int32_t k0, int32_t c0,
                                                          uint32_t flags) {
  return (flags & IREE_UK_FLAG_CONV_NCHWC_TYPE_MASK) == IREE_UK_FLAG_CONV_NCHWC_TYPE_F32F32F32 &&
         k0 == 16 && c0 > 0 && c0 % 16 == 0;
}

extern "C" int iree_uk_amd_hip_launch_conv_nchwc(const iree_uk_conv_nchwc_params_t* p,
                                                 void* stream_v, int kernel_mode,
                                                 const char** kernel_name) {
  hipStream_t stream = (hipStream_t)stream_v;
  if ((p->flags & IREE_UK_FLAG_CONV_NCHWC_TYPE_MASK) != IREE_UK_FLAG_CONV_NCHWC_TYPE_F32F32F32) {
    return (int)hipErrorInvalidValue;
  }
  ConvArgs a;
  a.in = (const float*)p->input_buffer + p->input_offset;
  a.flt = (const float*)p->filter_buffer + p->filter_offset;
  a.out = (float*)p->output_buffer + p->output_offset;
  a.in_sn = p->input_stride_n; a.in_sic = p->input_stride_ic_outer; a.in_sh = p->input_stride_h;
  a.f_soc = p->filter_stride_oc_outer; a.f_sic = p->filter_stride_ic_outer;
  a.f_sfh = p->filter_stride_fh;
  a.out_sn = p->output_stride_n; a.out_soc = p->output_stride_oc_outer;
  a.out_soh = p->output_stride_oh;
  a.OC = p->OC_outer; a.OH = p->OH; a.OW = p->OW; a.IC = p->IC_outer; a.FH = p->FH; a.FW = p->FW;
  a.k0 = p->k0; a.c0 = p->c0; a.stride_h = p->stride_h; a.stride_w = p->stride_w;
  a.accumulate = (p->flags & IREE_UK_FLAG_CONV_NCHWC_ACCUMULATE) != 0;
  a.total = p->N * p->OC_outer * p->OH * p->OW * (int64_t)p->k0;
  a.N = p->N;
  a.steps = 0;
  a.slices = 1;
  a.partials = nullptr;
  a.counters = nullptr;
  if (a.total == 0) {
    *kernel_name = "";
    return 0;
  }
  if (kernel_mode != IREE_UK_AMD_KERNEL_MODE_GENERIC &&
      iree_uk_amd_hip_conv_nchwc_has_mfma_kernel(p->k0, p->c0, p->flags)) {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
      (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    }
    const int64_t steps_per_ic = a.FH * a.FW * (a.c0 / 16);
    const int64_t steps = a.IC * steps_per_ic;
    // The direct and the split kernel address an image and the filters of a few channel
    // blocks with 32 bits; what is larger takes the LDS kernel, or the split kernel with
    // 64-bit addresses.
    const int64_t in_ext[] = {(a.OH - 1) * a.stride_h * a.in_sh, (a.OW - 1) * a.stride_w * a.c0,
                              (a.IC - 1) * a.in_sic, (a.FH - 1) * a.in_sh};
    const int64_t f_ext[] = {3 * a.f_soc, (a.IC - 1) * a.f_sic, (a.FH - 1) * a.f_sfh};
    a.in_low_px = std::min<int64_t>(in_ext[0], 0) + std::min<int64_t>(in_ext[1], 0);
    a.in_low_step = std::min<int64_t>(in_ext[2], 0) + std::min<int64_t>(in_ext[3], 0);
    a.f_low_oc = std::min<int64_t>(f_ext[0], 0);
    a.f_low_step = std::min<int64_t>(f_ext[1], 0) + std::min<int64_t>(f_ext[2], 0);
    int64_t in_span = a.FW * a.c0, f_span = a.FW * a.c0 * 16;   // floats
    for (int64_t e : in_ext) in_span += std::abs(e);
    for (int64_t e : f_ext) f_span += std::abs(e);
    const bool indexed = a.OH * a.OW < (1ll << 30) && steps < (1ll << 20);
    const bool direct = indexed && in_span < (1ll << 29) && f_span < (1ll << 29);
    a.steps = (int32_t)std::min<int64_t>(steps, INT32_MAX);
    if (direct && steps > 10) {
      const int st = launch_long(a, kLongTiles, INT64_MAX, INT64_MAX, cus, stream, kernel_name);
      if (st >= 0) return st;
    }
    // The tile whose fullest compute unit is done first: workgroups per unit,
    // rounded up, times the work of one, times what that costs in this tile.
    // Large tiles re-read less and cost less per block; small ones waste less
    // in the last round and at the edges.
    const MfmaTile* tile = nullptr;
    int64_t least = 0;
    for (const MfmaTile& t : kMfmaTiles) {
      const int step_cost = steps < 8 ? t.short_cost : t.cost;
      if (step_cost == 0) continue;
      const int64_t rounds = uk::ceil_div(mfma_blocks(a, t), (int64_t)cus);
      // (The LDS kernel takes layers of any extent, with any number of rounds.)
      if (direct && t.rounds == MfmaTile::kOne && rounds > 1) continue;
      if (direct ? t.rounds == MfmaTile::kMore && rounds <= 1 : t.rounds != MfmaTile::kMore) continue;
      // Each group of channel blocks reads the input again, from memory where
      // the layer is a large one: 288 -> 48 channels, 3x3, stride 2, 84x84,
      // batch 12 (394 MB of input) took 364 us one block at a time, 284 on 2x4.
      if (t.to == 1 && rounds > 1 && a.OC > 1) continue;
      const int64_t cost = rounds * t.tw * t.to * step_cost;
      if (!tile || cost < least) {
        tile = &t;
        least = cost;
      }
    }
    if (!direct && indexed && steps >= 20) {
      // (The LDS tiles' costs are those of several rounds.)
      const bool one_round = mfma_blocks(a, *tile) <= cus;
      const int st = launch_long(a, kWideTiles, cus, one_round ? least * steps * 5 / 4 : least * steps, cus, stream, kernel_name);
      if (st >= 0) return st;
    }
    const int st = tile->launch(a, stream);
    if (st >= 0) {
      *kernel_name = tile->name;
      return st;
    }
  }
  *kernel_name = "conv_nchwc_generic";
  const int64_t blocks = uk::ceil_div(a.total, kThreads);
  const int64_t cap = 256 * 64;
  uk::launch(3, conv_nchwc_generic_kernel, dim3((uint32_t)(blocks < cap ? blocks : cap)),
             dim3(kThreads), 0, stream, a);
  return (int)hipGetLastError();
}
