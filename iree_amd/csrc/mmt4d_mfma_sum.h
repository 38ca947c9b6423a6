// Adds up the K slices of an mmt4d product (launch_slices of mmt4d_mfma_launch.h):
// row-major partial sums in, the caller's result out, with its ACCUMULATE input, its
// strides, its rounding and its scales.
//
// Bound by memory: 4 bytes a slice and element read once, coalesced (16 bytes a lane
// along a row), mostly from the memory-side cache that the slices were just written to:
// 5.0 us for four slices of 200 x 4096 into bf16 (13.1 MB: 2.6 TB/s with the launch),
// behind 36.6 us of the slices themselves. (One launch for both, the last workgroup of a
// block adding the others' sums up, would leave the adding to a quarter of the units.)
#ifndef IREE_UK_AMD_MMT4D_MFMA_SUM_H_
#define IREE_UK_AMD_MMT4D_MFMA_SUM_H_

#include "mmt4d_mfma_kernel.h"

namespace uk_mfma {

constexpr int kSumThreads = 128;

struct SumArgs {
  const char* partials;      // [slices][rows of whole tiles][pitch]
  int64_t slice_bytes, pitch;
  int32_t slices, rows, cols;  // rows, cols: of the result
  int32_t M0, N0;
  Divisor by_m0, by_n0;
  // Result and initial accumulators (null: none), addressed as in Args.
  char* out;
  int64_t out_stride;
  uint32_t out_sm0, out_spn;
  const char* acc;
  int64_t acc_stride;
  uint32_t acc_sm0, acc_spn;
  uint32_t vec;              // 4 consecutive columns of both are contiguous (and aligned enough)
  uint32_t dequant;
  const float* row_scale;
  const float* col_scale;
};

// A thread adds four columns of one row: even slices in order, odd slices in order, and
// those two sums (float errors of 16 slices are then not above those of four waves in
// eight workgroups: f16 128 x 1024 x 16384 in one order 1.67e-7, here 1.61e-7, there 1.61e-7).
template <typename Acc, typename Out>
__global__ __launch_bounds__(kSumThreads)
void mmt4d_sum_slices_kernel(SumArgs a) {
  constexpr int OB = Out::kOutBytes;
  using T = typename std::remove_reference<decltype(Acc{}[0])>::type;
  const int row = blockIdx.y;
  const int col = (blockIdx.x * kSumThreads + threadIdx.x) * 4;
  const int left = a.cols - col;
  if (left <= 0) return;
  const int pm = (int)a.by_m0.quotient(row), m0 = row - pm * a.M0;
  char* out = a.out + (int64_t)pm * a.out_stride + (int64_t)m0 * a.out_sm0;
  const char* init = a.acc + (int64_t)pm * a.acc_stride + (int64_t)m0 * a.acc_sm0;
  int64_t out_e[4], acc_e[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = min(col + e, a.cols - 1);
    const int pc = (int)a.by_n0.quotient(c), n0 = c - pc * a.N0;
    out_e[e] = (int64_t)pc * a.out_spn + n0 * OB;
    acc_e[e] = (int64_t)pc * a.acc_spn + n0 * OB;
  }
  const bool vec = a.vec && left >= 4;
  Acc v = {0, 0, 0, 0}, odd = {0, 0, 0, 0};
  if (a.acc) {
    if (vec) {
      v = Out::load4(init + acc_e[0]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < left) v[e] = Out::load1(init + acc_e[e]);
    }
  }
  // Rows of the partial sums are whole tiles long, not whole quads.
  typedef Acc Acc4 __attribute__((aligned(4)));
  const char* src = a.partials + row * a.pitch + (int64_t)col * 4;
  if (left >= 4) {
#pragma unroll 2
    for (int s = 0; s + 1 < a.slices; s += 2) {
      v += *reinterpret_cast<const Acc4*>(src + s * a.slice_bytes);
      odd += *reinterpret_cast<const Acc4*>(src + (s + 1) * a.slice_bytes);
    }
    if (a.slices % 2 != 0) v += *reinterpret_cast<const Acc4*>(src + (a.slices - 1) * a.slice_bytes);
  } else {
    for (int s = 0; s < a.slices; ++s) {
      const T* p = reinterpret_cast<const T*>(src + s * a.slice_bytes);
      Acc& sum = s % 2 != 0 ? odd : v;
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (e < left) sum[e] += p[e];
    }
  }
  v += odd;
  if constexpr (OB == 4) {
    if (a.dequant) {
      const float sm = a.row_scale ? a.row_scale[row] : 1.0f;
      v4f f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        f[e] = (float)v[e] * sm * (a.col_scale ? a.col_scale[min(col + e, a.cols - 1)] : 1.0f);
      typedef v4f v4f_a4 __attribute__((aligned(4)));
      if (vec) {
        *reinterpret_cast<v4f_a4*>(out + out_e[0]) = f;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < left) *reinterpret_cast<float*>(out + out_e[e]) = f[e];
      }
      return;
    }
  }
  if (vec) {
    Out::store4(out + out_e[0], v);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < left) Out::store1(out + out_e[e], v[e]);
  }
}

}  // namespace uk_mfma

#endif  // IREE_UK_AMD_MMT4D_MFMA_SUM_H_
