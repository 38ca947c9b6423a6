// Host-side selection and launch of the MFMA mmt4d kernels for one element
// type. Included by one translation unit per element type so that the kernel
// instantiations compile in parallel.
#ifndef IREE_UK_AMD_MMT4D_MFMA_LAUNCH_H_
#define IREE_UK_AMD_MMT4D_MFMA_LAUNCH_H_

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "mmt4d_mfma_kernel.h"
#include "mmt4d_mfma_narrow.h"
#include "mmt4d_mfma_persistent.h"
#include "mmt4d_mfma_sum.h"
#include "mmt4d_mfma_thin.h"
#include "uk_device_common.h"
#include "uk_hip_abi.h"
#include "uk_launch.h"

namespace uk_mfma {

// What the dispatcher hands to the per-type launcher: the problem in bytes.
struct Problem {
  const char* lhs;
  const char* rhs;
  char* out;
  int64_t lhs_stride, rhs_stride, out_stride;  // bytes between row panels
  // Output addressing beyond the panel stride (see Args in the kernel header):
  // bytes between rows inside a panel and between column panels, and how many
  // rows / columns exist counted from this problem's origin.
  int64_t out_sm0, out_spn;
  int64_t out_rows, out_cols;
  // Initial accumulators for ACCUMULATE, addressed like the output (the output
  // itself unless `dequant`), and the dequantizing store's scales, indexed
  // from this problem's origin (either may be null).
  const char* acc;
  int64_t acc_stride, acc_sm0, acc_spn;
  bool dequant;
  const float* row_scale;
  const float* col_scale;
  int32_t M1, N1, K1, M0, N0;
  int32_t rb, lrb;  // bytes per tile row and its log2
  bool accumulate;
  int32_t cus;      // compute units of the device, 0: the query failed, as the launch will (asked for once a call)
};

// Whether a shape has an instance for a K that ends inside a step (TAIL of the
// kernel): those that a call can reach by its sizes. Shapes that only a forced
// variant reaches decline such a K and leave it to the next one in line: with
// instances of theirs the library was half as large again. The 16-bit integers
// take K in whole steps only.
template <Elem E, int RBC, int TM, int TN, int WGM, int WGN, int PIPE>
constexpr bool has_tail_instance() {
  constexpr bool k64x64 = TM * WGM == 4 && TN * WGN == 4;
  if (E == Elem::kS16) return false;
  if (PIPE == 3) return E == Elem::kF32 || k64x64;
  if (PIPE == 5) {
    if (k64x64) return RBC < 16 && ElemTraits<E>::Out::kOutBytes == 4 && E != Elem::kF32;
    return E != Elem::kF32 && WGN != 8;  // (WGN == 8: 128x512)
  }
  return false;
}

// Launches one kernel variant over K-tiles [kt_begin, kt_begin + kt_count).
// Returns a HIP status, or -1 if the variant cannot serve the shape. SLICED: all
// of K in `kslices` parts, each into a result of its own (see the kernel).
template <Elem E, int RBC, int TM, int TN, int WGM, int WGN, int NKK, int PIPE, bool SLICED = false>
int launch_variant(const Problem& p, int kt_begin, int kt_count, bool accumulate,
                   hipStream_t stream, int kslices = 1) {
  using SH = Shape<E, TM, TN, WGM, WGN, NKK, PIPE, SLICED>;
  constexpr int R = RBC >= 16 ? 1 : 16 / RBC;
  if (SH::kLdsBytes > 160 * 1024) return -1;          // more LDS than a compute unit has
  if (p.rb > SH::KS) return -1;                       // a tile row must fit one step
  if (p.M0 > SH::BM || p.N0 > SH::BN) return -1;      // at least one whole panel
  if (p.M0 % R || p.N0 % R) return -1;                // pieces hold whole rows
  if (p.out_rows <= 0 || p.out_cols <= 0) return 0;   // a strip beyond the matrix: nothing to store
  Args a{};
  const int64_t kt_bytes_m = (int64_t)p.M0 << p.lrb, kt_bytes_n = (int64_t)p.N0 << p.lrb;
  a.lhs = p.lhs + kt_begin * kt_bytes_m;
  a.rhs = p.rhs + kt_begin * kt_bytes_n;
  a.out = p.out;
  a.lhs_stride = p.lhs_stride;
  a.rhs_stride = p.rhs_stride;
  a.out_stride = p.out_stride;
  a.out_sm0 = (uint32_t)p.out_sm0;
  a.out_spn = (uint32_t)p.out_spn;
  a.out_rows = (int32_t)std::min<int64_t>(p.out_rows, INT32_MAX);
  a.out_cols = (int32_t)std::min<int64_t>(p.out_cols, INT32_MAX);
  a.M1 = p.M1; a.N1 = p.N1; a.K1 = kt_count;
  a.M0 = p.M0; a.N0 = p.N0; a.rb = p.rb; a.lrb = p.lrb;
  a.bpm = SH::BM / p.M0;
  a.bpn = SH::BN / p.N0;
  const int64_t grid_m = uk::ceil_div(p.M1, a.bpm), grid_n = uk::ceil_div(p.N1, a.bpn);
  if (grid_m * grid_n * kslices >= (1ll << 31)) return -1;
  a.grid_m = (int32_t)grid_m;
  a.grid_n = (int32_t)grid_n;
  a.kslices = (uint32_t)kslices;
  const int64_t k_bytes = (int64_t)kt_count << p.lrb;
  a.steps = (int32_t)uk::ceil_div(k_bytes, SH::KS);
  if (a.steps < 1) a.steps = 1;
  a.tail = (k_bytes % SH::KS) != 0;
  constexpr bool kTail = !SLICED && has_tail_instance<E, RBC, TM, TN, WGM, WGN, PIPE>();
  if (PIPE != 0 && PIPE != 4 && ((a.tail && !kTail) || kt_count == 0)) return -1;
  a.accumulate = accumulate;
  // A launch that starts K reads the caller's accumulators; a later one
  // continues from what the previous launch left in the output. Only the
  // launch that finishes K applies the dequantizing store.
  const bool first = kt_begin == 0;
  a.acc = first ? p.acc : p.out;
  a.acc_stride = first ? p.acc_stride : p.out_stride;
  a.acc_sm0 = (uint32_t)(first ? p.acc_sm0 : p.out_sm0);
  a.acc_spn = (uint32_t)(first ? p.acc_spn : p.out_spn);
  a.dequant = p.dequant && kt_begin + kt_count == p.K1;
  a.row_scale = p.row_scale;
  a.col_scale = p.col_scale;
  // Block rows per rasterization band: an XCD's 32 resident workgroups should
  // cover a near-square patch of the output (4 x 8 blocks of 256x256, 8 x 4 of
  // 128x512: 3072 operand rows either way).
  a.band = (WGM == 1 && WGN == 8) ? 8 : 4;
  // Four consecutive output columns of one row are contiguous when they lie in
  // one tile row (N0 % 4 == 0) or when column panels follow each other without
  // a gap (row-major output, or tiles that are single rows). (Of four that reach
  // over a workgroup's last column the kernel takes its own, one by one: f16 ->
  // f32 16x9x16 1037 x 4990 x 256, 256x128 blocks of 126 columns, 12.9 us; all
  // elements one by one 22.7.) 4-byte outputs need no more alignment than their
  // own; 2-byte outputs move as 8-byte vectors and need that alignment.
  constexpr int OB = ElemTraits<E>::Out::kOutBytes;
  auto vector_ok = [&](const char* base, int64_t stride, int64_t sm0, int64_t spn) {
    const bool contiguous4 = p.N0 % 4 == 0 || spn == (int64_t)p.N0 * OB;
    const bool aligned4 = OB == 4 || (((uintptr_t)base | (uint64_t)stride | (uint64_t)sm0 |
                                       (uint64_t)spn) % 8) == 0;
    return contiguous4 && aligned4;
  };
  a.vec_out = vector_ok(p.out, p.out_stride, p.out_sm0, p.out_spn) &&
              (!accumulate || vector_ok(a.acc, a.acc_stride, a.acc_sm0, a.acc_spn));
  if (a.vec_out && a.bpn * p.N0 % 4 != 0) a.vec_out = 2;
  // The launch that finishes K stores non-temporally when the output is
  // larger than the memory-side cache can hand to its reader.
  a.nt_out = kt_begin + kt_count == p.K1 &&
             (int64_t)p.M1 * p.M0 * p.N1 * p.N0 * OB >= (192ll << 20);
  // 32-bit offsets inside a workgroup's share of each operand.
  const int64_t span_m = (int64_t)a.bpm * p.lhs_stride + (int64_t)p.K1 * kt_bytes_m;
  const int64_t span_n = (int64_t)a.bpn * p.rhs_stride + (int64_t)p.K1 * kt_bytes_n;
  const int64_t span_o = (int64_t)a.bpm * p.out_stride + (int64_t)p.M0 * p.out_sm0 +
                         (int64_t)p.N1 * p.out_spn;
  const int64_t span_a = (int64_t)a.bpm * a.acc_stride + (int64_t)p.M0 * a.acc_sm0 +
                         (int64_t)p.N1 * a.acc_spn;
  if (span_m >= (1ll << 31) || span_n >= (1ll << 31) || span_o >= (1ll << 31) ||
      span_a >= (1ll << 31)) {
    return -1;
  }
  set_divisors(a);
  auto go = [&](auto tail_c) {
    auto kernel = mmt4d_mfma_kernel<E, RBC, TM, TN, WGM, WGN, NKK, PIPE, decltype(tail_c)::value, SLICED>;
    if (SH::kLdsBytes > 64 * 1024) {
      // Raising the dynamic LDS limit is a per-function setting; do it once.
      static hipError_t attr = hipFuncSetAttribute(
          reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
          (int)SH::kLdsBytes);
      if (attr != hipSuccess) return (int)attr;
    }
    uk::launch(2, kernel, dim3((uint32_t)(grid_m * grid_n * kslices)), dim3(WGM * WGN * 64),
               SH::kLdsBytes, stream, a);
    return (int)hipGetLastError();
  };
  if constexpr (kTail) {
    if (a.tail) return go(std::true_type{});
  }
  return go(std::false_type{});
}

// Workspace of a K split over workgroups (the barrier-free kernel's, the K slices' of
// launch_slices, the split convolution's): `partial_bytes` of partial accumulators and
// `n_counters` arrival counters that are zero between launches. Defined in mmt4d_mfma.hip: ordinary calls get a buffer
// the library allocates per host thread and stream (grow-only; none while the
// stream is being captured into a graph and nothing fits yet), calls through
// iree_uk_amd_mmt4d_no_alloc get the library's static device array. Returns 0
// and the pointers, 1 when there is no workspace but the call can run without
// the split, or a status (> 1) that has to fail the call.
struct KSplitWorkspace {
  char* partials;
  uint32_t* counters;
};
int acquire_ksplit_workspace(size_t partial_bytes, uint32_t n_counters, hipStream_t stream,
                             KSplitWorkspace* ws);
// A buffer of `bytes` for s4 weights expanded to s8 (mmt4d_mfma_s8s4.hip), kept
// per host thread and stream like the K split's workspace and apart from it
// (the s8 launch that reads the expanded weights may itself split K). Returns
// 0 and the pointer, or 1 when there is none to be had: under
// iree_uk_amd_mmt4d_no_alloc, while the stream is being captured into a graph,
// or when the allocation fails.
int acquire_expand_workspace(size_t bytes, hipStream_t stream, char** base);
// Regroups the K tiles of an operand so that every tile row holds 16 bytes:
// `panels` panels of K1 tiles of R0 rows of `rb` bytes (rb = 1, 2, 4 or 8; panel
// n at src + n * src_stride) become ceil(K1 * rb / 16) tiles of R0 rows of 16
// bytes at dst + n * (that count * R0 * 16), the last one filled up with zero
// bytes. src_bits = 4: the source holds signed nibbles, low nibble first, half
// as many bytes, and `rb` counts the bytes they widen to. dst 16-byte aligned.
void retile_rows(const char* src, int64_t src_stride, int panels, int R0, int rb, int K1, int src_bits,
                 char* dst, hipStream_t stream);
// K slices set with iree_uk_amd_set_k_slices on this thread; 0 = choose.
int k_slices_override();
// 1: the calling thread has declared its weights streamed from HBM
// (iree_uk_amd_set_streamed_weights).
int streamed_weights();
// Records the slice count of the launch for iree_uk_amd_last_k_slices.
void note_k_slices(int n);

// Workgroup count set with iree_uk_amd_set_persistent_workgroups on this
// thread; 0 = one per compute unit (defined in mmt4d_mfma.hip).
int persistent_workgroups_override();

// Compute units of the current device (one persistent workgroup each).
inline int compute_units() {
  static thread_local int cached_device = -1, cached_cus = 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (dev != cached_device) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cached_device = dev;
    cached_cus = cus;
  }
  return cached_cus;
}

// Launches the persistent kernel (mmt4d_mfma_persistent.h) over K-tiles
// [0, kt_count): one workgroup per CU, each walking several output blocks
// without draining its pipeline in between. Returns a HIP status, or -1 if
// the kernel cannot serve the shape (or would not gain: fewer than two blocks
// per workgroup).
template <Elem E, int TM, int TN, int WGM, int WGN>
int launch_persistent(const Problem& p, int kt_count, bool force, hipStream_t stream) {
  constexpr int BM = WGM * TM * 16, BN = WGN * TN * 16, KS = 64;
  auto pow2 = [](int v) { return v > 0 && (v & (v - 1)) == 0; };
  if (p.rb < 16 || p.rb > KS) return -1;
  if (!pow2(p.M0) || !pow2(p.N0) || p.N0 < 4 || p.M0 > BM || p.N0 > BN) return -1;
  if (p.dequant) return -1;
  const int bpm = BM / p.M0, bpn = BN / p.N0;
  if (p.M1 % bpm || p.N1 % bpn) return -1;
  if (p.out_rows < (int64_t)p.M1 * p.M0 || p.out_cols < (int64_t)p.N1 * p.N0) return -1;
  const int64_t k_bytes = (int64_t)kt_count << p.lrb;
  if (k_bytes % (4 * KS) || k_bytes / KS < 8 || k_bytes / KS >= (1 << 24)) return -1;
  const int64_t grid_m = p.M1 / bpm, grid_n = p.N1 / bpn;
  const int64_t total = grid_m * grid_n;
  int cus = p.cus & ~7;  // a multiple of the 8 XCDs keeps blocks on their XCD
  if (persistent_workgroups_override() > 0) cus = persistent_workgroups_override();
  if (cus < 1 || total >= (1ll << 30)) return -1;
  if (!force && total < 2 * (int64_t)cus) return -1;
  const int64_t grid = std::min<int64_t>(total, cus);
  Args a{};
  a.lhs = p.lhs; a.rhs = p.rhs; a.out = p.out;
  a.lhs_stride = p.lhs_stride; a.rhs_stride = p.rhs_stride; a.out_stride = p.out_stride;
  a.out_sm0 = (uint32_t)p.out_sm0; a.out_spn = (uint32_t)p.out_spn;
  a.out_rows = (int32_t)std::min<int64_t>(p.out_rows, INT32_MAX);
  a.out_cols = (int32_t)std::min<int64_t>(p.out_cols, INT32_MAX);
  a.M1 = p.M1; a.N1 = p.N1; a.K1 = kt_count;
  a.M0 = p.M0; a.N0 = p.N0; a.rb = p.rb; a.lrb = p.lrb;
  a.bpm = bpm; a.bpn = bpn;
  a.grid_m = (int32_t)grid_m; a.grid_n = (int32_t)grid_n;
  a.steps = (int32_t)(k_bytes / KS);
  a.accumulate = p.accumulate;
  a.band = (WGM == 1 && WGN == 8) ? 8 : 4;
  a.vec_out = 1;
  a.acc = p.acc; a.acc_stride = p.acc_stride;
  a.acc_sm0 = (uint32_t)p.acc_sm0; a.acc_spn = (uint32_t)p.acc_spn;
  while ((1 << a.lm0) < p.M0) ++a.lm0;
  while ((1 << a.ln0) < p.N0) ++a.ln0;
  const int64_t kt_bytes_m = (int64_t)p.M0 << p.lrb, kt_bytes_n = (int64_t)p.N0 << p.lrb;
  const int64_t span_m = (int64_t)bpm * p.lhs_stride + (int64_t)p.K1 * kt_bytes_m;
  const int64_t span_n = (int64_t)bpn * p.rhs_stride + (int64_t)p.K1 * kt_bytes_n;
  const int64_t span_o = (int64_t)bpm * p.out_stride + (int64_t)p.M0 * p.out_sm0 +
                         (int64_t)p.N1 * p.out_spn;
  const int64_t span_a = (int64_t)bpm * p.acc_stride + (int64_t)p.M0 * p.acc_sm0 +
                         (int64_t)p.N1 * p.acc_spn;
  if (span_m >= (1ll << 31) || span_n >= (1ll << 31) || span_o >= (1ll << 31) ||
      span_a >= (1ll << 31)) {
    return -1;
  }
  constexpr size_t kLds = 4 * (size_t)BM * KS;
  set_divisors(a);
  auto kernel = mmt4d_mfma_persistent_kernel<E, TM, TN, WGM, WGN>;
  uk::launch(2, kernel, dim3((uint32_t)grid), dim3(WGM * WGN * 64), kLds, stream, a);
  return (int)hipGetLastError();
}

// Launches the narrow-row kernel (mmt4d_mfma_narrow.h: tile rows of 2 or 4
// bytes, N0 = 16, RHS fragments loaded straight into registers) over K-tiles
// [0, kt_count). Returns a HIP status, or -1 if it cannot serve the shape.
template <Elem E, int RBC, int TM, int WGM, int WGN>
int launch_narrow(const Problem& p, int kt_count, hipStream_t stream) {
  constexpr int BM = WGM * TM * 16, BN = WGN * 64, KS = 64;
  if (p.rb != RBC || p.N0 != 16 || p.M0 % (16 / RBC) || p.M0 > BM || BM % p.M0) return -1;
  if (p.dequant) return -1;
  if (p.out_rows <= 0 || p.out_cols <= 0) return 0;
  if (p.out_cols < (int64_t)p.N1 * p.N0) return -1;   // a row-major matrix narrower than the tiles
  const int64_t k_bytes = (int64_t)kt_count << p.lrb;
  if (kt_count <= 0 || k_bytes % KS) return -1;
  Args a{};
  a.lhs = p.lhs; a.rhs = p.rhs; a.out = p.out;
  a.lhs_stride = p.lhs_stride; a.rhs_stride = p.rhs_stride; a.out_stride = p.out_stride;
  a.out_sm0 = (uint32_t)p.out_sm0; a.out_spn = (uint32_t)p.out_spn;
  a.out_rows = (int32_t)std::min<int64_t>(p.out_rows, INT32_MAX);
  a.out_cols = (int32_t)std::min<int64_t>(p.out_cols, INT32_MAX);
  a.M1 = p.M1; a.N1 = p.N1; a.K1 = kt_count;
  a.M0 = p.M0; a.N0 = p.N0; a.rb = p.rb; a.lrb = p.lrb;
  a.bpm = BM / p.M0; a.bpn = BN / p.N0;
  const int64_t grid_m = uk::ceil_div(p.M1, a.bpm), grid_n = uk::ceil_div(p.N1, a.bpn);
  if (grid_m * grid_n >= (1ll << 31)) return -1;
  a.grid_m = (int32_t)grid_m; a.grid_n = (int32_t)grid_n;
  a.steps = (int32_t)(k_bytes / KS);
  a.accumulate = p.accumulate;
  a.band = (WGM == 1 && WGN == 8) ? 8 : 4;
  a.vec_out = 1;
  a.acc = p.acc; a.acc_stride = p.acc_stride;
  a.acc_sm0 = (uint32_t)p.acc_sm0; a.acc_spn = (uint32_t)p.acc_spn;
  const int64_t kt_bytes_m = (int64_t)p.M0 << p.lrb, kt_bytes_n = (int64_t)p.N0 << p.lrb;
  const int64_t span_m = (int64_t)a.bpm * p.lhs_stride + (int64_t)p.K1 * kt_bytes_m;
  const int64_t span_n = (int64_t)a.bpn * p.rhs_stride + (int64_t)p.K1 * kt_bytes_n;
  const int64_t span_o = (int64_t)a.bpm * p.out_stride + (int64_t)p.M0 * p.out_sm0 +
                         (int64_t)p.N1 * p.out_spn;
  const int64_t span_a = (int64_t)a.bpm * p.acc_stride + (int64_t)p.M0 * p.acc_sm0 +
                         (int64_t)p.N1 * p.acc_spn;
  if (span_m >= (1ll << 31) || span_n >= (1ll << 31) || span_o >= (1ll << 31) ||
      span_a >= (1ll << 31)) {
    return -1;
  }
  constexpr size_t kLds = 3 * (size_t)BM * KS;
  set_divisors(a);
  uk::launch(2, mmt4d_mfma_narrow_kernel<E, RBC, TM, WGM, WGN>, dim3((uint32_t)(grid_m * grid_n)),
             dim3(WGM * WGN * 64), kLds, stream, a);
  return (int)hipGetLastError();
}

// Launches the M-thin kernel (mmt4d_mfma_thin.h) over all of K. Returns a HIP
// status, or -1 if it cannot serve the shape.
// `swapped`: the caller's problem is N-thin and is computed as its transpose
// (out^T = rhs * lhs^T): the kernel's rows are the caller's columns.
// A K that ends inside a step is served where TAIL_OK says that there is an
// instance for it.
template <Elem E, int RBC, int TM, int TN, int KSPLIT, int D, bool TAIL_OK = false, int CH = 0>
int launch_thin(const Problem& caller, bool swapped, hipStream_t stream, bool allow_k_slices = false,
                int max_k_slices = 8) {
  constexpr int OBYTES = ElemTraits<E>::Out::kOutBytes;
  Problem p = caller;
  if (swapped) {
    std::swap(p.lhs, p.rhs);
    std::swap(p.lhs_stride, p.rhs_stride);
    std::swap(p.M1, p.N1);
    std::swap(p.M0, p.N0);
    std::swap(p.out_rows, p.out_cols);
    std::swap(p.row_scale, p.col_scale);
    // Element (row i, col j) of the caller sits at
    //   (i / M0) * stride + (i % M0) * sm0 + (j / N0) * spn + (j % N0) * elem;
    // the kernel's row is j and its column is i.
    std::swap(p.out_stride, p.out_spn);
    std::swap(p.acc_stride, p.acc_spn);
  }
  constexpr int KS = 64 * ElemTraits<E>::kHalves;
  constexpr int OB = OBYTES;
  constexpr bool S4 = E == Elem::kS8S4;  // rb, lrb describe the LHS; RHS rows are half as wide
  if (p.rb > KS || p.rb < (S4 ? 16 : std::min(RBC, 8))) return -1;
  const int64_t k_bytes = (int64_t)p.K1 << p.lrb;
  const bool tail = k_bytes % KS != 0;
  if (k_bytes == 0 || (tail && !TAIL_OK)) return -1;
  // 4-bit RHS: the accumulators hold 16 * sum; |sum| <= K * 128 * 8 must stay
  // below 2^27 for that to be exact.
  if (S4 && k_bytes >= 131072) return -1;
  if (p.out_rows <= 0 || p.out_cols <= 0) return 0;
  Args a{};
  a.lhs = p.lhs; a.rhs = p.rhs; a.out = p.out;
  a.lhs_stride = p.lhs_stride; a.rhs_stride = p.rhs_stride; a.out_stride = p.out_stride;
  a.out_sm0 = (uint32_t)(swapped ? OBYTES : p.out_sm0);
  a.out_sn0 = (uint32_t)(swapped ? p.out_sm0 : OBYTES);
  a.out_spn = (uint32_t)p.out_spn;
  a.out_rows = (int32_t)std::min<int64_t>(p.out_rows, INT32_MAX);
  a.out_cols = (int32_t)std::min<int64_t>(p.out_cols, INT32_MAX);
  a.M1 = p.M1; a.N1 = p.N1; a.K1 = p.K1; a.M0 = p.M0; a.N0 = p.N0; a.rb = p.rb; a.lrb = p.lrb;
  // Rows and columns that are stored: blocks wholly beyond them (tile padding of
  // a fused row-major result) are not computed at all.
  const int64_t grid_m = uk::ceil_div(std::min<int64_t>((int64_t)p.M1 * p.M0, p.out_rows), TM * 16);
  const int64_t grid_n = uk::ceil_div(std::min<int64_t>((int64_t)p.N1 * p.N0, p.out_cols), TN * 16);
  if (grid_m * grid_n >= (1ll << 31) || p.out_sm0 >= (1ll << 32) || p.out_spn >= (1ll << 32) ||
      p.acc_sm0 >= (1ll << 32) || p.acc_spn >= (1ll << 32)) {
    return -1;
  }
  a.grid_m = (int32_t)grid_m;
  a.grid_n = (int32_t)grid_n;
  a.steps = (int32_t)uk::ceil_div(k_bytes, (int64_t)KS);
  a.accumulate = p.accumulate;
  a.acc = p.acc; a.acc_stride = p.acc_stride;
  a.acc_sm0 = (uint32_t)(swapped ? OBYTES : p.acc_sm0);
  a.acc_sn0 = (uint32_t)(swapped ? p.acc_sm0 : OBYTES);
  a.acc_spn = (uint32_t)p.acc_spn;
  a.dequant = p.dequant; a.row_scale = p.row_scale; a.col_scale = p.col_scale;
  a.col_scale_first = swapped;
  auto vector_ok = [&](const char* base, int64_t stride, int64_t sm0, int64_t spn) {
    const bool contiguous4 = p.N0 % 4 == 0 || spn == (int64_t)p.N0 * OB;
    const bool aligned4 = OB == 4 || (((uintptr_t)base | (uint64_t)stride | (uint64_t)sm0 |
                                       (uint64_t)spn) % 8) == 0;
    return contiguous4 && aligned4;
  };
  a.vec_out = !swapped && vector_ok(p.out, p.out_stride, p.out_sm0, p.out_spn) &&
              (!p.accumulate || vector_ok(p.acc, p.acc_stride, p.acc_sm0, p.acc_spn));
  // 32-bit operand offsets inside a workgroup's panels.
  const int64_t span_m = (int64_t)(TM * 16 / p.M0 + 2) * p.lhs_stride + k_bytes * p.M0;
  const int64_t span_n =
      (int64_t)(TN * 16 / p.N0 + 2) * p.rhs_stride + k_bytes * p.N0 / (S4 ? 2 : 1);
  if (span_m >= (1ll << 31) || span_n >= (1ll << 31)) return -1;
  // Still too few output blocks for the chip, and a long K: split K over
  // workgroups as well, aiming at one workgroup per compute unit. The split costs
  // 1.5 to 2.5 us at the end of the launch (the slices meet through device-scope
  // accesses, three dependent round trips to where the XCDs meet), so a slice
  // keeps at least as many operand bytes as a workgroup streams in several times
  // that: 192 KB (16 rows, weights not cached: s8 1024 x 16384, 512 KB a block, 10.6
  // -> 9.3 us in two slices; s8 1024 x 4096, 128 KB, 4.7 against 6.2; f16 64 rows
  // 1024 x 4096, 640 KB, 13.8 -> 11.1 in three); 128 KB with 8-byte rows, two loads an
  // operand (s8 1024 x 14336 8.8 us in two slices, 8.2 in three). With so few blocks that
  // most units would idle, 64 KB. In any case 16 steps.
  int64_t kslices = 1;
  if (allow_k_slices) {
    const int64_t blocks = grid_m * grid_n;
    const int cus = p.cus;
    if (k_slices_override() > 0) {
      kslices = k_slices_override();
    } else if (cus > 0 && 2 * blocks <= cus) {
      const int64_t share = k_bytes * 16 * (TM + TN) - (S4 ? k_bytes * 8 * TN : 0);
      const int64_t least = TM * TN >= 16 || 8 * blocks <= cus ? 65536 : RBC == 8 ? 131072 : 196608;
      kslices = std::min<int64_t>(std::min<int64_t>(max_k_slices, cus / blocks), share / least);
    }
    kslices = std::max<int64_t>(1, std::min<int64_t>(kslices, a.steps / 16));
    if (blocks * kslices >= (1ll << 31)) kslices = 1;
  }
  if (kslices > 1) {
    KSplitWorkspace ws{};
    const int got = acquire_ksplit_workspace((size_t)(grid_m * grid_n * kslices) * TM * TN * 1024,
                                             (uint32_t)(grid_m * grid_n), stream, &ws);
    if (got > 1) return got;
    if (got == 0) {
      a.kslices = (uint32_t)kslices;
      a.ws_partials = ws.partials;
      a.ws_counters = ws.counters;
      note_k_slices((int)kslices);
    } else {
      kslices = 1;
    }
  }
  // (An XCD's share in as few bands as keep its blocks in a near-square patch.)
  a.column_bands = grid_n >= grid_m;
  a.band = (uint32_t)std::min<int64_t>(uk::ceil_div(std::max(grid_m, grid_n), (int64_t)8), 8);
  set_divisors(a);
  const dim3 grid((uint32_t)(grid_m * grid_n * kslices)), block(KSPLIT * 64);
  // Rows in twos (PAIRED). 8-byte rows, one a load / RHS in twos / both: four layers of 33 x
  // 14336 x 4096 s8 94.4 / 87.5 / 83.1 us, 16 rows 68.5 / 65.5; f16 32 rows 134 / 120; in 64x64
  // blocks s8 300 x 4096 x 2000 12.7 / 11.1 / 10.1, 2000 x 300 x 4099 12.6 / 11.1 / 10.6, f16 19.3
  // / 16.7, 96 x 4096 x 4096 in 32x64 15.0 / 12.5. 4-byte rows of f32, whose products take a
  // word at a time: 128 x 2048 x 4096 24.0 / 20.0, 96 x 4096 x 4096 38.7 / 33.7, 2000 x 300 x
  // 4099 53.8 / 50.0, 1000 x 1501 x 777 26.4 / 26.0, six blocks a unit, but 1500 x 1500 x 1500,
  // nine, 68.5 / 73. Other types put them together with moves that cost more than the loads:
  // bf16 16x16x2 1000 x 1501 x 777 11.5 / 14.0, s8 16x16x4 96 x 4096 x 4096 9.5 / 10.7. (Tiles
  // of an odd number of such rows are regrouped to rows of 16 bytes before they come here.)
  constexpr bool kPairs8 = TN % 2 == 0 && RBC == 8;
  constexpr bool kPairs4 = TN % 2 == 0 && RBC == 4 && E == Elem::kF32 && KSPLIT > 2;
  // No non-temporal instances where K may end inside a step: weights that the caller has
  // declared streamed are read by several row blocks there, which then wait for HBM one after
  // the other (64x64 blocks, ordinary / non-temporal us: f16 200 x 8192 x 4096 34.6 / 44.5, s8
  // 80 x 8192 x 8192 21.4 / 25.0, 128 x 4096 x 14336 34.9 / 35.6; at best f8 192 x 4096 x 8192
  // 21.6 / 21.1). Else where they are too large for the L2s anyway.
  const bool streamed =
      !TAIL_OK && streamed_weights() && (int64_t)p.N1 * p.N0 * k_bytes / (S4 ? 2 : 1) >= (16ll << 20);
  auto go = [&](auto paired_c) {
    constexpr bool P = decltype(paired_c)::value;
    if constexpr (TAIL_OK) {
      auto kernel = tail ? mmt4d_thin_kernel<E, RBC, TM, TN, KSPLIT, D, false, true, CH, P>
                         : mmt4d_thin_kernel<E, RBC, TM, TN, KSPLIT, D, false, false, CH, P>;
      uk::launch(2, kernel, grid, block, 0, stream, a);
    } else {
      auto kernel = streamed ? mmt4d_thin_kernel<E, RBC, TM, TN, KSPLIT, D, true, false, 0, P>
                             : mmt4d_thin_kernel<E, RBC, TM, TN, KSPLIT, D, false, false, 0, P>;
      uk::launch(2, kernel, grid, block, 0, stream, a);
    }
    return (int)hipGetLastError();
  };
  if constexpr (kPairs4) {
    if (grid_m * grid_n <= 6 * (int64_t)p.cus) return go(std::true_type{});
  }
  return go(std::bool_constant<kPairs8>{});
}

// The thin kernel with TM 16-row blocks against `wide_cols` columns (rows of the
// right-hand side; N-thin problems come transposed). The launch streams the
// weights, so what counts is how evenly they lie on the compute units and how
// many loads a unit has in flight:
//   * one 16-column block a workgroup, its K over eight waves, up to one block a
//     unit, and for up to 16 rows wherever the most loaded unit gets fewer columns
//     that way. us in 1x1 blocks of eight waves against 1x1 / 1x2 of four, weights
//     not cached: s4 4 x 4096 x 16384 11.1 / 15.5 / 15.1; s8 8-byte rows 16 x 2048 x
//     4096 6.5 / 6.8 / 8.4; f16 4 x 4096 x 4096 9.0 / 9.8 / 11.0; f8 4 x 10240 x 4096
//     10.6 / 10.8 / 11.8;
//   * 16 columns over four waves where there are more such blocks than units and K is
//     short, eight steps and less a wave: these are stores and launches of waves (f32 16
//     x 6144 x 1024 6.7, 7.8 in 32 columns; s8 32 x 7168 x 1536 4.9 / 5.6; s8 8-byte rows
//     16 x 10240 x 512 4.2, 5.6 in eight waves). The K up to which they are ahead was
//     measured for each number of rows and row width on 4352 to 20480 columns;
//   * else 32 columns a workgroup over four waves: s8 4 x 6144 x 16384 20.8 against
//     21.2, 32 x 14336 x 4096 15 % and 64 x 14336 x 4096 20 to 40 % ahead (a second
//     column block shares the rows' loads).
// With 16 and fewer rows four steps are in flight in a wave, with more two (their
// registers: 2x1 and 4x1 blocks of eight waves 1 to 5 % ahead of four steps).
template <Elem E, int RBC, int TM>
int launch_thin_rows(const Problem& p, bool swapped, int64_t wide_cols, hipStream_t stream) {
  constexpr int H = ElemTraits<E>::kHalves;
  const int64_t rows = swapped ? std::min<int64_t>((int64_t)p.N1 * p.N0, p.out_cols)
                               : std::min<int64_t>((int64_t)p.M1 * p.M0, p.out_rows);
  const int64_t row_blocks = std::max<int64_t>(1, uk::ceil_div(rows, (int64_t)(TM * 16)));
  const int64_t cus = std::max(p.cus, 1);
  const int64_t blocks16 = row_blocks * uk::ceil_div(wide_cols, (int64_t)16);
  const int64_t blocks32 = row_blocks * uk::ceil_div(wide_cols, (int64_t)32);
  constexpr bool kInteger = std::is_same<typename ElemTraits<E>::Acc, v4i>::value;
  constexpr int64_t kShort = E == Elem::kF32 || TM == 1 ? 4096
                             : TM == 2                  ? (RBC == 8 ? 1024 : 2560)
                             : H == 2                   ? 0
                                                        : (RBC == 8 ? 512 : 1536);
  // (Where eight waves would take a float's K in 32 parts, they do.)
  const int64_t short_k = blocks32 < cus ? kShort : TM == 1 && kInteger ? 1024 : 0;
  if (blocks16 > cus && ((int64_t)p.K1 << p.lrb) <= short_k)
    return launch_thin<E, RBC, TM, 1, 4, 4>(p, swapped, stream, true);
  // (Not for 8-byte rows in twos, whose loads are half as many in 32 columns: s8, 8-byte rows,
  // in 16 columns over eight waves / so, four layers, 4 x 11008 x 4096 64.3 / 60.8 us, 16 x
  // 28672 x 8192 221 / 191. Floats keep the parts of K that eight waves have.)
  constexpr bool paired = kInteger && RBC == 8;
  const bool narrow = blocks16 <= cus ||
                      (TM == 1 && !paired && uk::ceil_div(blocks16, cus) < 2 * uk::ceil_div(blocks32, cus));
  if (narrow) return launch_thin<E, RBC, TM, 1, 8, TM == 1 && H == 1 ? 4 : 2>(p, swapped, stream, true);
  return launch_thin<E, RBC, TM, 2, 4, TM == 4 ? 3 : 4>(p, swapped, stream, true);
}

// The thin kernel for `thin_rows` rows: the fewest 16-row blocks a workgroup that still
// leave at most one workgroup a compute unit, as long as the weights that several row
// blocks then read are no more than what the L2s hold (us, f16 64 x 2048 x 8 KB in one
// 64-row block / two of 32: 10.9 / 7.5; s8 64 x 300 x 4 KB in one / four of 16: 8.3 / 4.1).
template <Elem E, int RBC>
int launch_thin_any(const Problem& p, bool swapped, int64_t thin_rows, int64_t wide_cols, hipStream_t stream) {
  const int64_t cus = p.cus, cols16 = uk::ceil_div(wide_cols, (int64_t)16);
  const bool cached = wide_cols * ((int64_t)p.K1 << p.lrb) <= (16ll << 20);
  if (thin_rows <= 16 || (cached && uk::ceil_div(thin_rows, (int64_t)16) * cols16 <= cus))
    return launch_thin_rows<E, RBC, 1>(p, swapped, wide_cols, stream);
  if (thin_rows <= 32 || (cached && uk::ceil_div(thin_rows, (int64_t)32) * cols16 <= cus))
    return launch_thin_rows<E, RBC, 2>(p, swapped, wide_cols, stream);
  return launch_thin_rows<E, RBC, 4>(p, swapped, wide_cols, stream);
}

// Status of the second, accumulating launch over the remainder of K. The
// first launch has already written the output: "not served" (negative) must
// not reach the dispatcher, which would recompute the whole problem on the
// scalar kernel on top of it.
inline int finish_k(int st) { return st < 0 ? (int)hipErrorUnknown : st; }

// Few 128x128 blocks and a long K: K in slices of the LDS-direct pipeline, each
// slice's sums as a row-major matrix in the K split's workspace, and a second launch
// that adds them up (mmt4d_mfma_sum.h). Returns a HIP status, or -1 where K is no
// whole number of steps, `slices` are too many for it, or there is no workspace (a
// stream under capture, iree_uk_amd_mmt4d_no_alloc with a large result).
template <Elem E, int RBC>
int launch_slices(const Problem& p, int slices, hipStream_t stream) {
  // 16-bit results: the sums of the slices are 32-bit floats like those of a block.
  constexpr Elem P = E == Elem::kF16F16 ? Elem::kF16 : E == Elem::kBF16BF16 ? Elem::kBF16 : E;
  using Out = typename ElemTraits<E>::Out;
  constexpr int KS = 64 * ElemTraits<E>::kHalves;
  const int64_t k_bytes = (int64_t)p.K1 << p.lrb;
  if (p.out_rows <= 0 || p.out_cols <= 0) return 0;
  if (k_bytes % KS || slices < 2 || k_bytes / KS < 16 * slices) return -1;
  const int64_t rows = (int64_t)p.M1 * p.M0, cols = (int64_t)p.N1 * p.N0;
  if (p.out_sm0 >= (1ll << 32) || p.out_spn >= (1ll << 32) || p.acc_sm0 >= (1ll << 32) ||
      p.acc_spn >= (1ll << 32) || rows * cols * slices >= (1ll << 26)) {
    return -1;
  }
  KSplitWorkspace ws{};
  const int got = acquire_ksplit_workspace((size_t)(slices * rows * cols) * 4, 1, stream, &ws);
  if (got != 0) return got > 1 ? got : -1;
  Problem q = p;
  q.out = ws.partials;
  q.out_stride = p.M0 * cols * 4;
  q.out_sm0 = cols * 4;
  q.out_spn = p.N0 * 4;
  q.acc = q.out; q.acc_stride = q.out_stride; q.acc_sm0 = q.out_sm0; q.acc_spn = q.out_spn;
  // What exists of the partial sums are this problem's own rows and columns: of a part of
  // a larger problem the result may have more, and a row here has no room for them.
  q.out_rows = std::min(p.out_rows, rows);
  q.out_cols = std::min(p.out_cols, cols);
  q.accumulate = q.dequant = false;
  int st = launch_variant<P, RBC, 4, 2, 2, 4, 1, 5, true>(q, 0, q.K1, false, stream, slices);
  if (st != 0) return st;
  note_k_slices(slices);
  SumArgs s{};
  s.partials = ws.partials;
  s.slice_bytes = rows * cols * 4;
  s.pitch = cols * 4;
  s.slices = slices;
  s.rows = (int32_t)std::min(rows, p.out_rows);
  s.cols = (int32_t)std::min(cols, p.out_cols);
  s.M0 = p.M0; s.N0 = p.N0;
  s.by_m0 = Divisor::by((uint32_t)p.M0); s.by_n0 = Divisor::by((uint32_t)p.N0);
  s.out = p.out; s.out_stride = p.out_stride;
  s.out_sm0 = (uint32_t)p.out_sm0; s.out_spn = (uint32_t)p.out_spn;
  s.acc = p.accumulate ? p.acc : nullptr; s.acc_stride = p.acc_stride;
  s.acc_sm0 = (uint32_t)p.acc_sm0; s.acc_spn = (uint32_t)p.acc_spn;
  s.dequant = p.dequant; s.row_scale = p.row_scale; s.col_scale = p.col_scale;
  constexpr int OB = Out::kOutBytes;
  auto vector_ok = [&](const char* base, int64_t stride, int64_t sm0, int64_t spn) {
    const bool contiguous4 = p.N0 % 4 == 0 || spn == (int64_t)p.N0 * OB;
    const bool aligned4 = OB == 4 || (((uintptr_t)base | (uint64_t)stride | (uint64_t)sm0 |
                                       (uint64_t)spn) % 8) == 0;
    return contiguous4 && aligned4;
  };
  s.vec = vector_ok(p.out, p.out_stride, p.out_sm0, p.out_spn) &&
          (!p.accumulate || vector_ok(p.acc, p.acc_stride, p.acc_sm0, p.acc_spn));
  const dim3 grid((uint32_t)uk::ceil_div(s.cols, 4 * kSumThreads), (uint32_t)s.rows);
  uk::launch(2, mmt4d_sum_slices_kernel<typename ElemTraits<E>::Acc, Out>, grid, dim3(kSumThreads), 0, stream, s);
  return finish_k((int)hipGetLastError());
}

// Number of workgroups a BM x BN blocking gives for the problem.
inline int64_t workgroups(const Problem& p, int BM, int BN) {
  const int bpm = BM / p.M0, bpn = BN / p.N0;
  if (bpm < 1 || bpn < 1) return 0;
  return uk::ceil_div(p.M1, bpm) * uk::ceil_div(p.N1, bpn);
}

// Steps of loads in flight in a wave of 32x32 to 64x64 blocks: two, three with 8-byte rows
// (3 % ahead of two in 32x32, 4 % in 32x64, 5 % in 64x64 blocks; else 1 to 20 % behind).
template <Elem E, int RBC>
constexpr int steps_ahead() {
  return RBC == 8 ? 3 : 2;
}

// 16x16 blocks, K over their waves, with two steps in flight, with rows of 2 and 4 bytes four
// (s8 16x16x2 12 %, bf16 16x16x2 3 % ahead of two in the mean; 8-byte rows 2 % behind). f32,
// whose products are slower: four, with rows under 16 bytes three (eight 5 to 7 % behind in the
// mean, up to 17 %), of 4 bytes from 20 KB of K on, which the L2s hold no longer, eight (98 x 270 x
// 10742 in three 32.5 us, so 25.2, 84 x 484 x 5767 18.8 / 16.1; but 90 x 265 x 3392 10.0 / 10.4).
template <Elem E, int RBC, int KSPLIT>
int launch_16x16(const Problem& p, hipStream_t stream) {
  if constexpr (E == Elem::kF32) {
    if constexpr (RBC == 4) {
      if (((int64_t)p.K1 << p.lrb) >= 20480) return launch_thin<E, RBC, 1, 1, KSPLIT, 8, true>(p, false, stream);
    }
    return launch_thin<E, RBC, 1, 1, KSPLIT, RBC < 16 ? 3 : 4, true>(p, false, stream);
  } else {
    return launch_thin<E, RBC, 1, 1, KSPLIT, RBC < 8 ? 4 : 2, true>(p, false, stream);
  }
}

// What `blocks` workgroups of a kernel take, in us, by the KB of K. A unit's blocks are
// loaded one beside the other, and a last round of few blocks is not a whole one; below
// `least` blocks a unit a block's own chain of steps is what it takes. Where a unit holds
// `resident` blocks at a time (0: all), those of a last turn take as long as `last` of them.
struct BlockCost {
  double launch, round, k, k_block, least, resident = 0, last = 0;
};
inline double block_us(const BlockCost& c, int64_t cus, int64_t blocks, double kb) {
  const double units = (double)blocks / (double)cus, rounds = std::ceil(units);
  const double whole = c.resident > 0 && units > c.resident ? c.resident * (std::ceil(units / c.resident) - 1) : 0;
  const double rest = std::max(whole > 0 ? c.last : c.least, std::min(rounds, units + 0.6) - whole);
  return c.launch + c.round * rounds + kb * (c.k + c.k_block * (whole + rest));
}

// f32: the barrier-free kernel in 32x32 blocks, K over four waves and over two, in 32x48
// blocks over four, 48x48 over eight; and those it is weighed against: 128x128 blocks, the 64x64
// K split, 64x64 blocks, with rows of 4 bytes and more than 8 KB of K the regrouping ones. Fitted,
// like block_costs below, to 600 to 725 products of 65 to 4096 rows and 256 B to 24 KB of K a class of
// rows (16, 8, 4 bytes); the choice is 0.2 to 0.3 % behind the fastest in the geometric mean.
enum F32Kind { kF32x32, kF32x32Two, kF32x48, kF48x48, kF128x128, kF64x64Split, kF64x64, kF64x64Long, kF32Kinds };
template <int RBC>
inline const BlockCost* f32_costs() {
  static constexpr BlockCost rows16[kF32Kinds] = {
      {2.80, 0.34, 0.18, 0.93, 1.31, 6, 2.80}, {1.02, 0.23, 0.47, 1.08, 4.15, 10, 4.66},
      {3.60, 0.41, 0.03, 1.40, 0.00, 4, 2.53}, {1.66, 2.80, 0.02, 2.06, 1.02, 1, 1.00},
      {3.06, 3.39, 1.22, 13.32, 0.57}, {4.23, 1.94, 0.06, 3.60, 0.95},
      {3.36, 0.73, 0.63, 3.90, 0.95}, {1e30, 0, 0, 0, 0}};
  static constexpr BlockCost rows8[kF32Kinds] = {
      {3.04, 0.27, 0.30, 0.96, 0.00, 5, 3.04}, {2.28, 0.29, 1.00, 0.93, 4.51, 8, 3.00},
      {3.44, 0.69, 0.21, 1.53, 0.56, 5, 1.30}, {1.92, 2.73, 0, 2.25, 0.96, 9, 1.62},
      {2.87, 4.49, 4.10, 14.36, 0.35}, {4.68, 0.15, 0, 3.84, 0.95},
      {3.64, 1.26, 1.11, 4.63, 1.01}, {1e30, 0, 0, 0, 0}};
  static constexpr BlockCost rows4[kF32Kinds] = {
      {2.73, 0.44, 0.31, 0.98, 1.05, 5, 2.22}, {2.76, 0.38, 1.23, 0.86, 0.00, 10, 4.47},
      {3.24, 0.63, 0.30, 1.43, 1.08, 4, 1.61}, {2.02, 2.51, 0, 2.31, 0.97, 9, 1.91},
      {2.62, 4.69, 3.94, 14.31, 0.80}, {1e30, 0, 0, 0, 0},
      {3.49, 1.23, 1.23, 4.51, 0.98}, {3.82, 1.91, 2.86, 3.20, 1.01}};
  return RBC >= 16 ? rows16 : RBC == 8 ? rows8 : rows4;
}

// Problems whose 64x64 blocks leave compute units idle or take a last round that is
// nearly empty: the barrier-free kernel in small blocks, several waves of a block sharing K,
// so that the chain of K steps a wave walks through is short and many more loads are in flight
// than one workgroup a unit keeps. f32, and what launch_by_cost does not choose for. `b128`,
// `ksplit64`, `b32x64`: whether it would be the 128x128 kernels, the 64x64 K split (or what
// takes its place) or 32x64 blocks through LDS otherwise (else 64x64). Any K, any tile rows.
// Returns a HIP status, or -1 where those kernels are the better ones. `parts` (f32): that K split
// would have K in workgroups too, up to 128 parts; up to three 16x16 blocks a unit then have it in
// four or eight waves of sixteen chains, and as small an error (128 x 128 x 6144 41 us, 1.77e-7 /
// 11.3, 1.56e-7; 128 x 1024 x 6144 31.8 / 22.5). us otherwise / in these blocks:
//   one 16x16 block a unit or fewer, from 256 bytes of K (rows under 16 bytes: 64): f16 220 x
//     215, K 512 B 4.5 / 4.2, 7.6 KB 14.9 / 5.4; s8 16x16x2 128 x 512, 100 B 4.4 / 3.8; f32
//     16x16x1 220 x 215, 3 KB 22.1 / 5.9 (there up to three blocks a unit: 374 x 391, 1 KB 11.1
//     / 5.5);
//   f32, whose MFMAs are slow enough to hide the loads of 32x32 blocks, by f32_costs: in the
//     larger blocks a unit's L1 and L2 carry fewer bytes a sum. 16x16x4 515 x 1027 x 768 11.2 (48x48;
//     13.8 in 32x32 blocks before), 3140 x 237 x 2088 35.9 / 28.3 (32x48); 16x16x2 2173 x 674 x 3168
//     95.7 / 77.3 (32x48); 16x16x1 515 x 1027 x 769 12.1 (48x48), 958 x 810 x 690 20.4 / 13.5, 1500 x
//     1500 x 1000 42.8 (32x48), 3582 x 3328 x 1792 382 / 331 (32x32); but 1564 x 1150 x 2621, seven
//     32x32 blocks a unit, of which it holds six at a time, 80 / 91 (64x64);
//   other types, where K ends inside a step of a thin product: two 32x32 blocks a unit or fewer,
//     from 1 KB (8-bit floats, two loads an operand: 7/4; rows of 2 bytes: one).
template <Elem E, int RBC>
int launch_small_blocks(const Problem& p, int64_t rows, int64_t cols, bool b128, bool ksplit64, bool parts,
                        bool b32x64, hipStream_t stream, const char** name) {
  constexpr bool F32 = E == Elem::kF32;
  constexpr int kAhead = steps_ahead<E, RBC>();
  const int64_t k_bytes = (int64_t)p.K1 << p.lrb;
  const int64_t cus = p.cus;
  if (cus < 1) return -1;
  const int64_t b16 = uk::ceil_div(rows, (int64_t)16) * uk::ceil_div(cols, (int64_t)16);
  const int64_t b32 = uk::ceil_div(rows, (int64_t)32) * uk::ceil_div(cols, (int64_t)32);
  int st = -1;
  if constexpr (F32 && RBC >= 8) {   // (choice 6 only)
    if (parts) {
      if (b16 > 3 * cus) return -1;
      st = b16 <= cus ? launch_thin<E, RBC, 1, 1, 8, 4, true, 16>(p, false, stream)
                      : launch_thin<E, RBC, 1, 1, 4, 4, true, 16>(p, false, stream);
      if (st >= 0) *name = "mmt4d_mfma_16x16_ksplit";
      return st;
    }
  }
  if (b16 <= cus && k_bytes >= (RBC < 16 ? 64 : 256)) {
    st = launch_16x16<E, RBC, F32 ? 4 : 8>(p, stream);
    if (st >= 0) *name = "mmt4d_mfma_16x16_ksplit";
    return st;
  }
  if constexpr (F32) {
    // (Below 1 KB of K not with many blocks: rows of 16 bytes more than two 32x32 blocks a unit,
    // others in the place of 128x128 blocks, unless those are more than two a unit: 16x16x2 2988 x
    // 3666 x 218 62.7 us, so 53.6, 16x16x1 63.5 / 55.2, but 2048 x 4096 x 240 42.5 / 45.6.)
    if (k_bytes < ((RBC >= 16 ? b32 > 2 * cus : b128 && workgroups(p, 128, 128) <= 2 * cus) ? 1024 : 256)) return -1;
    if (b16 <= 3 * cus) {
      st = launch_16x16<E, RBC, 4>(p, stream);
      if (st >= 0) *name = "mmt4d_mfma_16x16_ksplit";
      return st;
    }
    const double kb = (double)k_bytes / 1024;
    auto blocks = [&](int bm, int bn) {
      return uk::ceil_div(rows, (int64_t)bm) * uk::ceil_div(cols, (int64_t)bn);
    };
    const BlockCost* costs = f32_costs<RBC>();
    auto us_of = [&](int kind, int64_t n) { return n < 1 ? 1e30 : block_us(costs[kind], cus, n, kb); };
    double us[4] = {us_of(kF32x32, b32), 1e30, us_of(kF32x48, blocks(32, 48)), us_of(kF48x48, blocks(48, 48))};
    // K in two parts instead of four only with many rounds of blocks and few steps, where it
    // was in two before, and not in the place of the 64x64 K split: the error is larger.
    const double rounds = (double)uk::ceil_div(b32, cus), turns = std::min(rounds, (double)b32 / (double)cus + 0.6);
    if (!ksplit64 && (RBC >= 16 ? 0.11 * rounds + 0.04 * kb * turns > 0.05 + 1.2 * kb
                                : 0.09 * rounds + 0.04 * kb * turns > 0.1 + 1.17 * kb)) {
      us[1] = us_of(kF32x32Two, b32);
    }
    if (b32x64) us[2] = us[3] = 1e30;   // (64 rows and fewer)
    static const char* const names[4] = {"mmt4d_mfma_32x32_ksplit", "mmt4d_mfma_32x32_ksplit", "mmt4d_mfma_32x48_ksplit",
                                         "mmt4d_mfma_48x48_ksplit"};
    const int best = (int)(std::min_element(us, us + 4) - us);
    if (b32x64) {
      if (2 * b32 > 7 * uk::ceil_div(workgroups(p, 64, 64), cus) * cus) return -1;
    } else {
      const double other = b128                            ? us_of(kF128x128, workgroups(p, 128, 128))
                           : ksplit64                      ? us_of(kF64x64Split, workgroups(p, 64, 64))
                           : RBC >= 16 || k_bytes <= 8192  ? us_of(kF64x64, workgroups(p, 64, 64))
                                                           : us_of(kF64x64Long, workgroups(p, 64, 64));
      if (us[best] > other) return -1;
    }
    switch (best) {
      case 0: st = launch_thin<E, RBC, 2, 2, 4, kAhead, true>(p, false, stream); break;
      case 1: st = launch_thin<E, RBC, 2, 2, 2, kAhead, true>(p, false, stream); break;
      case 2: st = launch_thin<E, RBC, 2, 3, 4, kAhead, true>(p, false, stream); break;
      default: st = launch_thin<E, RBC, 3, 3, 8, 2, true>(p, false, stream); break;
    }
    if (st >= 0) *name = names[best];
    return st;
  } else {
    // (8-bit floats, two loads an operand: 7/4 blocks a unit, 5/4 with 6 KB of K and more,
    // but in the place of 32x64 blocks. Rows of 2 bytes: one.)
    const int64_t most4 = RBC == 2 ? 4 : ElemTraits<E>::kHalves == 2 && !b32x64 ? (ksplit64 ? 5 : 7) : 8;
    if (4 * b32 > most4 * cus || k_bytes < 1024) return -1;
    st = launch_thin<E, RBC, 2, 2, 4, kAhead, true>(p, false, stream);
  }
  if (st >= 0) *name = "mmt4d_mfma_32x32_ksplit";
  return st;
}

// The kernels between the thin ones and 256x256 blocks, by what they take: the barrier-free
// kernel in blocks of 32x32, 32x64 and 64x64, four waves sharing K; 64x64 blocks with the
// RHS in registers (rows of 2 bytes: regrouped, 256 bytes of K a step); 64x64 and 128x128
// blocks of the LDS-direct pipeline. Fitted, for each class of tile rows, to 1000 products a
// type of 65 to 4096 rows, 65 to 16384 columns, 64 B to 24 KB of K, each on all of these kernels
// with operands that are not cached, for a choice near the fastest (0.1 to 0.6 % behind in the
// geometric mean; single kernels are estimated 4 to 11 % off). us by numbers of blocks / so: f16
// 512 x 2048 x 2048 17.5 / 11.8, 700 x 900 x 1504 11.2 / 8.7, 1500 x 1500 x 1504 20.1 / 18.1; f8
// 900 x 1100 x 1300 8.8 / 6.9; 8-byte rows s8 957 x 2717 x 634 17.5 / 9.2, 2010 x 277 x 2943 13.7 /
// 8.7, f16 3402 x 147 x 2069 19.8 / 13.1; bf16 16x16x2 1000 x 1500 x 784 17.2 / 10.8; s8 16x16x2
// 2000 x 700 x 2000 17.5 / 13.4, 155 x 799 x 1919 7.6 / 6.5. Geometric means of 250 other
// products where the choice differs: 16-byte rows f16 1.25, s8 1.29, bf16 -> bf16 1.35, f8 1.30,
// 8-byte rows 1.58, 4-byte 1.30, 2-byte 1.55; 7 of 2500 are 4 % and more behind, 8 % at worst.
enum BlockKind { k32x32, k32x64, k64x64Split, k64x64, k64x64Lds, k128x128, kBlockKinds };
template <Elem E, int RBC>
inline const BlockCost* block_costs() {
  constexpr double no = 1e30;
  static constexpr BlockCost f8[kBlockKinds] = {{2.62, 0.23, 0.12, 0.67, 1.10}, {2.56, 0.94, 0.29, 0.87, 0},
                                                {1.42, 3.00, 0.16, 1.45, 0.72}, {3.58, 0.57, 0.24, 1.77, 0},
                                                {no, 0, 0, 0, 0}, {3.25, 1.03, 3.53, 2.46, 0.09}};
  static constexpr BlockCost rows16[kBlockKinds] = {{3.06, 0.20, 0.13, 0.59, 0.94}, {3.20, 0.51, 0.32, 0.90, 0.62},
                                                    {3.53, 1.11, 0.18, 1.26, 0.89}, {3.37, 0.54, 1.37, 1.45, 0.38},
                                                    {no, 0, 0, 0, 0}, {5.14, 1.01, 1.20, 2.75, 0.24}};
  static constexpr BlockCost rows8[kBlockKinds] = {{2.74, 0.35, 0.05, 0.71, 1.13}, {3.35, 0.40, 0.29, 1.07, 0.26},
                                                   {3.13, 1.22, 0.50, 1.40, 0.37}, {no, 0, 0, 0, 0},
                                                   {1.09, 4.57, 0.13, 2.02, 0.81}, {3.04, 2.63, 3.02, 1.91, 0.69}};
  static constexpr BlockCost rows4[kBlockKinds] = {{2.94, 0.10, 0.12, 0.93, 0.13}, {3.26, 0.47, 0.10, 1.35, 0.90},
                                                   {3.23, 1.22, 0, 1.82, 1.07}, {no, 0, 0, 0, 0},
                                                   {0.85, 5.24, 0.16, 1.92, 0.84}, {2.93, 2.54, 2.92, 2.10, 0.71}};
  static constexpr BlockCost rows2[kBlockKinds] = {{1.90, 0.96, 0.38, 1.58, 0.96}, {2.97, 0.97, 0.20, 2.66, 0.89},
                                                   {no, 0, 0, 0, 0}, {3.10, 0.83, 0.25, 2.58, 1.40},
                                                   {1.96, 3.68, 0.12, 1.97, 0.07}, {3.84, 0.82, 1.87, 2.83, 0.11}};
  return ElemTraits<E>::kHalves == 2 ? f8 : RBC >= 16 ? rows16 : RBC == 8 ? rows8 : RBC == 4 ? rows4 : rows2;
}
// `parts`: a float's K stays in four parts, as it is in kernels whose waves share it and in
// the 64x64 blocks in registers.
template <Elem E, int RBC>
int launch_by_cost(const Problem& p, int64_t rows, int64_t cols, bool parts, hipStream_t stream, const char** name) {
  static_assert(E != Elem::kF32, "launch_small_blocks");
  constexpr bool kInteger = std::is_same<typename ElemTraits<E>::Acc, v4i>::value;
  const int64_t k_bytes = (int64_t)p.K1 << p.lrb, cus = p.cus;
  if (cus < 1) return -1;
  if (uk::ceil_div(rows, (int64_t)16) * uk::ceil_div(cols, (int64_t)16) <= cus && k_bytes >= (RBC < 16 ? 64 : 256)) {
    const int st = launch_16x16<E, RBC, 8>(p, stream);
    if (st >= 0) { *name = "mmt4d_mfma_16x16_ksplit"; return st; }
  }
  // (LDS blocks hold whole panels, the others need not)
  const int64_t r32 = uk::ceil_div(rows, (int64_t)32), r64 = uk::ceil_div(rows, (int64_t)64);
  const int64_t c32 = uk::ceil_div(cols, (int64_t)32), c64 = uk::ceil_div(cols, (int64_t)64);
  const int64_t b64 = workgroups(p, 64, 64), b128 = workgroups(p, 128, 128);
  const int64_t blocks[kBlockKinds] = {r32 * c32, r32 * c64, r64 * c64, b64, b64, b128};
  const double kb = (double)k_bytes / 1024;
  double us[kBlockKinds];
  for (int k = 0; k < kBlockKinds; ++k) {
    us[k] = blocks[k] < 1 ? 1e30 : block_us(block_costs<E, RBC>()[k], cus, blocks[k], kb);
    // (The 64x64 blocks in registers have a float's K in four parts from 96 steps on. 8-bit
    // floats: the matrix instructions round to 1.5e-5, however K is divided.)
    if (parts && !kInteger && ElemTraits<E>::kHalves == 1 && k > k64x64Split &&
        !(k == k64x64 && RBC >= 16 && k_bytes >= 6144)) {
      us[k] = 1e30;
    }
  }
  // With less than 1 KB of K a block of 128x128 is its stores, estimated low (f16 3428 x 704 x
  // 132 in 64x64 blocks 6.3 us, in these 7.6).
  if (k_bytes < 1024 && b128 < 192) us[k128x128] = 1e30;
  // With 256 bytes of K, of which some waves of the barrier-free blocks get no step, and more than
  // four 32x32 blocks a unit, launching and adding up those is what they take: f8 1090 x 1412 x
  // 105 6.3 us, so 4.9, s8 716 x 2957 x 256 7.8 / 6.5. (16-bit results, of which the 64x64 blocks
  // store half as much at a time, only from eight to twelve blocks a unit on. 16-bit floats, whose
  // sums of 64 to 128 products in one chain are 1.05 to 1.26 times as far off as in four, with one
  // step only.)
  constexpr int64_t kShort = kInteger || ElemTraits<E>::kHalves == 2 ? 256 : 64;
  if (RBC >= 16 && ElemTraits<E>::Out::kOutBytes == 4 && k_bytes <= kShort && r32 * c32 > 4 * cus)
    us[k32x32] = us[k32x64] = us[k64x64Split] = 1e30;
  // 2-byte results: the LDS-direct 64x64 shape takes K in whole steps.
  if (ElemTraits<E>::Out::kOutBytes == 2 && k_bytes % 256 != 0) us[k64x64Lds] = 1e30;
  for (;;) {
    const int k = (int)(std::min_element(us, us + kBlockKinds) - us);
    if (us[k] >= 1e30) return -1;
    us[k] = 1e30;
    int st = -1;
    if (k == k32x32) {
      st = launch_thin<E, RBC, 2, 2, 4, steps_ahead<E, RBC>(), true>(p, false, stream);
      if (st >= 0) *name = "mmt4d_mfma_32x32_ksplit";
    } else if (k == k32x64) {
      st = launch_thin<E, RBC, 2, 4, 4, steps_ahead<E, RBC>(), true>(p, false, stream);
      if (st >= 0) *name = "mmt4d_mfma_32x64_ksplit";
    } else if (k == k64x64Split) {
      if constexpr (RBC >= 4) st = launch_thin<E, RBC, 4, 4, 4, steps_ahead<E, RBC>(), true>(p, false, stream);
      if (st >= 0) *name = "mmt4d_mfma_64x64_ksplit";
    } else if (k == k64x64) {
      if constexpr (RBC >= 16) st = launch_variant<E, RBC, 2, 2, 2, 2, 1, 3>(p, 0, p.K1, p.accumulate, stream);
      else st = launch_variant<E, RBC, 2, 2, 2, 2, 4 / ElemTraits<E>::kHalves, 4>(p, 0, p.K1, p.accumulate, stream);
      if (st >= 0) *name = RBC >= 16 ? "mmt4d_mfma_64x64_rhs_direct" : "mmt4d_mfma_64x64_deep";
    } else if (k == k64x64Lds) {
      if constexpr (RBC < 16) st = launch_variant<E, RBC, 2, 1, 2, 4, 4, 5>(p, 0, p.K1, p.accumulate, stream);
      if (st >= 0) *name = "mmt4d_mfma_64x64_lds_direct";
    } else {
      st = launch_variant<E, RBC, 4, 2, 2, 4, 1, 5>(p, 0, p.K1, p.accumulate, stream);
      if (st >= 0) *name = "mmt4d_mfma_128x128_lds_direct";
    }
    if (st >= 0) return st;
  }
}

// K slices for launch_slices, one workgroup a compute unit or fewer; 0 where the blocks
// that a problem of few 128x128 blocks and 6 KB of K and more has otherwise take less.
// A 64x64 block loads 128 rows of K for 64x64 sums, at 2 us a KB whatever the type: each
// unit's L1 and L2 traffic bounds these calls. A 128x128 block needs half as much for
// each sum, but then the slices' sums pass through memory (a write and a read of 4 bytes
// each) and a second launch. The constants are fitted to 30 calls with weights from HBM,
// and lie on the side of the blocks in place where the two are close. us before / in
// slices (how many):
//   bf16 -> bf16 200 x 4096 x 14336 59.9 / 45.1 (4), 128 x 4096 x 14336 50.3 / 34.1 (8),
//     300 x 4096 x 8192 52.6 / 43.1 (2), 100 x 14336 x 4096 43.6 / 36.3 (2)
//   f16 512 x 2048 x 16384 61.9 / 49.5 (4), 256 x 8192 x 8192 66.5 / 52.7 (2), 512 x 512 x
//     16384 29.2 / 22.3 (16), 70 x 16384 x 4096 45.0 / 36.2 (2)
//   s8 256 x 2048 x 16384 30.8 / 22.6 (8), 512 x 4096 x 8192 33.9 / 31.1 (2), 8-byte rows 200
//     x 4096 x 14336 41.2 / 29.9 (4); f8 512 x 4096 x 8192 41.5 / 31.8 (2)
//   but f16 640 x 3072 x 3072 24.8 / 26.6 (2), f8 128 x 8192 x 8192 26.8 / 28.9 (4), f16 256 x
//     1024 x 4096 9.5 / 15.4 (8)
// A slice has 2 KB of K at least, with 24 KB of K and more 1.5 KB, where 32 64x64 blocks
// have K in 32 parts: 16 slices of two sums each are as many (f16 128 x 1024 x 12288, 26.3
// us and an error of 1.45e-7 there, 20.1 and 1.58e-7 in 12 slices, 18.9 and 1.43e-7 in 16;
// 8-bit floats, whose matrix instructions round to 1.5e-5, stay at 16 steps and 2 KB).
template <Elem E, int RBC>
int slices_that_pay(const Problem& p, int64_t rows, int64_t cols, bool long_k) {
  const int64_t cus = p.cus;
  const int64_t k_bytes = (int64_t)p.K1 << p.lrb, b128 = workgroups(p, 128, 128);
  const int64_t b64 = workgroups(p, 64, 64);
  const int64_t b32 = uk::ceil_div(rows, (int64_t)32) * uk::ceil_div(cols, (int64_t)32);
  const int64_t b16 = uk::ceil_div(rows, (int64_t)16) * uk::ceil_div(cols, (int64_t)16);
  // (With fewer than 32 64x64 blocks K is in more parts there than it would be here.)
  if (cus < 1 || b128 < 1 || b64 < 32 || b16 <= cus) return 0;
  const int64_t least_k = long_k && ElemTraits<E>::kHalves == 1 ? 1536 : 2048;
  const int64_t slices = std::min<int64_t>(std::min<int64_t>(cus / b128, 16), k_bytes / least_k);
  if (slices < 2) return 0;
  const double kb = (double)k_bytes / 1024;
  const double here = 5 + 4.3 * kb / (double)slices + 2.4e-6 * (double)(slices * rows * cols);
  const double units = (double)b64 / (double)cus;
  double blocks = 2 + (RBC == 8 ? 2.8 : 2.05) * kb * std::max(1.0, std::min(std::ceil(units), units + 0.3));
  if (!long_k && b32 <= 2 * cus) blocks = 2 + 0.9 * kb * (double)uk::ceil_div(b32, cus);
  else if (long_k && 2 * b64 <= cus) blocks = 15 + 2.05 * kb / (double)(cus / b64);
  return here < blocks ? (int)slices : 0;
}

// Whether 64x64 blocks with less than 8 KB of K, or with a K that ends inside a step, are
// faster in the kernels that stage through LDS than with K over the waves of a block,
// whose operands pass through the L1s twice as often: from about one block a unit on, 16-bit
// results earlier, 8-bit floats always (their two loads an operand bound the K split). us
// in them / K over the waves: f16 2159 x 786 x 3602 25.1 / 35.7, 3124 x 410 x 8936 55.9 / 82.2;
// bf16 -> bf16 2308 x 521 x 3072 22.0 / 34.8; s8 2898 x 418 x 7936 26.8 / 38.0, 8-byte rows 1083
// x 950 x 16353 37.8 / 42.6; f8 508 x 1287 x 6400 12.9 / 19.7. Up to one block a unit (results
// of 2 bytes and 8-byte rows 3/4) K over the waves is 1.11
// times as fast in the geometric mean of 69 calls, 0.85 at worst; 175 others 1.20 times as
// fast in these kernels, 0.82 at worst.
template <Elem E, int RBC>
bool direct_before_ksplit(const Problem& p) {
  constexpr bool kInteger = std::is_same<typename ElemTraits<E>::Acc, v4i>::value;
  if (E == Elem::kF32 || !(RBC >= 16 || (RBC == 8 && kInteger))) return false;
  const int64_t k_bytes = (int64_t)p.K1 << p.lrb, b64 = workgroups(p, 64, 64), cus = p.cus;
  if (k_bytes >= 8192 && k_bytes % (64 * ElemTraits<E>::kHalves) == 0) return false;
  if (ElemTraits<E>::kHalves == 2) return k_bytes < 24576 || 2 * b64 > cus;   // (else in workgroups, too)
  return 8 * b64 > (ElemTraits<E>::Out::kOutBytes == 2 || RBC == 8 ? 6 : 8) * cus;
}

// Variant choice for row-bytes class RBC:
//   big   256x256 workgroup tile, 8 waves of 128x64, software-pipelined, both
//         operands through LDS-direct loads, any K; f32: RHS straight to
//         registers, any K, or with rows under 16 bytes both operands regrouped
//         in registers, where a remainder of K is a second, accumulating launch;
//   mid   128x128, 8 waves (f32 rows under 16 bytes: 4), any K;
//   small 64x64, 4 or 8 waves, any K: for problems with too few 128x128 blocks to
//         occupy the 256 CUs;
// `forced` (1 big, 2 mid, 3 small, 4 thin, 5 thin on the transposed problem,
// 6 the 64x64 K-split kernel, 7 the 256x128 shape, 8 the 128x512 shape,
// 9 / 10 the persistent kernel in the 128x512 / 256x256 shape, 11 the 64x64
// shape with 256-byte steps three steps ahead (tile rows under 16 bytes),
// 12 .. 15 the narrow-row kernel (tile rows of 2 or 4 bytes, N0 = 16) in the
// 256x256 / 128x512 / 128x128 / 64x64 shape, 16 / 17 / 18 / 19 the LDS-direct
// ping-pong pipeline in the 256x256 / 128x512 / 128x128 / 64x64 shape, 20 in the
// 256x128 shape, 21 the K slices of launch_slices, as many as
// iree_uk_amd_set_k_slices says; 0 = choose) overrides the size heuristic for tests
// and tuning.
//   thin  M-thin (decode-shaped) problems, up to 64 rows, which are bound by
//         streaming the RHS: the barrier-free kernel of mmt4d_mfma_thin.h (16,
//         32 or 64 rows x 16 or 32 columns per workgroup, K split over its 4 or
//         8 waves: launch_thin_rows) when rows are at least 8 bytes wide and K
//         is a whole number of steps. Else launch_small_blocks where that serves
//         (a K that ends inside a step, rows of 2 bytes and more), else 32 rows x 64
//         columns through LDS with loads three steps ahead.
template <Elem E, int RBC>
int launch_class(const Problem& p, int forced, hipStream_t stream, const char** name) {
  constexpr int H = ElemTraits<E>::kHalves;
  constexpr int NKK2 = 2 / H;             // 128 bytes of K per step
  // Three RHS fragment buffers fit the register file only with one fragment
  // register quad per block (all types but f8).
  constexpr int BIG_PIPE = RBC >= 16 ? (ElemTraits<E>::kHalves == 1 ? 3 : 2) : 1;
  constexpr int BIG_KS = 64 * H;
  // Rows / columns that exist in the result (fewer than the tiles hold when a
  // fused call drops tile padding: a decode step of 16 rows in 32-row tiles).
  const int64_t rows_m = std::min<int64_t>((int64_t)p.M1 * p.M0, p.out_rows);
  const int64_t cols_n = std::min<int64_t>((int64_t)p.N1 * p.N0, p.out_cols);
  int choice;
  if (forced == 11 || forced == 15) {
    choice = 3;  // 64x64: the deep pipeline (11) or the narrow-row kernel (15)
  } else if (forced == 12 || forced == 13) {
    choice = 1;  // the narrow-row kernel in the 256x256 (12) or 128x512 (13) shape
  } else if (forced == 14) {
    choice = 2;  // the narrow-row kernel in the 128x128 shape
  } else if (forced == 16 || forced == 17) {
    choice = 1;  // the LDS-direct ping-pong pipeline in the 256x256 (16) or 128x512 (17) shape
  } else if (forced == 20) {
    choice = 7;  // the same pipeline in the 256x128 shape
  } else if (forced == 18) {
    choice = 2;  // the same pipeline in the 128x128 shape
  } else if (forced == 19) {
    choice = 3;  // and in the 64x64 shape with 256-byte steps
  } else if (forced >= 8 && forced <= 10) {
    // The big variant in its 128x512 shape (8), the persistent kernel in that
    // shape (9) or in the square one (10); the plain square shape where the
    // requested one cannot serve.
    choice = 1;
  } else if (forced == 21) {
    choice = 6;  // K in slices over 128x128 blocks, where they serve
  } else if (forced >= 1 && forced <= 7) {
    choice = forced;
  } else if (rows_m <= (RBC >= 8 ? 64 : 32) && workgroups(p, 32, 64) >= 1) {
    choice = 4;
  } else if (RBC >= 8 && cols_n <= 64) {
    choice = 5;
  } else if (workgroups(p, 256, 256) >= 192) {
    choice = 1;
  } else if (RBC >= 16 && workgroups(p, 256, 128) >= 192 && workgroups(p, 256, 128) <= 256) {
    // One round of 256x128 blocks (measured 5-7 % ahead of 128x128 there).
    choice = 7;
  } else if (workgroups(p, 128, 128) >= 192) {
    choice = 2;
  } else if (RBC >= 8 && ((int64_t)p.K1 << p.lrb) >= 6144) {
    // Measured: with 6 KiB of K per row and more, the 64x64 blocks' operands
    // outgrow the L2 and the K-split kernel's deeper queue of loads wins (f16 1000
    // x 1000, 7.6 KB: 21.8 -> 17.1 us).
    choice = 6;
  } else {
    choice = 3;
  }
  // K of less than one step fills no pipeline, and the smaller blocks, several to
  // a unit, overlap their prologues and stores (s8 16x16x2 7070 x 2547 x 16: 21.9
  // us in 256x256 blocks, 17.5 in 128x128).
  if (forced == 0 && (choice == 1 || choice == 7) && ((int64_t)p.K1 << p.lrb) < BIG_KS) choice = 2;
  if (choice == 1 && forced == 0) {
    // Tile quantization: a last row or column of 256x256 workgroups that is
    // mostly padding can cost a whole extra round on the 256 CUs. Compare, in
    // units of one round of big tiles, keeping it in the big launch against
    // splitting it off as a strip that the smaller variants compute (at
    // roughly 0.45 of the big variant's rate, and never faster than about a
    // quarter round: their K loop is as long).
    const int bpm = 256 / p.M0, bpn = 256 / p.N0;
    const int64_t gm_c = uk::ceil_div(p.M1, bpm), gn_c = uk::ceil_div(p.N1, bpn);
    const int64_t gm_f = p.M1 / bpm, gn_f = p.N1 / bpn;
    auto rounds = [](int64_t wgs) { return (double)uk::ceil_div(wgs, 256); };
    auto strip_cost = [&](int64_t panels_m, int64_t panels_n) {
      const double tiles = (double)(panels_m * p.M0) * (double)(panels_n * p.N0) / 65536.0;
      return std::max(0.25, tiles / 256.0 / 0.45);
    };
    double best = rounds(gm_c * gn_c);
    int split_m = 0, split_n = 0;
    for (int fm = 0; fm < 2; ++fm) {
      for (int fn = 0; fn < 2; ++fn) {
        if (!fm && !fn) continue;
        if (fm && (gm_f == 0 || gm_f == gm_c)) continue;
        if (fn && (gn_f == 0 || gn_f == gn_c)) continue;
        const int64_t gm = fm ? gm_f : gm_c, gn = fn ? gn_f : gn_c;
        double cost = rounds(gm * gn);
        const int64_t main_n = fn ? gn_f * bpn : p.N1;
        if (fn) cost += strip_cost(p.M1, p.N1 - main_n);
        if (fm) cost += strip_cost(p.M1 - gm_f * bpm, main_n);
        if (cost < best - 0.1) { best = cost; split_m = fm; split_n = fn; }
      }
    }
    int32_t main_m = split_m ? (int32_t)(gm_f * bpm) : p.M1;
    int32_t main_n = split_n ? (int32_t)(gn_f * bpn) : p.N1;
    if constexpr (RBC >= 16) {
      // Round quantization of the 128x512 shape: a problem it tiles exactly
      // whose last round of blocks fills at most half of the compute units
      // runs those block columns as a launch of their own, which then takes a
      // smaller shape that occupies every unit (f8 2048 x 28672 x 8192, 3.5
      // rounds: 392-399 us as one launch, 313 us for three rounds + 62 us for
      // the last 4096 columns in 256x128 blocks).
      const int bpm_w = 128 / p.M0, bpn_w = 512 / p.N0;
      if (!split_m && !split_n && bpm_w >= 1 && bpn_w >= 1 && p.M1 % bpm_w == 0 && p.N1 % bpn_w == 0) {
        const int64_t gm = p.M1 / bpm_w, gn = p.N1 / bpn_w, cus = p.cus;
        const int64_t rem = cus > 0 ? (gm * gn) % cus : 0;
        if (gm * gn > cus && rem > 0 && 2 * rem <= cus && rem % gm == 0) {
          split_n = 1;
          main_n = (int32_t)((gn - rem / gm) * bpn_w);
        }
      }
    }
    if (split_m || split_n) {
      // Each part has the rows and columns of its own panels and no more: kernels
      // store groups of four columns whole where as many exist, and a part may end
      // inside a group (tiles of 7, 9 or 10 columns).
      const int64_t own_rows = std::min(p.out_rows, (int64_t)main_m * p.M0);
      const int64_t own_cols = std::min(p.out_cols, (int64_t)main_n * p.N0);
      Problem q = p;
      q.M1 = main_m;
      q.N1 = main_n;
      q.out_rows = own_rows;
      q.out_cols = own_cols;
      int st = launch_class<E, RBC>(q, 0, stream, name);
      if (st != 0) return st;
      const char* strip_name = nullptr;
      if (split_n) {  // columns [main_n, N1), all rows
        q = p;
        q.rhs = p.rhs + (int64_t)main_n * p.rhs_stride;
        q.out = p.out + (int64_t)main_n * p.out_spn;
        q.acc = p.acc + (int64_t)main_n * p.acc_spn;
        if (p.col_scale) q.col_scale = p.col_scale + (int64_t)main_n * p.N0;
        q.out_cols = p.out_cols - (int64_t)main_n * p.N0;
        q.N1 = p.N1 - main_n;
        st = launch_class<E, RBC>(q, 0, stream, &strip_name);
        // The main part has run: "not served" must not reach the caller, who
        // would recompute (and with ACCUMULATE, re-add) the whole problem.
        if (st != 0) return st < 0 ? (int)hipErrorUnknown : st;
      }
      if (split_m) {  // rows [main_m, M1), columns [0, main_n)
        q = p;
        q.lhs = p.lhs + (int64_t)main_m * p.lhs_stride;
        q.out = p.out + (int64_t)main_m * p.out_stride;
        q.acc = p.acc + (int64_t)main_m * p.acc_stride;
        if (p.row_scale) q.row_scale = p.row_scale + (int64_t)main_m * p.M0;
        q.out_rows = p.out_rows - (int64_t)main_m * p.M0;
        q.out_cols = own_cols;
        q.M1 = p.M1 - main_m;
        q.N1 = main_n;
        st = launch_class<E, RBC>(q, 0, stream, &strip_name);
        if (st != 0) return st < 0 ? (int)hipErrorUnknown : st;
      }
      return 0;
    }
  }
  // The pipelines that need K in whole steps get those; what is left of K (less
  // than one step) goes to the two-stage variant of the same or a smaller
  // workgroup shape, as a second, accumulating launch: large f32 products in tile
  // rows under 16 bytes, and forced variants. (All others run any K, see
  // has_tail_instance: a second launch over less than one step cost as much as a
  // small product, and a pass over the output: s8 300 x 500 x 400 10.6 -> 5.5 us,
  // f16 3000 x 3000 x 333 40.1 -> 18.7, s8 4095 x 2049 x 2049 53.6 -> 31.2.)
  const int kts_per_step = BIG_KS >> p.lrb;
  // 16-bit outputs are rounded once, after all of K (the reference's
  // SKIP_INTERMEDIATE_ROUNDINGS semantics): a second launch would continue from
  // a rounded value. With a K remainder they take the variants that run any K
  // in one launch.
  constexpr bool kOneLaunchOnly = ElemTraits<E>::Out::kOutBytes == 2;
  int kt_main = kts_per_step > 0 ? (p.K1 / kts_per_step) * kts_per_step : 0;
  if (kOneLaunchOnly && kt_main != p.K1) kt_main = 0;
  constexpr bool NARROW = (RBC == 2 || RBC == 4) && H == 1 && ElemTraits<E>::Out::kOutBytes == 4;
  if (choice == 1) {
    if constexpr (RBC < 16 && H == 1) {
      // Tile rows of 2, 4 or 8 bytes through the LDS-direct ping-pong pipeline
      // (PIPE 5 of mmt4d_mfma_kernel.h: the loads copy the K-tiles as they lie
      // in memory, the fragment reads gather each row's pieces).
      // Measured against the register-regrouping kernels at 8192^3: s8 16x16x2
      // 496 -> 382 us, bf16 16x16x2 932 -> 726 us, s8 16x16x8 486 -> 383 us; at
      // 4096^3 s8 16x16x2 76 -> 57 us. (f32 keeps its kernels, as below.)
      if (forced == 16 || forced == 17 || (forced == 0 && E != Elem::kF32)) {
        int st = -1;
        if (forced == 17) {
          st = launch_variant<E, RBC, 8, 4, 1, 8, 1, 5>(p, 0, p.K1, p.accumulate, stream);
          if (st == 0) *name = "mmt4d_mfma_128x512_lds_direct";
        }
        if (st < 0) {
          st = launch_variant<E, RBC, 8, 4, 2, 4, 1, 5>(p, 0, p.K1, p.accumulate, stream);
          if (st == 0) *name = "mmt4d_mfma_256x256_lds_direct";
        }
        if (st >= 0) return st;
      }
    }
    if constexpr (NARROW) {
      // Tile rows of 2 or 4 bytes with N0 = 16 (the x86-style tiles): the RHS
      // goes straight to registers here too (mmt4d_mfma_narrow.h).
      // Measured: at 8192^3 (four rounds of blocks) it is ahead of the kernel
      // with both operands through LDS (s8 16x16x2: 540 us against 558 us,
      // bf16 16x16x2: 880 us against 955 us), at 4096^3 (one round) behind it
      // (76 us against 69 us, 122 us against 117 us), so it is chosen from two
      // rounds on. The square shape is the faster one for 2-byte rows (540 us
      // against 567 us) and equal to the wide one for 4-byte rows, so the wide
      // shape is taken only when asked for.
      if (kt_main > 0 && ((forced == 0 && workgroups(p, 256, 256) >= 512) || forced == 12 || forced == 13)) {
        int st = -1;
        const char* nm = "";
        if (forced == 13) {
          st = launch_narrow<E, RBC, 8, 1, 8>(p, kt_main, stream);
          nm = "mmt4d_mfma_128x512_narrow";
        }
        if (st < 0 && forced != 13) {
          st = launch_narrow<E, RBC, 8, 2, 4>(p, kt_main, stream);
          nm = "mmt4d_mfma_256x256_narrow";
        }
        if (st == 0) {
          *name = nm;
          if (kt_main == p.K1) return 0;
          return finish_k(launch_variant<E, RBC, 4, 4, 2, 2, NKK2, 0>(p, kt_main, p.K1 - kt_main, true, stream));
        }
        if (st > 0) return st;
      }
    }
    if constexpr (RBC >= 16) {
      // Both operands through LDS-direct loads, two wave groups alternating
      // between memory and compute phases (PIPE 5 of mmt4d_mfma_kernel.h): the
      // default for the big problems of the 8- and 16-bit types (s8 8192^3
      // 413 -> 388 us, bf16 8192^3 779 -> 718 us, f16 4096^3 102 -> 98 us, f8
      // 8192^3 415 -> 390 us against the register-direct-RHS pipeline in its
      // best shape). f32
      // keeps that pipeline (matrix-pipe bound there: 925 against 959 us).
      constexpr bool kDefault = E != Elem::kF32;
      int st = -1;
      if (forced == 17) {
        st = launch_variant<E, RBC, 8, 4, 1, 8, 1, 5>(p, 0, p.K1, p.accumulate, stream);
        if (st == 0) *name = "mmt4d_mfma_128x512_lds_direct";
      }
      if (st < 0 && (forced == 16 || forced == 17 || (forced == 0 && kDefault))) {
        st = launch_variant<E, RBC, 8, 4, 2, 4, 1, 5>(p, 0, p.K1, p.accumulate, stream);
        if (st == 0) *name = "mmt4d_mfma_256x256_lds_direct";
      }
      if (st >= 0) return st;
    }
    if (kt_main > 0) {
      int st = -1;
      bool wide = false;
      const int kt_big = E == Elem::kF32 && BIG_PIPE == 3 ? p.K1 : kt_main;  // (runs any K)
      if constexpr (RBC >= 16 && H == 1 && ElemTraits<E>::Out::kOutBytes == 4) {
        // One persistent workgroup per CU whose pipeline runs across block
        // boundaries. Measured equal to the one-block-per-workgroup launches
        // below (s8 8192^3: 410-420 us either way: the time is not in the block
        // boundaries), so it is taken only when asked for.
        if (forced == 9) {
          st = launch_persistent<E, 8, 4, 1, 8>(p, kt_main, true, stream);
          if (st == 0) *name = "mmt4d_mfma_128x512_persistent";
        }
        if (st < 0 && forced == 10) {
          st = launch_persistent<E, 8, 4, 2, 4>(p, kt_main, true, stream);
          if (st == 0) *name = "mmt4d_mfma_256x256_persistent";
        }
        if (st == 0) {
          if (kt_main == p.K1) return 0;
          return finish_k(launch_variant<E, RBC, 4, 4, 2, 2, NKK2, 0>(p, kt_main, p.K1 - kt_main, true, stream));
        }
        if (st > 0) return st;
      }
      if constexpr (RBC >= 16) {
        // 128 rows x 512 columns, the 8 waves side by side (each 128x64): no two
        // waves load the same RHS fragments and the LDS holds half as much LHS,
        // i.e. fewer bytes moved per MFMA, which is what a power-bound kernel
        // is short of (8192^3 s8 418-423 -> 403-412 us, 4096^3 f16 101 -> 98 us,
        // 8192^3 f8 401-408 -> 389 us, 8192^3 bf16 unchanged). Taken where it tiles the problem exactly;
        // ragged problems keep the square shape and its strip logic.
        const int bpm_w = 128 / p.M0, bpn_w = 512 / p.N0;
        if (forced == 8 || (forced == 0 && bpm_w >= 1 && bpn_w >= 1 && p.M1 % bpm_w == 0 &&
                            p.N1 % bpn_w == 0 && workgroups(p, 128, 512) >= 192)) {
          st = launch_variant<E, RBC, 8, 4, 1, 8, 1, BIG_PIPE>(p, 0, kt_big, p.accumulate, stream);
          wide = st == 0;
        }
      }
      if (st < 0) {
        st = launch_variant<E, RBC, 8, 4, 2, 4, 1, BIG_PIPE>(p, 0, kt_big, p.accumulate, stream);
      }
      if (st == 0) {
        *name = wide ? "mmt4d_mfma_128x512_rhs_direct"
                     : (RBC >= 16 ? "mmt4d_mfma_256x256_rhs_direct" : "mmt4d_mfma_256x256_regroup");
        if (kt_big == p.K1) return 0;
        return finish_k(launch_variant<E, RBC, 4, 4, 2, 2, NKK2, 0>(p, kt_main, p.K1 - kt_main, true, stream));
      }
      if (st > 0) return st;
    }
    choice = 2;
  }
  if (choice == 7) {
    // 256 rows x 128 columns, 8 waves of 128x32: for problems with too few
    // 256x256 blocks to fill the CUs; moves fewer L1 bytes per MFMA than the
    // 128x128 shape.
    if constexpr (RBC >= 16) {
      if (forced == 20 || (forced == 0 && E != Elem::kF32)) {
        int st = launch_variant<E, RBC, 8, 2, 2, 4, 1, 5>(p, 0, p.K1, p.accumulate, stream);
        if (st == 0) *name = "mmt4d_mfma_256x128_lds_direct";
        if (st >= 0) return st;
      }
      int st = launch_variant<E, RBC, 8, 2, 2, 4, 1, 3>(p, 0, p.K1, p.accumulate, stream);
      if (st == 0) *name = "mmt4d_mfma_256x128_rhs_direct";
      if (st >= 0) return st;
    }
    choice = 2;
  }
  // (With 24 KB of K and more the 64x64 blocks below split K over workgroups.)
  const bool long_k = ((int64_t)p.K1 << p.lrb) >= 24576;
  if constexpr (RBC >= 8 && E != Elem::kF32) {
    if (choice == 6 && (forced == 21 || (forced == 0 && k_slices_override() == 0))) {
      const int slices = forced == 21 ? k_slices_override() : slices_that_pay<E, RBC>(p, rows_m, cols_n, long_k);
      const int st = launch_slices<E, RBC>(p, slices, stream);
      if (st >= 0) { *name = "mmt4d_mfma_128x128_kslices"; return st; }
    }
  }
  const bool splits_k = long_k && (E != Elem::kF32 || 2 * workgroups(p, 64, 64) <= p.cus);
  if constexpr (E == Elem::kF32) {
    if (forced == 0 && (choice == 2 || choice == 3 || choice == 6 || (RBC < 8 && choice == 4))) {
      const int st = launch_small_blocks<E, RBC>(p, rows_m, cols_n, choice == 2, choice == 6, choice == 6 && splits_k,
                                                 choice == 4 && RBC != 2, stream, name);
      if (st >= 0) return st;
    }
  } else {
    // (Costs as fitted: up to 330 128x128 blocks; with 24 KB of K and more 64x64 blocks have
    // it in workgroups, too. Calls that direct_before_ksplit keeps in the kernels that stage
    // through LDS stay there, and rows under 16 bytes with less than 1 KB of K, 8-byte ones 512 bytes.)
    const int64_t k_bytes = (int64_t)p.K1 << p.lrb;
    const bool by_cost = !long_k && (RBC >= 16 || k_bytes >= (RBC == 8 ? 512 : 1024)) &&
                         ((choice == 2 && workgroups(p, 128, 128) <= 330) || choice == 3 ||
                          (choice == 6 && !direct_before_ksplit<E, RBC>(p)) || (RBC == 2 && choice == 4));
    if (forced == 0 && by_cost) {
      const int64_t b32 = uk::ceil_div(rows_m, (int64_t)32) * uk::ceil_div(cols_n, (int64_t)32);
      const bool parts = choice == 6 || (choice != 2 && b32 <= 2 * (int64_t)p.cus && k_bytes >= 1024) ||
                         (choice == 3 && RBC >= 16 && k_bytes >= 6144);
      const int st = launch_by_cost<E, RBC>(p, rows_m, cols_n, parts, stream, name);
      if (st >= 0) return st;
    } else if (forced == 0 && (choice == 3 || (choice == 6 && !splits_k) || (RBC < 8 && choice == 4))) {
      const int st = launch_small_blocks<E, RBC>(p, rows_m, cols_n, false, choice == 6, false,
                                                 choice == 4 && RBC != 2, stream, name);
      if (st >= 0) return st;
    }
  }
  if (forced == 0 && choice == 6 && direct_before_ksplit<E, RBC>(p)) choice = 3;
  if (choice == 6) {
    // Few 64x64 blocks and a long K: the barrier-free kernel with a 64x64
    // block per workgroup, whose four waves split K.
    if constexpr (RBC >= 8) {
      // K over workgroups too where the 64x64 blocks are fewer than half the
      // compute units and K is long: the meeting of the slices costs about 15
      // us with blocks of this size, so only from 24 KB of K per row on (f16
      // 128 x 128 x 65536, four blocks: 177 -> 52 us; 256 x 256 x 32768: 80 ->
      // 35; 512 x 512 x 16384: 44 -> 27; with 8 KB of K per row, 384 x 384 x
      // 4096, it loses: 16 -> 20 us).
      int st = launch_thin<E, RBC, 4, 4, 4, steps_ahead<E, RBC>(), true>(p, false, stream, long_k, 32);
      if (st >= 0) { *name = "mmt4d_mfma_64x64_ksplit"; return st; }
    }
    choice = 3;
  }
  // The thin kernel for a problem with `thin_rows` rows on its thin side and
  // `wide_cols` columns on the other (M-thin as it is, N-thin transposed).
  // (A generic lambda: its body is only instantiated for the row widths that call it.)
  auto thin_launch = [&](auto swapped_c, int64_t thin_rows, int64_t wide_cols) {
    const bool swapped = swapped_c;
    return launch_thin_any<E, RBC>(p, swapped, thin_rows, wide_cols, stream);
  };
  if (choice == 5) {
    // N-thin (a few columns against many rows, e.g. the last column strip of
    // a ragged problem): the thin kernel on the transposed problem.
    if constexpr (RBC >= 8) {
      int st = thin_launch(std::true_type{}, cols_n, rows_m);
      if (st >= 0) { *name = "mmt4d_mfma_thin_transposed"; return st; }
      // (K ends inside a step)
      if (forced == 0) st = launch_small_blocks<E, RBC>(p, rows_m, cols_n, false, false, false, false, stream, name);
      if (st >= 0) return st;
    }
    choice = 3;
  }
  if (choice == 4) {
    if constexpr (RBC >= 8) {
      int st = thin_launch(std::false_type{}, rows_m, cols_n);
      if (st >= 0) { *name = "mmt4d_mfma_thin"; return st; }
      if (forced == 0) st = launch_small_blocks<E, RBC>(p, rows_m, cols_n, false, false, false, true, stream, name);
      if (st >= 0) return st;
    }
    // With 2-byte rows a 16-byte piece spans 8 rows and 32 rows do not fill a
    // loader block; that combination takes the 64x64 variant.
    if constexpr (RBC != 2) {
      // 256 bytes of K per step: these problems are bound by memory latency,
      // and a longer step keeps more bytes in flight per workgroup, as do the
      // three steps of loads ahead of the MFMAs.
      int st = launch_variant<E, RBC, 2, 1, 1, 4, 4 / H, 4>(p, 0, p.K1, p.accumulate, stream);
      if (st >= 0) { *name = "mmt4d_mfma_32x64"; return st; }
    }
    choice = 3;
  }
  if (choice == 2) {
    // The LDS-direct ping-pong pipeline with 8 waves of 64x32 (measured against
    // the kernels below: s8 2048^3 16x16x2 20.6 -> 14.7 us, 16x16x16 14.8 ->
    // 14.5 us; 3072^3 40.5 -> 36.3 us; bf16 2048^3 23.4 -> 22.6 us).
    if (forced == 18 || (forced == 0 && E != Elem::kF32)) {
      int st = launch_variant<E, RBC, 4, 2, 2, 4, 1, 5>(p, 0, p.K1, p.accumulate, stream);
      if (st == 0) *name = "mmt4d_mfma_128x128_lds_direct";
      if (st >= 0) return st;
    }
    if constexpr (NARROW) {
      // (Not chosen by size: measured level with or behind the 128x128 kernel
      // that sends both operands through LDS.)
      if (kt_main > 0 && forced == 14) {
        int st = launch_narrow<E, RBC, 4, 2, 2>(p, kt_main, stream);
        if (st == 0) {
          *name = "mmt4d_mfma_128x128_narrow";
          if (kt_main == p.K1) return 0;
          return finish_k(launch_variant<E, RBC, 4, 4, 2, 2, NKK2, 0>(p, kt_main, p.K1 - kt_main, true, stream));
        }
        if (st > 0) return st;
      }
    }
    if constexpr (RBC >= 16) {
      int st = launch_variant<E, RBC, 4, 2, 2, 4, 1, 3>(p, 0, p.K1, p.accumulate, stream);
      if (st == 0) *name = "mmt4d_mfma_128x128_rhs_direct";
      if (st >= 0) return st;
    }
    int st = launch_variant<E, RBC, 4, 4, 2, 2, NKK2, 0>(p, 0, p.K1, p.accumulate, stream);
    if (st >= 0) { *name = "mmt4d_mfma_128x128"; return st; }
  }
  if constexpr (H == 1) {
    // 64x64 blocks, 8 waves of 32x16, 256 bytes of K per step.
    // Chosen for narrow tile rows when the 64x64 blocks fill the compute units
    // (s8 1024^3 16x16x2: 7.0 -> 6.4 us; with rows of 16 bytes and more the
    // register-direct kernel below is level or ahead: 5.7 against 5.9 us) and K
    // is a whole step at least. Its stages take the LDS of a compute unit, the deep
    // kernel below runs two and more workgroups on one and wins where there is no
    // pipeline to fill (s8 16x16x2 5000 x 200 x 124 5.0 against 8.7 us, 1400 x 1700
    // x 124 8.2 against 12.5), and with 16-bit outputs, which would need the
    // instance for a K that ends inside a step, at any such K (bf16 16x16x2 1400 x
    // 1700 x 508: 16.1 against 20.9 us).
    const int64_t k_bytes = (int64_t)p.K1 << p.lrb;
    const bool small_default = forced == 0 && RBC < 16 && E != Elem::kF32 && workgroups(p, 64, 64) >= 192 &&
                               k_bytes >= 256 && (!kOneLaunchOnly || k_bytes % 256 == 0);
    if (forced == 19 || small_default) {
      int st = launch_variant<E, RBC, 2, 1, 2, 4, 4, 5>(p, 0, p.K1, p.accumulate, stream);
      if (st == 0) *name = "mmt4d_mfma_64x64_lds_direct";
      if (st >= 0) return st;
    }
  }
  if constexpr (RBC >= 16) {
    int st = launch_variant<E, RBC, 2, 2, 2, 2, 1, 3>(p, 0, p.K1, p.accumulate, stream);
    if (st == 0) *name = "mmt4d_mfma_64x64_rhs_direct";
    if (st >= 0) return st;
  }
  if constexpr (NARROW) {
    if (kt_main > 0 && forced == 15) {
      int st = launch_narrow<E, RBC, 2, 2, 1>(p, kt_main, stream);
      if (st == 0) {
        *name = "mmt4d_mfma_64x64_narrow";
        if (kt_main == p.K1) return 0;
        return finish_k(launch_variant<E, RBC, 2, 2, 2, 2, NKK2, 0>(p, kt_main, p.K1 - kt_main, true, stream));
      }
      if (st > 0) return st;
    }
  }
  if constexpr (RBC < 16) {
    // Narrow tile rows, small problem: latency-bound (a 64x64 block computes a
    // 64-byte step in 64 MFMA cycles against a global round trip of well over a
    // thousand). 256-byte steps with the loads three steps ahead put the whole K
    // of such a problem in flight at once.
    if (forced == 11 || (forced == 0 && ((int64_t)p.K1 << p.lrb) <= 8192)) {
      int st = launch_variant<E, RBC, 2, 2, 2, 2, 4 / H, 4>(p, 0, p.K1, p.accumulate, stream);
      if (st >= 0) { *name = "mmt4d_mfma_64x64_deep"; return st; }
    }
  }
  int st = launch_variant<E, RBC, 2, 2, 2, 2, NKK2, 0>(p, 0, p.K1, p.accumulate, stream);
  if (st >= 0) { *name = "mmt4d_mfma_64x64"; return st; }
  st = launch_variant<E, RBC, 4, 4, 2, 2, NKK2, 0>(p, 0, p.K1, p.accumulate, stream);
  if (st >= 0) *name = "mmt4d_mfma_128x128";
  return st;
}

}  // namespace uk_mfma

#endif  // IREE_UK_AMD_MMT4D_MFMA_LAUNCH_H_
