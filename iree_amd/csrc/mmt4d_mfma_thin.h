// mmt4d on the gfx950 matrix cores for M-thin (decode-shaped) problems: a few
// rows of LHS against a long RHS. Such a call streams the RHS once and is
// bound by memory, so the kernel is built around keeping loads in flight:
//
//   * no LDS staging and no barrier in the K loop. A workgroup owns TM x TN
//     output blocks of 16x16; its KSPLIT waves take the K steps (64 bytes of K
//     per row, 128 for f8) round robin (wave w: steps w, w + KSPLIT, ...), so
//     together they read the workgroup's RHS panels front to back;
//   * each lane loads its MFMA operands straight from global memory, the RHS
//     from HBM and the (small, shared) LHS from L2, D steps ahead of the MFMAs
//     through D register buffers;
//   * the KSPLIT partial accumulators meet in LDS once, at the end; each wave adds
//     up, in wave order, and stores its share of the output blocks;
//     what that and the addresses cost bounds the small products and the decode layers
//     (one K step a wave, f16 512 x 2048 in 64x64 blocks: 6.7 us with the sums and the
//     stores in one wave and a vector division for each address, 4.6 so; with all of K =
//     2048 11.3 -> 10.0; s8 16 x 14336 x 4096 14.7 -> 13.7, f16 8 x 4096 x 4096 9.0 -> 8.4);
//   * when the problem has too few output blocks to occupy the chip (a decode
//     step against a weight matrix with few rows and a long K), K is split
//     over several workgroups per block as well: each publishes its partial
//     block in a workspace, and the one that arrives last (an atomic counter
//     per block) adds the slices in slice order and stores.
//
// Operand layout, K-order freedom of the MFMA and the output addressing are
// those of mmt4d_mfma_kernel.h, whose Args this kernel takes. With TM = TN = 4
// the same kernel serves problems of few 64x64 blocks and a long K, where the
// split of K over the waves matters more than operand reuse. The launcher may
// hand the operands over swapped (RHS as LHS) to serve N-thin problems: rows
// and columns then trade places in Args, four consecutive columns of the
// kernel are four rows of the caller's matrix (so `vec_out` is 0), and the
// scales of a dequantizing store are applied column scale first. Row widths of 16
// bytes and more load one 16-byte piece per operand; 8-byte rows load the two
// 8-byte halves from two K-tiles (chunk g of a step holds K-tiles g and
// g + 4), 4- and 2-byte rows likewise from four and eight. A K that
// ends inside a step (TAIL): the pieces beyond it are zero in both operands (what
// lies there may be an infinity).
//
// s8 x s4 -> s32 (Elem::kS8S4) runs here too. A lane loads 8 RHS bytes (16
// nibbles, the same 16 K elements as its 16 LHS bytes) and turns them into two
// groups of eight signed bytes without unpacking to true values: (x << 4) &
// 0xF0F0F0F0 holds 16 * (low nibble as s4) in every byte and x & 0xF0F0F0F0
// holds 16 * (high nibble as s4), i.e. the even and the odd K elements; the
// LHS bytes are split into even and odd positions to match (v_perm_b32). The
// MFMA then accumulates 16 times the true sum, exactly (the launcher bounds K
// so that this cannot wrap), and the store path shifts it back before it adds
// the ACCUMULATE input.
#ifndef IREE_UK_AMD_MMT4D_MFMA_THIN_H_
#define IREE_UK_AMD_MMT4D_MFMA_THIN_H_

#include "mmt4d_mfma_kernel.h"

namespace uk_mfma {

typedef int v2i __attribute__((ext_vector_type(2)));

// Loads from a buffer resource (its base, the same in all lanes), a lane's bytes and a
// scalar's: a lane's address is one register that the K loop never touches, where an
// address of its own takes a vector addition for every load, in the pipe that the f32
// matrix instructions keep busy (f32 16x16x1 in 32x32 blocks: 515 x 1027 x 769 17.0 ->
// 15.0 us, 700 x 700 x 3000 41.0 -> 34.6, 1500 x 1500 x 1000 52.6 -> 44.9). What lies
// kBeyond in a lane is outside the resource: such a load returns zeros and reads nothing.
// NT: non-temporal.
constexpr uint32_t kBeyond = 0x80000000u;
struct Operand {
  __amdgpu_buffer_rsrc_t buffer;
  const char* base;
};
__device__ __forceinline__ Operand operand_at(const char* base) {
  return {__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, (int)kBeyond, 0x00027000), base};
}
template <bool NT>
__device__ __forceinline__ v4i load16(const Operand& from, uint32_t lane_bytes, uint32_t bytes) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(from.buffer, lane_bytes, bytes, NT ? 2 : 0));
}
template <bool NT>
__device__ __forceinline__ v2i load8(const Operand& from, uint32_t lane_bytes, uint32_t bytes) {
  return __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(from.buffer, lane_bytes, bytes, NT ? 2 : 0));
}
template <bool NT>
__device__ __forceinline__ int load4(const Operand& from, uint32_t lane_bytes, uint32_t bytes) {
  return (int)__builtin_amdgcn_raw_buffer_load_b32(from.buffer, lane_bytes, bytes, NT ? 2 : 0);
}
template <bool NT>
__device__ __forceinline__ int load2(const Operand& from, uint32_t lane_bytes, uint32_t bytes) {
  return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(from.buffer, lane_bytes, bytes, NT ? 2 : 0);
}

// Sums of floats whose K eight waves share are in several chains, steps i, i + chains, ..
// of a wave apart: as many parts of K and more, each a shorter chain of roundings, as four
// waves in up to eight workgroups add up. Error against 64 bits of 32 x 512 results in one
// chain / here / in those workgroups, 1e-7: f16, K = 4096 1.56 / 1.03 / 1.03; f32, K = 2048
// 2.94 / 1.60 / 1.59. (The matrix instructions of 8-bit floats round to 1.5e-5 by
// themselves, however K is divided.)
template <Elem E, int TM, int KSPLIT>
constexpr int thin_chains() {
  using TT = ElemTraits<E>;
  return KSPLIT < 8 || TT::kHalves == 2 || std::is_same<typename TT::Acc, v4i>::value ? 1 : TM == 1 ? 4 : 2;
}

// Workgroup -> output block: bands of `a.band` block rows, or with `a.column_bands` of
// block columns, along the longer side, one after the other, each walked across; every
// XCD takes an equal share of that order. Its L2 then reads the shorter operand and its
// share of the longer one, whatever the numbers of blocks (in plain order both, where
// they are no multiple of 8).
__device__ __forceinline__ void block_in_bands(uint32_t wg, const Args& a, int* bm, int* bn) {
  const uint32_t total = (uint32_t)a.grid_m * (uint32_t)a.grid_n, xcd = wg & 7;
  const uint32_t id = xcd * (total >> 3) + min(xcd, total & 7) + (wg >> 3);
  const uint32_t along = (uint32_t)(a.column_bands ? a.grid_n : a.grid_m);
  const uint32_t across = (uint32_t)(a.column_bands ? a.grid_m : a.grid_n);
  const uint32_t b = a.by_band_blocks.quotient(id), in_band = id - b * (a.band * across);
  const bool whole = a.band <= along - b * a.band;
  const uint32_t width = whole ? a.band : along - b * a.band;
  const uint32_t step = (whole ? a.by_band : a.by_last_band).quotient(in_band);
  const uint32_t at = b * a.band + (in_band - step * width);
  *bm = (int)(a.column_bands ? step : at);
  *bn = (int)(a.column_bands ? at : step);
}

// STREAMED: the wide operand (the kernel's RHS: weights) is loaded
// non-temporally. For callers that say their weights come from HBM every time
// (iree_uk_amd_set_streamed_weights): a layer's weights then pass through the
// caches without displacing what is used again.
// CH: chains of a wave's sums (0: thin_chains).
// PAIRED: rows of 8 and 4 bytes in twos, those of the RHS and, with an even number of row
// blocks, of the LHS. A lane loads two neighbouring rows of a K-tile at once, half as many
// loads for the same bytes, and what it gets belongs to the same lane of two blocks: the one
// then holds the even and the other the odd rows or columns of 32. Rows are stored where
// they belong; columns are put back in order by the waves that add up and store. Each sum
// has the same products in the same order. N0 (M0) is even: others come here with rows of 16
// bytes. (These blocks are bound by how many loads a unit's L1 and the waves' loops take, the
// thin ones beside by HBM: launch_thin has the figures.)
template <Elem E, int RBC, int TM, int TN, int KSPLIT, int D, bool STREAMED = false, bool TAIL = false, int CH = 0,
          bool PAIRED = false>
__global__ __launch_bounds__(KSPLIT * 64, PAIRED && TM * TN >= 16 ? 2 : 1)   // (else two registers too many for two)
void mmt4d_thin_kernel(Args a) {
  using TT = ElemTraits<E>;
  using Acc = typename TT::Acc;
  using Out = typename TT::Out;
  constexpr int OB = Out::kOutBytes;
  constexpr int HALVES = TT::kHalves;
  constexpr int NCH = 4 * HALVES;             // 16-byte chunks per row per step
  constexpr int KS = NCH * 16;                // bytes of K per row per step
  constexpr bool S4 = E == Elem::kS8S4;       // 4-bit RHS: half the bytes per row
  constexpr int CHAINS = CH > 0 ? CH : thin_chains<E, TM, KSPLIT>();
  static_assert(RBC >= 2, "rows narrower than 2 bytes take the LDS kernels");
  // Rows of 2 and 4 bytes in 16x16 blocks, which are bound by how many loads a unit takes, load
  // from addresses: a unit takes more narrow loads of these than from a buffer resource, and
  // the vector addition that each costs is hidden here. us from resources / so, four steps
  // ahead: s8 16x16x2 100 x 128 x 20480 21.0 / 12.6 (14.4 with the addition in scalar
  // registers), 16x16x4 126 x 408 x 19584 11.9 / 9.9; bf16 16x16x2 100 x 128 x 10240 11.9 / 9.9;
  // f32 16x16x1 540 x 115 x 7400 30.1 / 25.8. (Rows of 8 bytes: level.)
  constexpr bool BY_ADDRESS = RBC <= 4 && TM * TN == 1;
  static_assert(!PAIRED || ((RBC == 8 || RBC == 4) && TN % 2 == 0 && HALVES == 1), "two rows a load, columns of two blocks");
  constexpr bool PAIRED_A = PAIRED && TM % 2 == 0;
  static_assert(!S4 || (RBC >= 16 && !TAIL), "4-bit RHS: LHS rows of at least 16 bytes, K in whole steps");

  // The blocks that a wave adds up and stores: OWN, or for the last ones fewer.
  static_assert(KSPLIT > 1, "several waves share K");
  constexpr int NB = TM * TN, OWN = (NB + KSPLIT - 1) / KSPLIT;
  __shared__ v4i partial[KSPLIT][NB][64];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t q = lane >> 4, r = lane & 15;
  // With K split over workgroups, consecutive workgroups share an output block.
  const uint32_t kslices = a.kslices > 1 ? a.kslices : 1;
  const uint32_t block_id = kslices > 1 ? blockIdx.x / kslices : blockIdx.x;
  const uint32_t slice = kslices > 1 ? blockIdx.x - block_id * kslices : 0;
  int bm, bn;
  if (kslices > 1) {
    bm = (int)a.by_grid_n.quotient(block_id);
    bn = (int)(block_id - (uint32_t)bm * a.grid_n);
  } else {
    block_in_bands(blockIdx.x, a, &bm, &bn);
  }
  // K steps of this workgroup: [step_begin, step_begin + wg_steps).
  uint32_t step_begin = 0;
  int wg_steps = a.steps;
  if (kslices > 1) {
    step_begin = (uint32_t)(((uint64_t)slice * (uint32_t)a.steps) / kslices);
    wg_steps = (int)((((uint64_t)(slice + 1) * (uint32_t)a.steps) / kslices) - step_begin);
  }
  const int lrb = a.lrb;
  const int lrb_b = S4 ? lrb - 1 : lrb;       // log2 of the RHS row bytes
  const uint32_t kt_m = (uint32_t)a.M0 << lrb, kt_n = (uint32_t)a.N0 << lrb_b;
  const uint32_t kts_per_step = KS >> lrb;
  const uint32_t sstep_a = kts_per_step * kt_m, sstep_b = kts_per_step * kt_n;

  // Byte offset of the lane's (first) piece of block row `x` (a row of 16 rows of
  // the M or N dimension) at K step 0, kBeyond for rows outside the problem or the
  // result (tile padding), which only reach accumulators that are never stored.
  // Offsets are relative to the first panel the workgroup touches.
  const int pa0 = (int)a.by_m0.quotient(bm * TM * 16), pb0 = (int)a.by_n0.quotient(bn * TN * 16);
  const Operand from_a = operand_at(a.lhs + (int64_t)pa0 * a.lhs_stride);
  const Operand from_b = operand_at(a.rhs + (int64_t)pb0 * a.rhs_stride);
  auto operand_offsets = [&](uint32_t (&off)[HALVES], uint32_t row, int X0, const Divisor& by_x0, int X1, int rows,
                             int p0, int64_t stride, uint32_t kt_bytes, int lrb, uint32_t piece_bytes) {
    const uint32_t pabs = by_x0.quotient(row);
    const uint32_t x0 = row - pabs * X0;
    const bool ok = (int)pabs < X1 && (int)row < rows;
    const uint32_t pl = pabs - (uint32_t)p0;
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const uint32_t g = (uint32_t)h * 4 + q;
      uint32_t o;
      if constexpr (RBC >= 16) {
        const uint32_t kb = g * piece_bytes;
        o = (kb >> lrb) * kt_bytes + (x0 << lrb) + (kb & ((1u << lrb) - 1));
      } else {
        o = g * kt_bytes + x0 * RBC;
      }
      off[h] = ok ? pl * (uint32_t)stride + o : kBeyond;
    }
  };
  uint32_t offa[TM][HALVES], offb[TN][HALVES];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
    operand_offsets(offa[tm], (uint32_t)(bm * TM + (PAIRED_A ? tm & ~1 : tm)) * 16 + (PAIRED_A ? 2 * r : r), a.M0, a.by_m0,
                    a.M1, a.out_rows, pa0, a.lhs_stride, kt_m, lrb, 16);
#pragma unroll
  for (int tn = 0; tn < TN; ++tn)
    operand_offsets(offb[tn], (uint32_t)(bn * TN + (PAIRED ? tn & ~1 : tn)) * 16 + (PAIRED ? 2 * r : r), a.N0, a.by_n0,
                    a.N1, a.out_cols, pb0, a.rhs_stride, kt_n, lrb_b, S4 ? 8 : 16);

  // Whether piece t of chunk (h, q) of K step s lies inside K.
  auto in_k = [&](uint32_t s, int h, int t) {
    if constexpr (RBC >= 16) {
      return s * KS + ((uint32_t)h * 4 + q) * 16 < (uint32_t)a.K1 << lrb;
    } else {
      return s * kts_per_step + (uint32_t)h * 4 + q + (uint32_t)t * NCH < (uint32_t)a.K1;
    }
  };
  // One lane operand of step s, `adv` bytes on from step 0. `ends`: K ends inside the
  // step, and what lies beyond it is zero.
  auto load_operand = [&](auto nontemporal, auto ends, const Operand& from, uint32_t off, uint32_t adv,
                          uint32_t kt_bytes, uint32_t s, int h) {
    auto at = [&](int t) { return !decltype(ends)::value || in_k(s, h, t) ? off : kBeyond; };
    constexpr bool NT = decltype(nontemporal)::value;
    const uint32_t piece = NCH * kt_bytes;   // from one piece to the next
    if constexpr (BY_ADDRESS && !decltype(ends)::value) {
      // (Rows outside the problem: the first one's bytes, whose sums are not stored either.)
      auto address = [&](int t) { return from.base + ((off == kBeyond ? 0u : off + t * piece) + adv); };
      if constexpr (RBC == 4) {
        typedef int int_g __attribute__((aligned(1)));
        auto load = [&](int t) { return *reinterpret_cast<const int_g*>(address(t)); };
        return v4i{load(0), load(1), load(2), load(3)};
      } else {
        typedef uint16_t u16_g __attribute__((aligned(1)));
        v8i v;
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = *reinterpret_cast<const u16_g*>(address(t));
        return v;
      }
    } else if constexpr (RBC >= 16) {
      return load16<NT>(from, at(0), adv);
    } else if constexpr (RBC == 8) {
      const v2i lo = load8<NT>(from, at(0), adv), hi = load8<NT>(from, at(1), adv + piece);
      return v4i{lo[0], lo[1], hi[0], hi[1]};
    } else if constexpr (RBC == 4) {
      return v4i{load4<NT>(from, at(0), adv), load4<NT>(from, at(1), adv + piece),
                 load4<NT>(from, at(2), adv + 2 * piece), load4<NT>(from, at(3), adv + 3 * piece)};
    } else {
      v8i v;
#pragma unroll
      for (int t = 0; t < 8; ++t) v[t] = load2<NT>(from, at(t), adv + t * piece);
      return v;
    }
  };
  // PAIRED: half of the pieces of two blocks' lane operands, the first half for the even one.
  auto load_pair = [&](auto nontemporal, auto ends, const Operand& from, uint32_t off, uint32_t adv,
                       uint32_t kt_bytes, uint32_t s, int h, int odd) {
    constexpr int HALF = RBC == 8 ? 1 : 2;
    auto at = [&](int t) { return !decltype(ends)::value || in_k(s, h, t) ? off : kBeyond; };
    constexpr bool NT = decltype(nontemporal)::value;
    const uint32_t piece = NCH * kt_bytes, first = adv + odd * HALF * piece;
    const int t0 = odd * HALF;
    if constexpr (RBC == 8) {
      return load16<NT>(from, at(t0), first);
    } else {
      const v2i lo = load8<NT>(from, at(t0), first), hi = load8<NT>(from, at(t0 + 1), first + piece);
      return v4i{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  // The lane operands of the two blocks from what was loaded so.
  auto unpair = [&](const v4i& lo, const v4i& hi, v4i& even, v4i& odd) {
    if constexpr (RBC == 8) {
      even = v4i{lo[0], lo[1], hi[0], hi[1]};
      odd = v4i{lo[2], lo[3], hi[2], hi[3]};
    } else {
      even = v4i{lo[0], lo[2], hi[0], hi[2]};
      odd = v4i{lo[1], lo[3], hi[1], hi[3]};
    }
  };
  // Rows of 2 bytes: a register for each piece until the step is computed (put together
  // as they come, they would be waited for as they are asked for).
  using AFrag = typename std::conditional<RBC == 2, v8i, v4i>::type;
  using BFrag = typename std::conditional<S4, v2i, AFrag>::type;
  AFrag fa[D][TM][HALVES];
  BFrag fb[D][TN][HALVES];
  // ---- K steps -----------------------------------------------------------------
  // Local step i of this wave is K step step_begin + wave + i * KSPLIT; the wave that
  // has the step K ends inside (TAIL) takes that one first and the others after it, so
  // that no load of the K loop asks whether it is that step (a branch beside every load
  // kept products and loads apart: f32 184 x 88 x 4811 14.3 us, so 10.9).
  const int my_steps = wg_steps > wave ? (wg_steps - wave + KSPLIT - 1) / KSPLIT : 0;
  const uint32_t last_step = (uint32_t)a.steps - 1;
  const bool tail_first =
      TAIL && my_steps > 0 && step_begin + (uint32_t)(wave + (my_steps - 1) * KSPLIT) == last_step;
  const uint32_t first_step = step_begin + (uint32_t)wave - (tail_first ? KSPLIT : 0);   // (of i = 0: may wrap)
  // `at_a`, `at_b`: how far the step's K-tiles are from those of step 0, in bytes.
  auto load_at = [&](int d, uint32_t at_a, uint32_t at_b, uint32_t s, auto ends) {
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        if constexpr (S4) {
          fb[d][tn][h] = load8<STREAMED>(from_b, offb[tn][h], at_b);
        } else if constexpr (PAIRED) {
          fb[d][tn][h] = load_pair(std::bool_constant<STREAMED>{}, ends, from_b, offb[tn][h], at_b, kt_n, s, h, tn % 2);
        } else {
          fb[d][tn][h] = load_operand(std::bool_constant<STREAMED>{}, ends, from_b, offb[tn][h], at_b, kt_n, s, h);
        }
      }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        if constexpr (PAIRED_A)
          fa[d][tm][h] = load_pair(std::false_type{}, ends, from_a, offa[tm][h], at_a, kt_m, s, h, tm % 2);
        else
          fa[d][tm][h] = load_operand(std::false_type{}, ends, from_a, offa[tm][h], at_a, kt_m, s, h);
      }
  };
  // Local step i. (Its number is kept from the compiler, which would hold the offsets of all
  // steps of an unrolled round in scalar registers of their own, and spill them, or in
  // vector registers, and loop over the lanes at every load.)
  auto load_step = [&](int d, int i) {
    uint32_t s = __builtin_amdgcn_readfirstlane(first_step + (uint32_t)(i * KSPLIT));
    if constexpr (!BY_ADDRESS) asm volatile("" : "+s"(s));
    load_at(d, s * sstep_a, s * sstep_b, s, std::false_type{});
  };

  // ---- output addressing (see for_each_output in mmt4d_mfma_kernel.h) ------
  // Lane (q, r) of block b = tm * TN + tn holds output row r, columns 4q..4q+3 (PAIRED_A: row
  // 2r or 2r + 1 of two blocks' 32).
  // f4(i, p) / f1(i, e, p) for the i-th of this wave's blocks.
  // PAIRED: of two neighbouring own blocks the first holds columns 8q..8q+3 of their 32,
  // the second 8q+4..8q+7.
  const int first_own = wave * OWN;
  auto row_of = [&](int tm) {
    return PAIRED_A ? (bm * TM + (tm & ~1)) * 16 + 2 * (int)r + (tm & 1) : (bm * TM + tm) * 16 + (int)r;
  };
  auto first_col = [&](int tn) {
    return PAIRED ? (bn * TN + (tn & ~1)) * 16 + 8 * (int)q + 4 * (tn & 1) : (bn * TN + tn) * 16 + 4 * (int)q;
  };
  auto for_each_own = [&](auto f) {
#pragma unroll
    for (int i = 0; i < OWN; ++i)
      if ((NB % OWN == 0 && first_own < NB) || first_own + i < NB) f(i, (first_own + i) / TN, (first_own + i) % TN);
  };
  auto for_each_output = [&](const char* base, int64_t s_panel, uint32_t s_m0, uint32_t s_pn,
                             uint32_t s_n0, auto f4, auto f1) {
    for_each_own([&](int i, int tm, int tn) {
      const int row = row_of(tm);
      const int pl = (int)a.by_m0.quotient(row), m0 = row - pl * a.M0;
      const bool row_ok = pl < a.M1 && row < a.out_rows;
      char* row_base = const_cast<char*>(base) + (int64_t)pl * s_panel + (int64_t)m0 * s_m0;
      const int col = first_col(tn);
      if (a.vec_out) {
        const int pc = (int)a.by_n0.quotient(col), n0 = col - pc * a.N0;
        const int left = a.out_cols - col;
        char* p = row_base + (int64_t)pc * s_pn + (int64_t)n0 * s_n0;
        if (row_ok && pc < a.N1 && left >= 4) {
          f4(i, p);
        } else if (row_ok && pc < a.N1) {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (e < left) f1(i, e, p + e * s_n0);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = col + e;
          const int pc = (int)a.by_n0.quotient(c), n0 = c - pc * a.N0;
          if (row_ok && pc < a.N1 && c < a.out_cols)
            f1(i, e, row_base + (int64_t)pc * s_pn + (int64_t)n0 * s_n0);
        }
      }
    });
  };

  Acc chains[CHAINS][TM][TN];
  Acc (&acc)[TM][TN] = chains[0];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) chains[c][tm][tn] = Acc{0, 0, 0, 0};

  // ---- K loop ---------------------------------------------------------------
  if (tail_first) load_at(0, last_step * sstep_a, last_step * sstep_b, last_step, std::true_type{});
  else if (my_steps > 0) load_step(0, 0);
#pragma unroll
  for (int d = 1; d < D; ++d)
    if (d < my_steps) load_step(d, d);
  // The waves that store fetch what the store needs now, under the K loop: the
  // initial accumulators, which the sums are added to at the end (with K split over
  // workgroups only to the first slice's), and the scales of the dequantizing store
  // (indices beyond the matrix are clamped; their elements are never stored).
  Acc cin[OWN];
  float sm[OWN];
  v4f sn[OWN];
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    cin[i] = Acc{0, 0, 0, 0};
    sm[i] = 1.0f;
    sn[i] = v4f{1.0f, 1.0f, 1.0f, 1.0f};
  }
  if (a.accumulate && slice == 0) {
    for_each_output(a.acc, a.acc_stride, a.acc_sm0, a.acc_spn, a.acc_sn0,
                    [&](int i, char* p) { cin[i] = Out::load4(p); },
                    [&](int i, int e, char* p) { cin[i][e] = Out::load1(p); });
  }
  if (OB == 4 && a.dequant) {
    if (a.row_scale) {
      for_each_own([&](int i, int tm, int) {
        sm[i] = a.row_scale[max(min(row_of(tm), a.out_rows - 1), 0)];
      });
    }
    if (a.col_scale) {
      for_each_own([&](int i, int, int tn) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          sn[i][e] = a.col_scale[max(min(first_col(tn) + e, a.out_cols - 1), 0)];
      });
    }
  }
  // The products of a step, whose operands are in registers d, onto chain c.
  auto compute = [&](int d, int c) {
    if constexpr (S4) {
      // LHS: even K bytes, then odd K bytes; RHS: low nibbles, then high ones.
      v4i ea[TM], eb[TN];
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        const v4i x = fa[d][tm][0];
        ea[tm] = v4i{(int)__builtin_amdgcn_perm((uint32_t)x[1], (uint32_t)x[0], 0x06040200u),
                     (int)__builtin_amdgcn_perm((uint32_t)x[3], (uint32_t)x[2], 0x06040200u),
                     (int)__builtin_amdgcn_perm((uint32_t)x[1], (uint32_t)x[0], 0x07050301u),
                     (int)__builtin_amdgcn_perm((uint32_t)x[3], (uint32_t)x[2], 0x07050301u)};
      }
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        const uint32_t x0 = (uint32_t)fb[d][tn][0][0], x1 = (uint32_t)fb[d][tn][0][1];
        eb[tn] = v4i{(int)((x0 << 4) & 0xF0F0F0F0u), (int)((x1 << 4) & 0xF0F0F0F0u),
                     (int)(x0 & 0xF0F0F0F0u), (int)(x1 & 0xF0F0F0F0u)};
      }
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = TT::mfma(&eb[tn], &ea[tm], acc[tm][tn]);
    } else if constexpr (RBC == 2 || PAIRED || E == Elem::kF32) {
      auto whole = [](const auto& v) {
        if constexpr (sizeof(v) == sizeof(v8i)) {
          return v4i{(int)__builtin_amdgcn_perm((uint32_t)v[1], (uint32_t)v[0], 0x05040100u),
                     (int)__builtin_amdgcn_perm((uint32_t)v[3], (uint32_t)v[2], 0x05040100u),
                     (int)__builtin_amdgcn_perm((uint32_t)v[5], (uint32_t)v[4], 0x05040100u),
                     (int)__builtin_amdgcn_perm((uint32_t)v[7], (uint32_t)v[6], 0x05040100u)};
        } else {
          return v;
        }
      };
      v4i ea[TM], eb[TN];
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        if constexpr (!PAIRED_A) ea[tm] = whole(fa[d][tm][0]);
        else if (tm % 2 == 0) unpair(fa[d][tm][0], fa[d][tm + 1][0], ea[tm], ea[tm + 1]);
      }
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        if constexpr (!PAIRED) eb[tn] = whole(fb[d][tn][0]);
        else if (tn % 2 == 0) unpair(fb[d][tn][0], fb[d][tn + 1][0], eb[tn], eb[tn + 1]);
      }
      if constexpr (E == Elem::kF32) {
        // A word of all blocks before the next one: products of one block wait for each other.
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
          for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
              chains[c][tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(v4f, eb[tn])[w],
                                                                       __builtin_bit_cast(v4f, ea[tm])[w],
                                                                       chains[c][tm][tn], 0, 0, 0);
      } else {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) chains[c][tm][tn] = TT::mfma(&eb[tn], &ea[tm], chains[c][tm][tn]);
      }
    } else {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          chains[c][tm][tn] = TT::mfma(fb[d][tn], fa[d][tm], chains[c][tm][tn]);
    }
  };
  constexpr int U = D > CHAINS ? D : CHAINS;   // steps unrolled: whole rounds of both
  static_assert(U % D == 0 && U % CHAINS == 0, "");
  int i = 0;
  // Steady state: every step computed is followed by the load of the step D
  // further on, which exists. (All loads so far have come when it begins: they were issued
  // under conditions, and the compiler, which cannot tell how many are behind the first,
  // would wait for every load in flight at the head of each round.)
  if (i + U + D <= my_steps) {
    wait_vmem_in_flight<0>();
    do {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        compute(u % D, u % CHAINS);
        load_step(u % D, i + u + D);
        // (Left alone the compiler brings the products of several steps together and their
        // loads behind them, so that none is a step ahead: f32 170 x 184 x 5000 15.5 us.)
        __builtin_amdgcn_sched_barrier(0);
      }
      i += U;
    } while (i + U + D <= my_steps);
  }
  // The products of the last steps: a chain's sum is read, to be added up or copied, soon
  // after them, and the compiler counts the instructions that have to lie in between
  // along the longer of two paths through `if (compute) { if (load) }` (too few on the
  // shorter one: sums without their last product). So they lie behind the product itself.
  auto compute_last = [&](int d, int c) {
    compute(d, c);
    if constexpr (CHAINS > 1) settle_products();
  };
  // Fewer than U + D steps left: the same with bounds.
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (i + u < my_steps) {
      compute_last(u % D, u % CHAINS);
      if (i + u + D < my_steps) load_step(u % D, i + u + D);
    }
  }
#pragma unroll
  for (int u = U; u < U + D; ++u)
    if (i + u < my_steps) compute_last(u % D, u % CHAINS);
  settle_products();
#pragma unroll
  for (int c = 1; c < CHAINS; ++c)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) acc[tm][tn] += chains[c][tm][tn];

  // ---- meet the partial sums ---------------------------------------------------
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) partial[wave][tm * TN + tn][lane] = __builtin_bit_cast(v4i, acc[tm][tn]);
  __syncthreads();
  if (kslices <= 1 && first_own >= NB) return;
  Acc sum[OWN];
  for_each_own([&](int i, int tm, int tn) {
    const int b = tm * TN + tn;
    auto part = [&](int w) {
      if constexpr (PAIRED) {
        const v2i even = reinterpret_cast<const v2i*>(&partial[w][b & ~1][lane])[b & 1];
        const v2i odd = reinterpret_cast<const v2i*>(&partial[w][b | 1][lane])[b & 1];
        return __builtin_bit_cast(Acc, v4i{even[0], odd[0], even[1], odd[1]});
      } else {
        return __builtin_bit_cast(Acc, partial[w][b][lane]);
      }
    };
    sum[i] = part(0);
#pragma unroll
    for (int w = 1; w < KSPLIT; ++w) sum[i] += part(w);
    // (4-bit RHS: every slice holds 16 times its part of the sum, so the shift is
    // exact per slice.)
    if constexpr (S4) sum[i] = sum[i] >> 4;
    sum[i] += cin[i];
  });

  // ---- meet the K slices of the other workgroups -----------------------------------
  // The workgroup publishes its partial blocks, then counts itself in; the
  // workgroup that arrives last adds the slices up in slice order (so a float
  // result does not depend on who arrived when) and goes on to store. The slices
  // run on different XCDs, each with an L2 of its own, so partials and counter are
  // moved with device-scope atomic accesses (relaxed 32-bit stores and loads: they
  // go through to the point where the XCDs meet and leave the caches alone). A
  // device-scope FENCE would be correct too and is far too expensive here: it
  // writes back and invalidates the whole L2, under the feet of every workgroup
  // that streams weights through it. What the counter increment has to wait for is
  // only that the workgroup's own partial stores are complete: every wave waits for
  // its own before the barrier.
  if (kslices > 1) {
    __shared__ uint32_t arrived_lds;
    uint32_t* mine = reinterpret_cast<uint32_t*>(a.ws_partials) +
                     (((size_t)block_id * kslices + slice) * (NB * 64) + lane) * 4;
    for_each_own([&](int i, int tm, int tn) {
      const v4i v = __builtin_bit_cast(v4i, sum[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        __hip_atomic_store(mine + (tm * TN + tn) * 256 + e, (uint32_t)v[e], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    });
    // All of the wave's stores above have been acknowledged before the barrier.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
      arrived_lds = __hip_atomic_fetch_add(a.ws_counters + block_id, 1u, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (arrived_lds != kslices - 1) return;
    // The reader side of the handoff. What the other slices stored is complete
    // at the point where the XCDs meet before their counter increments (their
    // agent-scope stores are acknowledged from there, and each waited for its
    // own before counting), and the agent-scope loads below go to that point
    // instead of a cache; this fence only keeps the compiler from moving those
    // loads above the test of the counter (workgroup scope: it costs no cache
    // write-back or invalidation).
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (threadIdx.x == 0) {
      __hip_atomic_store(a.ws_counters + block_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint32_t* all = reinterpret_cast<const uint32_t*>(a.ws_partials) +
                          ((size_t)block_id * kslices * (NB * 64) + lane) * 4;
#pragma unroll
    for (int i = 0; i < OWN; ++i) sum[i] = Acc{0, 0, 0, 0};
    for (uint32_t sl = 0; sl < kslices; ++sl) {
      for_each_own([&](int i, int tm, int tn) {
        v4i v;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = (int)__hip_atomic_load(all + ((size_t)sl * NB + tm * TN + tn) * 256 + e,
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sum[i] += __builtin_bit_cast(Acc, v);
      });
    }
  }

  // ---- store --------------------------------------------------------------------
  if constexpr (OB == 4) {
    if (a.dequant) {
      typedef v4f v4f_a4 __attribute__((aligned(4)));
      for_each_output(
          a.out, a.out_stride, a.out_sm0, a.out_spn, a.out_sn0,
          [&](int i, char* p) {
            v4f v = __builtin_convertvector(sum[i], v4f);
            if (a.col_scale_first) {
              v = v * sn[i];
              v = v * sm[i];
            } else {
              v = v * sm[i];
              v = v * sn[i];
            }
            *reinterpret_cast<v4f_a4*>(p) = v;
          },
          [&](int i, int e, char* p) {
            const float v = (float)sum[i][e];
            *reinterpret_cast<float*>(p) = a.col_scale_first ? v * sn[i][e] * sm[i] : v * sm[i] * sn[i][e];
          });
      return;
    }
  }
  for_each_output(a.out, a.out_stride, a.out_sm0, a.out_spn, a.out_sn0,
                  [&](int i, char* p) { Out::store4(p, sum[i]); },
                  [&](int i, int e, char* p) { Out::store1(p, sum[i][e]); });
}

}  // namespace uk_mfma

#endif  // IREE_UK_AMD_MMT4D_MFMA_THIN_H_
