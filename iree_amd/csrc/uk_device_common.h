// Shared device-side helpers for the gfx950 ukernel translation units.
#ifndef IREE_UK_AMD_DEVICE_COMMON_H_
#define IREE_UK_AMD_DEVICE_COMMON_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace uk {

// Unsigned 32-bit division by a runtime constant through a multiply-high:
// n / d == umulhi(n, mul) >> shift for every n < 2^31 (round-up method with a
// 32-bit multiplier; exact on that range for every d in [1, 2^31)).
struct FastDiv {
  uint32_t mul;
  uint32_t shift;
  uint32_t d;
  FastDiv() : mul(0), shift(0), d(1) {}
  explicit FastDiv(uint32_t divisor) : d(divisor) {
    if (divisor <= 1) {
      mul = 0;
      shift = 0;
      d = 1;
      return;
    }
    uint32_t l = 0;
    while ((1ull << l) < divisor) ++l;  // l = ceil(log2(d))
    // mul = floor(2^(32+l-1) / d) + 1 fits 32 bits and is exact for n < 2^31.
    uint64_t m = ((1ull << (32 + l - 1)) / divisor) + 1;
    mul = (uint32_t)m;
    shift = l - 1;
  }
  __host__ __device__ __forceinline__ uint32_t div(uint32_t n) const {
    if (d == 1) return n;
#if defined(__HIP_DEVICE_COMPILE__)
    return __umulhi(n, mul) >> shift;
#else
    return (uint32_t)(((uint64_t)n * mul) >> 32) >> shift;
#endif
  }
  __host__ __device__ __forceinline__ void divmod(uint32_t n, uint32_t& q,
                                                  uint32_t& r) const {
    q = div(n);
    r = n - q * d;
  }
};

// Has the kernel's arguments in scalar registers from here on. Left alone, the
// compiler loads each argument where it is first needed: a chain of scalar loads,
// each waited for (the first of every 64 bytes all the way to memory), before a
// short kernel's first global load.
template <typename T>
__device__ __forceinline__ void load_arguments_now(const T& v) {
  asm volatile("" : : "s"(v));
}
template <typename T, typename... Ts>
__device__ __forceinline__ void load_arguments_now(const T& v, const Ts&... vs) {
  load_arguments_now(v);
  load_arguments_now(vs...);
}

// A piece of N bytes (8 or 16) of a matrix row whose end may fall inside or
// before the piece. `clipped_offset` is where to load it from: the piece's own
// offset, or the last N bytes of the row where the piece reaches beyond them
// (the row must hold at least N bytes), so that every lane issues one
// unconditional load and the loads of a workgroup stay in flight together.
// `clip_piece` then moves the bytes of such a piece to where they belong and
// puts padding behind them; `left` = row bytes - piece offset, <= 0 for a piece
// that is all padding. (Element by element, the end of a row was a chain of up
// to sixteen dependent loads in every block of the last column: s8 100 x 97
// rows took 24 us to pack.)
template <int N>
__device__ __forceinline__ uint32_t clipped_offset(uint32_t off, uint32_t row_bytes) {
  return min(off, row_bytes - N);
}
template <int N>
__device__ __forceinline__ void clip_piece(uint32_t (&w)[N / 4], int32_t left, uint32_t pad32) {
  static_assert(N == 16 || N == 8 || N == 4, "whole words");
  if (left >= N) return;
  const uint64_t pad = ((uint64_t)pad32 << 32) | pad32;
  if (left <= 0) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) w[i] = pad32;
    return;
  }
  const uint32_t keep = 8 * (uint32_t)left, drop = 8 * N - keep;  // bits, both below 8 N
  if constexpr (N == 4) {
    const uint32_t mask = (1u << keep) - 1;
    w[0] = ((w[0] >> drop) & mask) | (pad32 & ~mask);
  } else if constexpr (N == 8) {
    const uint64_t x = ((uint64_t)w[1] << 32) | w[0];
    const uint64_t mask = (1ull << keep) - 1;
    const uint64_t y = ((x >> drop) & mask) | (pad & ~mask);
    w[0] = (uint32_t)y; w[1] = (uint32_t)(y >> 32);
  } else {
    uint64_t lo = ((uint64_t)w[1] << 32) | w[0], hi = ((uint64_t)w[3] << 32) | w[2];
    if (drop >= 64) {
      lo = hi >> (drop - 64);
      hi = 0;
    } else {
      lo = (lo >> drop) | (hi << (64 - drop));  // drop >= 8
      hi >>= drop;
    }
    const uint64_t mlo = keep >= 64 ? ~0ull : (1ull << keep) - 1;
    const uint64_t mhi = keep <= 64 ? 0ull : (1ull << (keep - 64)) - 1;
    lo = (lo & mlo) | (pad & ~mlo);
    hi = (hi & mhi) | (pad & ~mhi);
    w[0] = (uint32_t)lo; w[1] = (uint32_t)(lo >> 32); w[2] = (uint32_t)hi; w[3] = (uint32_t)(hi >> 32);
  }
}
// What a row of `row_bytes` (below 2^31) still holds from byte `off` on: 0 where
// it has ended. Tiles may pad a row by any amount, so the difference itself can
// be -2^31 and less and would come out positive.
__device__ __forceinline__ int32_t row_bytes_left(uint32_t row_bytes, uint32_t off) {
  return off < row_bytes ? (int32_t)(row_bytes - off) : 0;
}
// The same piece for a row of fewer than N bytes: the `left` bytes at `p` and
// padding behind them. At most N / 4 + 1 loads, none waiting for another (byte
// by byte, one after the other, they were a chain that took even a kernel of a
// single block from 4.0 to 8.1 us: s8 11277 x 14).
template <int N>
__device__ __forceinline__ void load_short_row(uint32_t (&w)[N / 4], const char* p, int32_t left, uint32_t pad32) {
  typedef uint32_t u32_a1 __attribute__((aligned(1)));
  typedef uint16_t u16_a1 __attribute__((aligned(1)));
#pragma unroll
  for (int i = 0; i < N / 4; ++i) w[i] = pad32;
  if (left <= 0) return;
  const uint32_t at = (uint32_t)left & ~3u;  // bytes in whole words
  uint32_t two = 0, one = 0;
  if (left & 2) two = *reinterpret_cast<const u16_a1*>(p + at);
  if (left & 1) one = (uint8_t)p[at + (left & 2)];
#pragma unroll
  for (int i = 0; i < N / 4 - 1; ++i)
    if (left >= 4 * i + 4) w[i] = *reinterpret_cast<const u32_a1*>(p + 4 * i);
  if (left & 3) {
    const uint32_t mask = (1u << 8 * (left & 3)) - 1;
    const uint32_t x = two | (one << 8 * (left & 2)) | (pad32 & ~mask);
#pragma unroll
    for (int i = 0; i < N / 4; ++i)
      if (at == 4u * i) w[i] = x;
  }
}
// Stores the first `n` bytes (0 < n < N) of a piece in at most four accesses.
template <int N>
__device__ __forceinline__ void store_head(char* p, const uint32_t (&w)[N / 4], uint32_t n) {
  typedef uint32_t u32_a1 __attribute__((aligned(1)));
  typedef uint16_t u16_a1 __attribute__((aligned(1)));
#pragma unroll
  for (int i = 0; i < N / 4; ++i)
    if (n >= 4u * i + 4) *reinterpret_cast<u32_a1*>(p + 4 * i) = w[i];
  const uint32_t at = n & ~3u;
  if (n & 3) {
    uint32_t x = w[0];  // word at / 4
    if constexpr (N == 8) x = (uint32_t)((((uint64_t)w[1] << 32) | w[0]) >> (8 * at));
    if constexpr (N == 16) {
      const uint64_t lo = ((uint64_t)w[1] << 32) | w[0], hi = ((uint64_t)w[3] << 32) | w[2];
      x = (uint32_t)((at & 8 ? hi : lo) >> (8 * (at & 4)));
    }
    if (n & 2) {
      *reinterpret_cast<u16_a1*>(p + at) = (uint16_t)x;
      x >>= 16;
    }
    if (n & 1) p[at + (n & 2)] = (char)x;
  }
}

// How a kernel stores what the next kernel reads.
enum class Store {
  kPlain,        // stays in the L2s, which are written back when the kernel ends
  kThrough,      // through the L2s into the memory-side cache as it is stored
  kNonTemporal,  // to HBM, past that cache too
};
// Stores `v`, 8 or 16 bytes, at `base` + `off`; `base` is the same in all lanes
// and `off` below 2^31.
template <Store S, typename V>
__device__ __forceinline__ void store_as(char* base, uint32_t off, V v) {
  if constexpr (S == Store::kThrough) {
    // (the cache policy operand's bit 4 is SC1: device scope, written through)
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, -1, 0x00027000);
    if constexpr (sizeof(V) == 16) __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, off, 0, 16);
    else __builtin_amdgcn_raw_buffer_store_b64(v, rsrc, off, 0, 16);
  } else if constexpr (S == Store::kNonTemporal) {
    __builtin_nontemporal_store(v, reinterpret_cast<V*>(base + off));
  } else {
    *reinterpret_cast<V*>(base + off) = v;
  }
}

// Largest power of two <= cap that divides v (v == 0 counts as divisible).
inline int64_t pow2_divisor(int64_t v, int64_t cap) {
  int64_t p = cap;
  if (v < 0) v = -v;
  while (p > 1 && (v % p) != 0) p >>= 1;
  return p;
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace uk

#endif  // IREE_UK_AMD_DEVICE_COMMON_H_
