// Software conversions between f32 and the 16-bit float formats, with the
// exact behaviour of the CPU ukernels' routines
// (runtime/src/iree/builtins/ukernel/common.h:651-792). Device code.
#ifndef IREE_UK_AMD_UK_FLOAT_CONVERT_H_
#define IREE_UK_AMD_UK_FLOAT_CONVERT_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace uk {

// Both are selections between values that every lane computes: with a branch for
// each case a wave took them one after the other, 128 times in the epilogue of a
// wave's 32 output blocks (bf16 4859 x 3738 x 24 into bf16: 50.5 us, 38.5 now).

// 16-bit float with EB exponent bits -> f32: exponent field 0 (zero and
// subnormals) gives a signed zero, NaN gives a quiet NaN with all mantissa
// bits set (runtime/src/iree/builtins/ukernel/common.h:665-699).
template <int EB>
__device__ __forceinline__ float small16_to_f32(uint16_t v) {
  constexpr int MB = 15 - EB;
  const uint32_t sign = (uint32_t)(v >> 15) << 31;
  const uint32_t e = (v >> MB) & ((1u << EB) - 1);
  const uint32_t m = v & ((1u << MB) - 1);
  uint32_t bits = ((e + 128u - (1u << (EB - 1))) << 23) | (m << (23 - MB));
  bits = e == 0 ? 0u : bits;
  bits = e == (1u << EB) - 1 ? (m ? 0x7FFFFFFFu : 0x7F800000u) : bits;
  return __uint_as_float(sign | bits);
}

// f32 -> 16-bit float, round to nearest even, with the exponent-range
// behaviour of runtime/src/iree/builtins/ukernel/common.h:701-770 (the range
// tests sit one binade late; f32 subnormals give zero).
template <int EB>
__device__ __forceinline__ uint16_t f32_to_small16(float value) {
  constexpr int MB = 15 - EB;
  const uint32_t u = __float_as_uint(value);
  const uint32_t sign16 = (u >> 31) << 15;
  const uint32_t e32 = (u >> 23) & 0xFF;
  const uint32_t m32 = u & 0x007FFFFFu;
  constexpr uint32_t emask16 = ((1u << EB) - 1) << MB;
  constexpr uint32_t mmask16 = (1u << MB) - 1;
  constexpr int drop = 23 - MB, half_range = 1 << (EB - 1);
  const int ex = (int)e32 - 128;
  // Half of what is dropped, less one where the last bit kept is even. A mantissa
  // that is rounded up to the next power of two carries into the exponent.
  const uint32_t rounded = m32 + (1u << (drop - 1)) - 1 + ((m32 >> drop) & 1);
  uint32_t bits = ((uint32_t)(ex + half_range) << MB) + (rounded >> drop);
  bits = ex >= half_range ? emask16 : bits;
  bits = e32 == 0 || ex < -half_range ? 0u : bits;
  bits = e32 == 0xFF ? (m32 ? emask16 | mmask16 : emask16) : bits;
  return (uint16_t)(sign16 | bits);
}

}  // namespace uk

#endif  // IREE_UK_AMD_UK_FLOAT_CONVERT_H_
