// Device-side helpers shared by the kernel translation units.
#ifndef IREE_AMD_CSRC_UK_DEVICE_H_
#define IREE_AMD_CSRC_UK_DEVICE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace uk {

// 16-bit float -> f32 with the reference's generic-path semantics
// (common.h:665-699): a zero exponent field (zeros AND subnormals) widens to a
// signed zero, NaNs become the all-ones-mantissa quiet NaN. EBITS is 5 for
// f16, 8 for bf16.
// (Without branches, and for a value in the upper half of a word, as two of them come out of memory: 6 and 9 instructions.)
template <int EBITS>
__host__ __device__ __forceinline__ float widen16_upper(uint32_t upper) {
  const uint32_t sign = upper & 0x80000000u;
  uint32_t mag = (upper & 0x7FFF0000u) >> (8 - EBITS), r = mag;  // exponent and mantissa where f32 has them
  if constexpr (EBITS < 8) r += (127u - ((1u << (EBITS - 1)) - 1u)) << 23;
  constexpr uint32_t INFINITE = ((1u << EBITS) - 1u) << 23;
  if constexpr (EBITS < 8) r = mag >= INFINITE ? 0x7F800000u : r;
  r = mag > INFINITE ? 0x7FFFFFFFu : r;
  r = mag < 0x00800000u ? 0u : r;
  return __builtin_bit_cast(float, sign | r);
}
template <int EBITS>
__host__ __device__ __forceinline__ float widen16(uint16_t h) { return widen16_upper<EBITS>((uint32_t)h << 16); }
// The two values of a word.
template <int EBITS>
__host__ __device__ __forceinline__ float widen16_first(uint32_t w) { return widen16_upper<EBITS>(w << 16); }
template <int EBITS>
__host__ __device__ __forceinline__ float widen16_second(uint32_t w) { return widen16_upper<EBITS>(w & 0xFFFF0000u); }

// f32 -> 16-bit float, round to nearest even, with the reference's quirks
// (common.h:701-770): f32 subnormals and results below the exponent range give
// zero, overflow gives infinity, and the lowest in-range exponent is encoded
// with exponent field 0 plus the rounded mantissa bits. This is the
// conversion spelled out step by step; narrow16 below is what the kernels call.
template <int EBITS>
__host__ __device__ __forceinline__ uint16_t narrow16_by_steps(float f) {
  constexpr int MBITS = 15 - EBITS;
  constexpr int HALF = 1 << (EBITS - 1);
  constexpr uint32_t EMASK = ((1u << EBITS) - 1u) << MBITS;
  constexpr uint32_t MMASK = (1u << MBITS) - 1u;
  const uint32_t bits = __builtin_bit_cast(uint32_t, f);
  const uint32_t sign = (bits >> 31) << 15;
  const uint32_t e32 = (bits >> 23) & 0xFFu;
  const uint32_t m32 = bits & 0x007FFFFFu;
  if (e32 == 0xFFu) return (uint16_t)(sign | EMASK | (m32 ? MMASK : 0u));
  if (e32 == 0) return (uint16_t)sign;
  int e = (int)e32 - 128;
  if (e >= HALF) return (uint16_t)(sign | EMASK);
  if (e < -HALF) return (uint16_t)sign;
  constexpr uint32_t EVEN = 1u << (23 - MBITS);
  constexpr uint32_t ODD = EVEN >> 1;
  uint32_t m = m32 + ((m32 & EVEN) ? ODD : ODD - 1u);
  if (m > 0x007FFFFFu) {
    m = 0;
    ++e;
  }
  return (uint16_t)(sign | ((uint32_t)(e + HALF) << MBITS) | (m >> (23 - MBITS)));
}

// The same function without branches (an epilogue that rounds 256 accumulators
// per lane with the steps above took 23 us of a 154 us f16f16f16 4096^3
// launch). For every f32 exponent field that the steps treat as in range
// (1 .. 254 for bf16, which has f32's exponent range; 112 .. 143 for f16) they
// amount to adding the rounding bias to the whole word, letting the mantissa
// carry into the exponent (common.h:741-752 says as much), and rebasing the
// exponent; that includes the reference's encodings at both ends of the f16
// range (field 0 with mantissa bits for 2^-15 <= |x| < 2^-14, field 31 with
// mantissa bits for 2^16 <= |x| < 2^17, and the carry out of that into bit
// 15). Below the range: signed zero; above: infinity; NaN: all mantissa bits.
// (The hardware's v_cvt_f16_f32 agrees with the steps between the smallest
// normal f16 and overflow only; a test of the range in front of it, as a
// branch per value, per four values or per wavefront, was slower than this.)
template <int EBITS>
__host__ __device__ __forceinline__ uint16_t narrow16(float f) {
  constexpr int MBITS = 15 - EBITS;
  constexpr int SHIFT = 23 - MBITS;                              // mantissa bits dropped
  constexpr uint32_t LOWEST = 128u - (1u << (EBITS - 1));        // lowest in-range f32 exponent field (0 for bf16)
  constexpr uint32_t EMASK = ((1u << EBITS) - 1u) << MBITS, MMASK = (1u << MBITS) - 1u;
  const uint32_t bits = __builtin_bit_cast(uint32_t, f);
  const uint32_t mag = bits & 0x7FFFFFFFu, sign = (bits >> 16) & 0x8000u;
  uint32_t r = ((mag + ((1u << (SHIFT - 1)) - 1u) + ((mag >> SHIFT) & 1u)) >> SHIFT) - (LOWEST << MBITS);
  if constexpr (EBITS == 8) {
    r = mag < 0x00800000u ? 0u : r;                              // zeros and f32 subnormals
  } else {
    r = mag < (LOWEST << 23) ? 0u : r;                           // below the range (zeros, f32 subnormals included)
    r = mag >= ((LOWEST + (2u << (EBITS - 1))) << 23) ? EMASK : r;   // above it, infinity included
  }
  r = mag == 0x7F800000u ? EMASK : r;
  r = mag > 0x7F800000u ? (EMASK | MMASK) : r;
  return (uint16_t)(sign | r);
}

// Two of them in a word. bf16: the conversion instruction rounds two values at a time; what it does not do as above, f32
// subnormals to zero and NaNs with all mantissa bits, is done to the values ahead of it: 6.5 instructions a value and not 14.
template <int EBITS>
__device__ __forceinline__ uint32_t narrow16_pair(float a, float b) {
  if constexpr (EBITS == 8) {
    typedef float v2f32 __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf16 __attribute__((ext_vector_type(2)));
    auto prepared = [](float f) {
      const uint32_t bits = __builtin_bit_cast(uint32_t, f);
      uint32_t r = __builtin_amdgcn_classf(f, 0x90) ? bits & 0x80000000u : bits;  // (subnormals of either sign)
      r = f != f ? bits | 0x7FFFFFFFu : r;
      return __builtin_bit_cast(float, r);
    };
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f32{prepared(a), prepared(b)}, v2bf16));
  } else {
    return (uint32_t)narrow16<EBITS>(a) | ((uint32_t)narrow16<EBITS>(b) << 16);
  }
}

// n / d, exactly, by multiplication with a reciprocal that the host has computed. (The compiler's division of 32 bits is 25
// dependent instructions, 100 to 150 cycles, and a workgroup divides before it can load.)
__host__ __device__ __forceinline__ uint32_t reciprocal_of(uint32_t d) { return 0xFFFFFFFFu / d; }
__host__ __device__ __forceinline__ uint32_t divide(uint32_t n, uint32_t d, uint32_t reciprocal) {
  const uint32_t q = (uint32_t)((uint64_t)n * reciprocal >> 32);  // one too few at most
  return q + (n - q * d >= d ? 1 : 0);
}

// Tile number `linear` of a grid of tile_rows x tile_cols tiles that are walked in bands of kBandRows rows, a band column by
// column. tile_cols below 2^29.
constexpr uint32_t kBandRows = 4;
__host__ __device__ __forceinline__ uint32_t band_reciprocal(uint32_t tile_cols) { return reciprocal_of(kBandRows * tile_cols); }
__host__ __device__ __forceinline__ void tile_of_number(uint32_t linear, uint32_t tile_rows, uint32_t tile_cols,
                                                        uint32_t reciprocal, int* tile_row, int* tile_col) {
  const uint32_t band_tiles = kBandRows * tile_cols;
  const uint32_t band = divide(linear, band_tiles, reciprocal);
  const uint32_t band_first = band * kBandRows, rows_left = tile_rows - band_first;
  const uint32_t band_rows = rows_left < kBandRows ? rows_left : kBandRows;
  const uint32_t in_band = linear - band * band_tiles;
  // ceil(2^31 / band_rows), of 1 to 4: exact for numbers below 2^31
  const uint32_t rows_reciprocal = band_rows == 3 ? 0x2AAAAAABu : 0x80000000u >> (band_rows >> 1);
  const uint32_t column = (uint32_t)((uint64_t)(2 * in_band) * rows_reciprocal >> 32);
  *tile_row = (int)(band_first + in_band - column * band_rows);
  *tile_col = (int)column;
}

}  // namespace uk

#endif  // IREE_AMD_CSRC_UK_DEVICE_H_
