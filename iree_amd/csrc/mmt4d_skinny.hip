// mmt4d for skinny left-hand sides in the narrow tile shapes that the
// reference's CPU targets pick for them: few lhs rows in total (e.g.
// M0 = 1, 2, 4 with M = 1) and row pieces (K0 elements) of 2, 4 or 8 bytes:
// the x86-64 1x16x2 int8 / bf16 and 1x16x1 f16 / f32 tiles, the Arm 1x8x4 and
// 1x8x8 int8 tiles and their 2- and 4-row siblings (mmt4d_x86_64_tiles.inl,
// mmt4d_arm_64_tiles.inl). An HBM-bandwidth kernel.
//
// With pieces that short, 16 contiguous bytes of the rhs are several rows of
// one k step, not one row: the wrong way round for an MFMA operand, and the
// matrix kernels cannot load an lhs whose tiles are narrower than 16 bytes per
// k step at all. Here nothing is transposed. The rhs of one tile row
// (N0 rows x K k steps, one contiguous stream) is read 16 bytes per lane, and
// each lane multiplies the 16 / G rows it holds with the lhs pieces of its
// k step on the VALU (v_dot4_i32_i8, v_dot2_i32_i16, FMAs on 16-bit floats
// widened to f32), keeping one accumulator per (lhs row, rhs row). The lhs is small and comes through the
// caches. At the end the lanes that hold the same rhs rows (they differ in
// k step) are summed by exchanges that halve the values in each step, the wavefronts of the
// workgroup (which split the stream between them) through LDS, both in a
// fixed order, so results do not depend on scheduling.
//
// f16f16f16 and bf16bf16bf16 are taken with the flag that skips the roundings
// between k steps (mmt4d_tile_generic.c:229-286, 319-376): f32 accumulators,
// one rounding to the 16-bit output at the end.
//
// Also here, because nothing else takes them but the generic kernel:
// s16s16s32 (v_dot2_i32_i16) and s16u4s32, the x86-64 VNNI tile 1x32x8 for
// 4-bit weights against 16-bit activations (mmt4d_x86_64_tiles.inl; unsigned
// nibbles, element 2j in the low nibble of byte j, mmt4d_tile_generic.c:108-142):
// a lane's 16 bytes are 4 rows x 8 nibbles of one k step, each byte is spread
// to a pair of 16-bit values and multiplied with the matching pair of the lhs.
// And s8s4s32 with the Arm tiles Mx8x8 and Mx8x16 (mmt4d_arm_64_tiles.inl;
// signed nibbles, mmt4d_tile_generic.c:11-51): the even and the odd nibbles of
// a dword are isolated in the high nibbles of two dwords (int8 values 16 times
// the weights) and multiplied with the even resp. odd lhs bytes of the k step,
// which are gathered once per lhs piece; the sums are shifted right by 4 at
// the end (exact; K * K0 < 131072 keeps 16x the sums inside int32). The Arm
// baseline tiles Mx16x2 have one byte per rhs row and k step: a lane's 16 bytes
// are 16 rows, and each row's two weights (x16, as above) are put beside each
// other in a dword for one v_dot4_i32_i8 with the lhs pair.
// And s16s8s32, for which the reference has the generic tile only
// (mmt4d_tile_generic.c:145-176): the rhs bytes are sign-extended to 16-bit
// pairs (v_perm_b32 with its sign-byte selectors) for v_dot2_i32_i16.
//
// And s8s8s32 Mx8x1 with M0 = 1, 2, 4 (the Arm baseline tiles without dot
// products, mmt4d_arm_64_tiles.inl:38-40): a k step of the rhs is 8 bytes, so a
// lane's 16 bytes are the tile's 8 rows at two consecutive k steps; each row's
// two bytes are put beside each other for one v_dot4_i32_i8 with the two lhs
// bytes of those k steps.
//
// More than 8 lhs rows are worked off in slabs of 8, each streaming the rhs
// again: what the block kernels can load they do faster (the caller prefers
// them), what they cannot is still far better off here than with one thread
// per output element.
#include <type_traits>

#include "uk_device.h"
#include "uk_internal.h"

namespace uk {
namespace {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef _Float16 v2f16 __attribute__((ext_vector_type(2)));
typedef short v2i16 __attribute__((ext_vector_type(2)));

enum Kind { kI8 = 0, kF16 = 1, kBF16 = 2, kF32 = 3, kI16 = 4, kI16U4 = 5, kI8I4 = 6, kI16I8 = 7 };

struct SkinnyArgs {
  const uint8_t* lhs;
  const uint8_t* rhs;
  uint8_t* out;
  int64_t lhs_stride_bytes, rhs_stride_bytes;
  int64_t out_stride0;  // elements
  int64_t tile_bytes;   // K * N0 * (bytes of an rhs row piece): one rhs tile row
  int32_t rows;         // M * M0
  int32_t row0;         // first lhs row of this launch (the kernel covers rows row0 .. row0 + ROWS - 1)
  int32_t N, K;
  int32_t log2_M0, log2_N0;
  int32_t accumulate;
};

template <int KIND> struct Acc { typedef float type; };
template <> struct Acc<kI8> { typedef int32_t type; };
template <> struct Acc<kI16> { typedef int32_t type; };
template <> struct Acc<kI16U4> { typedef int32_t type; };
template <> struct Acc<kI8I4> { typedef int32_t type; };
template <> struct Acc<kI16I8> { typedef int32_t type; };
// The lhs piece of one k step in registers. Same bytes as an rhs piece (G, zero-extended to two dwords), except:
// s16u4s32: 8 values of 16 bits against 8 nibbles; s8s4s32: 8 or 16 bytes against as many nibbles, kept as one
// dword of the even and one of the odd bytes per 8 (2 bytes as they are); s16s8s32: twice the bytes of the rhs piece.
template <int KIND> struct LhsPiece { typedef uint2 type; };
template <> struct LhsPiece<kI16U4> { typedef uint4 type; };
template <> struct LhsPiece<kI8I4> { typedef uint4 type; };
template <> struct LhsPiece<kI16I8> { typedef uint4 type; };

__device__ __forceinline__ int32_t dot2_i16(uint32_t a, uint32_t b, int32_t c) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(v2i16, a), __builtin_bit_cast(v2i16, b), c, false);
}

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ float f16_lo(uint32_t w) { return (float)__builtin_bit_cast(v2f16, w)[0]; }
__device__ __forceinline__ float f16_hi(uint32_t w) { return (float)__builtin_bit_cast(v2f16, w)[1]; }

template <int KIND, int G>
__device__ __forceinline__ typename LhsPiece<KIND>::type load_lhs_piece(const uint8_t* p) {
  if constexpr (KIND == kI16U4) return *(const uint4*)p;
  else if constexpr (KIND == kI16I8) {
    if constexpr (G == 2) return make_uint4(*(const uint32_t*)p, 0, 0, 0);
    else if constexpr (G == 4) {
      const uint2 half = *(const uint2*)p;
      return make_uint4(half.x, half.y, 0, 0);
    } else return *(const uint4*)p;
  } else if constexpr (KIND == kI8I4 && G == 1) return make_uint4(*(const uint16_t*)p, 0, 0, 0);
  else if constexpr (KIND == kI8I4) {
    uint4 raw = make_uint4(0, 0, 0, 0);
    if constexpr (G == 4) {
      const uint2 half = *(const uint2*)p;
      raw.x = half.x; raw.y = half.y;
    } else {
      raw = *(const uint4*)p;
    }
    return make_uint4(__builtin_amdgcn_perm(raw.y, raw.x, 0x06040200u), __builtin_amdgcn_perm(raw.y, raw.x, 0x07050301u),
                      __builtin_amdgcn_perm(raw.w, raw.z, 0x06040200u), __builtin_amdgcn_perm(raw.w, raw.z, 0x07050301u));
  } else if constexpr (G == 2) return make_uint2(*(const uint16_t*)p, 0);
  else if constexpr (G == 4) return make_uint2(*(const uint32_t*)p, 0);
  else return *(const uint2*)p;
}

// acc[r] += (row r of the 16 / G rows in `v`) . (lhs piece l), all of one k step.
template <int KIND, int G>
__device__ __forceinline__ void multiply_piece(const uint4 v, const typename LhsPiece<KIND>::type l,
                                               typename Acc<KIND>::type* acc) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  if constexpr (KIND == kI8I4 && G == 1) {
    // 16 rows of two nibbles each against the lhs pair in the low half of l.x.
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t evens = (w[d] << 4) & 0xF0F0F0F0u, odds = w[d] & 0xF0F0F0F0u;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // byte 0: row r of `evens`, byte 1: row r of `odds`, zeros above
        const uint32_t pair = __builtin_amdgcn_perm(odds, evens, 0x0C0C0400u + 0x0101u * r);
        acc[4 * d + r] = __builtin_amdgcn_sdot4((int)pair, (int)l.x, acc[4 * d + r], false);
      }
    }
  } else if constexpr (KIND == kI16I8) {
    const uint32_t lhs[4] = {l.x, l.y, l.z, l.w};
    // The four bytes of a dword as two pairs of 16-bit values. The selectors 8..11 of
    // v_perm_b32 give the sign of bytes 1, 3 (second operand) and 5, 7 (first operand)
    // as 0x00 or 0xFF; the dword shifted up by a byte has bytes 0 and 2 at 5 and 7.
    uint32_t pairs[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pairs[2 * i] = __builtin_amdgcn_perm(w[i] << 8, w[i], 0x08010A00u);
      pairs[2 * i + 1] = __builtin_amdgcn_perm(w[i] << 8, w[i], 0x09030B02u);
    }
    constexpr int PPR = G / 2;  // pairs per row piece
#pragma unroll
    for (int r = 0; r < 16 / G; ++r)
#pragma unroll
      for (int q = 0; q < PPR; ++q) acc[r] = dot2_i16(pairs[r * PPR + q], lhs[q], acc[r]);
  } else if constexpr (KIND == kI8I4) {
    static_assert(G == 4 || G == 8, "8 or 16 nibbles per row piece");
    const uint32_t lhs[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
    for (int i = 0; i < 16 / G; ++i) {
#pragma unroll
      for (int d = 0; d < G / 4; ++d) {
        const uint32_t nibbles = w[i * (G / 4) + d];
        acc[i] = __builtin_amdgcn_sdot4((int)((nibbles << 4) & 0xF0F0F0F0u), (int)lhs[2 * d], acc[i], false);
        acc[i] = __builtin_amdgcn_sdot4((int)(nibbles & 0xF0F0F0F0u), (int)lhs[2 * d + 1], acc[i], false);
      }
    }
  } else if constexpr (KIND == kI16U4) {
    static_assert(G == 4, "8 nibbles per row piece");
    const uint32_t lhs[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        // byte b of the row: its low nibble to bits 0..3, its high nibble to bits 16..19
        const uint32_t twice = __builtin_amdgcn_perm(0, w[i], 0x0C000C00u + 0x00010001u * b);
        const uint32_t pair = (twice & 0xFu) | ((twice >> 4) & 0x000F0000u);
        acc[i] = dot2_i16(pair, lhs[b], acc[i]);
      }
    }
  } else if constexpr (KIND == kI16) {
    if constexpr (G == 2) {
      // Two rows per dword: the lhs value in the low resp. high half, zero in the other.
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = dot2_i16(w[i], l.x, acc[2 * i]);
        acc[2 * i + 1] = dot2_i16(w[i], l.x << 16, acc[2 * i + 1]);
      }
    } else if constexpr (G == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = dot2_i16(w[i], l.x, acc[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = dot2_i16(w[2 * i + 1], l.y, dot2_i16(w[2 * i], l.x, acc[i]));
    }
  } else if constexpr (KIND == kI8 && G == 1) {
    // 8 rows at k step 2j (bytes 0..7) and at 2j + 1 (bytes 8..15); l.x holds the two lhs bytes.
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const uint32_t pair = __builtin_amdgcn_perm(w[2 + (r >> 2)], w[r >> 2], 0x0C0C0400u + 0x0101u * (r & 3));
      acc[r] = __builtin_amdgcn_sdot4((int)pair, (int)l.x, acc[r], false);
    }
  } else if constexpr (KIND == kI8) {
    if constexpr (G == 2) {
      // Two rows per dword: the lhs pair in the low resp. high half, zeros in the other.
      const int lo = (int)l.x, hi = (int)(l.x << 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = __builtin_amdgcn_sdot4((int)w[i], lo, acc[2 * i], false);
        acc[2 * i + 1] = __builtin_amdgcn_sdot4((int)w[i], hi, acc[2 * i + 1], false);
      }
    } else if constexpr (G == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_sdot4((int)w[i], (int)l.x, acc[i], false);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[i] = __builtin_amdgcn_sdot4((int)w[2 * i], (int)l.x, acc[i], false);
        acc[i] = __builtin_amdgcn_sdot4((int)w[2 * i + 1], (int)l.y, acc[i], false);
      }
    }
  } else if constexpr (KIND == kF32) {
    if constexpr (G == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(__uint_as_float(w[i]), __uint_as_float(l.x), acc[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[i] = fmaf(__uint_as_float(w[2 * i]), __uint_as_float(l.x), acc[i]);
        acc[i] = fmaf(__uint_as_float(w[2 * i + 1]), __uint_as_float(l.y), acc[i]);
      }
    }
  } else {
    // 16-bit floats, widened to f32 (exact) and accumulated in f32 in k0 order.
    auto lo = [](uint32_t x) { return KIND == kF16 ? f16_lo(x) : bf16_lo(x); };
    auto hi = [](uint32_t x) { return KIND == kF16 ? f16_hi(x) : bf16_hi(x); };
    if constexpr (G == 2) {
      const float l0 = lo(l.x);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = fmaf(lo(w[i]), l0, acc[2 * i]);
        acc[2 * i + 1] = fmaf(hi(w[i]), l0, acc[2 * i + 1]);
      }
    } else if constexpr (G == 4) {
      const float l0 = lo(l.x), l1 = hi(l.x);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(hi(w[i]), l1, fmaf(lo(w[i]), l0, acc[i]));
    } else {
      const float l0 = lo(l.x), l1 = hi(l.x), l2 = lo(l.y), l3 = hi(l.y);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[i] = fmaf(hi(w[2 * i]), l1, fmaf(lo(w[2 * i]), l0, acc[i]));
        acc[i] = fmaf(hi(w[2 * i + 1]), l3, fmaf(lo(w[2 * i + 1]), l2, acc[i]));
      }
    }
  }
}

// The value of lane `lane ^ S`.
template <int S>
__device__ __forceinline__ uint32_t exchange(uint32_t v) {
  if constexpr (S == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);        // quad_perm [1, 0, 3, 2]
  else if constexpr (S == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);   // quad_perm [2, 3, 0, 1]
  else if constexpr (S == 4)  // row_half_mirror is ^ 7, quad_perm [3, 2, 1, 0] ^ 3
    return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, v, 0x1B, 0xF, 0xF, true), 0x141, 0xF, 0xF, true);
  else if constexpr (S == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, true);  // row_ror:8
  else return __shfl_xor((int)v, S, 64);
}

// v[i] of the lanes with bit S clear and v[i + HALF] of those with it set are summed over the pair lane, lane ^ S.
template <int S, typename T>
__device__ __forceinline__ T sum_pair(T low, T high, bool set) {
  if constexpr (S >= 16) {
    // (The instruction swaps the upper lanes of the first operand with the lower ones of the second.)
    const uint32_t x = __builtin_bit_cast(uint32_t, low), y = __builtin_bit_cast(uint32_t, high);
    const auto both = S == 32 ? __builtin_amdgcn_permlane32_swap(x, y, false, false) : __builtin_amdgcn_permlane16_swap(x, y, false, false);
    return __builtin_bit_cast(T, (uint32_t)both[0]) + __builtin_bit_cast(T, (uint32_t)both[1]);
  } else {
    const T keep = set ? high : low, send = set ? low : high;
    return keep + __builtin_bit_cast(T, exchange<S>(__builtin_bit_cast(uint32_t, send)));
  }
}

// Sums V values over the lanes that are a multiple of `period` (a power of two) apart, each lane ending with 1 / (64 /
// period) of them or with one, and calls store(first, values, count). Half as many values in each step, not every value in
// every step: 32 values, period 2: 31 exchanges, not 160 (4 x 800 x 1280 f16: 1.0 of 6.9 us were these).
template <int S, int V, typename T, typename Store>
__device__ __forceinline__ void sum_lanes(const T* v, int lane, int period, int first, const Store& store) {
  if (S == 0 || S < period) {
    store(first, v, V);
    return;
  }
  if constexpr (S > 0) {
    const bool set = lane & S;
    if constexpr (V > 1) {
      T half[V / 2];
#pragma unroll
      for (int i = 0; i < V / 2; ++i) half[i] = sum_pair<S>(v[i], v[i + V / 2], set);
      sum_lanes<S / 2, V / 2>(half, lane, period, first + (set ? V / 2 : 0), store);
    } else {
      const T sum = v[0] + __builtin_bit_cast(T, exchange<S>(__builtin_bit_cast(uint32_t, v[0])));
      sum_lanes<S / 2, 1>(&sum, lane, period, first, store);
    }
  }
}

// Bytes of an lhs k step in registers, where one load takes the pieces of all rows.
template <int BYTES>
struct alignas(BYTES < 16 ? BYTES : 16) LhsStep { uint32_t dwords[BYTES / 4]; };

// Whether the lhs's row pieces are as long as the rhs's, and two rows of them whole dwords.
template <int KIND, int G>
constexpr bool kPackedLhs = G > 1 && (KIND == kI8 || KIND == kI16 || KIND == kF16 || KIND == kBF16 || KIND == kF32);

// G: bytes of a row piece; ROWS: lhs rows the kernel keeps accumulators for
// (a.rows <= ROWS); UNROLL: 1 KiB blocks of the rhs stream a wavefront has in
// flight, a ring of registers each loaded again as soon as it is multiplied;
// STREAMED: the rhs is read past the caches; NARROW: the output has the
// 16-bit type of the operands; PACKED: there is one lhs tile, of ROWS rows, whose
// k steps are loaded whole: with a load of 2 to 8 bytes for each of four rows
// beside 16 bytes of rhs, the loads' issue is the limit (4 x 2432 x 4988 f16
// 9.6 -> 6.7 us). One workgroup per rhs tile row.
template <int KIND, int G, int ROWS, int WAVES, int UNROLL, bool STREAMED, bool NARROW, bool PACKED>
__global__ __launch_bounds__(64 * WAVES) void mmt4d_skinny_kernel(const SkinnyArgs a) {
  static_assert(!NARROW || KIND == kF16 || KIND == kBF16, "16-bit outputs are floats");
  static_assert(!PACKED || (kPackedLhs<KIND, G> && ROWS > 1), "k steps of whole dwords");
  typedef typename Acc<KIND>::type acc_t;
  typedef typename LhsPiece<KIND>::type piece_t;
  // (One-byte pieces of int8: 8-row tiles, two k steps per lane.)
  constexpr bool TWO_KSTEPS = KIND == kI8 && G == 1;
  constexpr int R = TWO_KSTEPS ? 8 : 16 / G;  // rhs rows in a lane's 16 bytes
  __shared__ acc_t partial[WAVES][ROWS][32];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int32_t M0 = 1 << a.log2_M0, N0 = 1 << a.log2_N0;
  // One k step of the rhs is N0 * G bytes = `lanes_per_kstep` lanes; a block of
  // 1 KiB holds whole k steps, so a lane keeps its rows from block to block.
  const int log2_kstep_bytes = a.log2_N0 + (G == 1 ? 0 : (G == 2 ? 1 : (G == 4 ? 2 : 3)));
  const int log2_lanes_per_kstep = TWO_KSTEPS ? 0 : log2_kstep_bytes - 4;
  const int32_t kstep_in_block = TWO_KSTEPS ? 2 * lane : lane >> log2_lanes_per_kstep;
  constexpr int LHS_G = KIND == kI16U4 ? 16 : (KIND == kI8I4 || KIND == kI16I8 ? 2 * G : G);  // bytes of an lhs row piece
  const int32_t lhs_kstep_bytes = PACKED ? LHS_G * ROWS : LHS_G << a.log2_M0;

  const uint8_t* rhs = a.rhs + (int64_t)blockIdx.x * a.rhs_stride_bytes + 16 * lane;
  const int64_t lhs_lane = (int64_t)kstep_in_block * lhs_kstep_bytes;
  const int64_t lhs_block = (int64_t)lhs_kstep_bytes << (10 - log2_kstep_bytes);  // bytes of the lhs k steps of a block
  constexpr int LHS_ROWS = PACKED ? 1 : ROWS;
  const uint8_t* lhs_row[LHS_ROWS];
#pragma unroll
  for (int m = 0; m < LHS_ROWS; ++m) {
    const int row = PACKED ? 0 : min(a.row0 + m, a.rows - 1);  // clamp: computed, not stored
    lhs_row[m] = a.lhs + (int64_t)(row >> a.log2_M0) * a.lhs_stride_bytes + (row & (M0 - 1)) * LHS_G + lhs_lane;
  }

  acc_t acc[ROWS * R];
#pragma unroll
  for (int i = 0; i < ROWS * R; ++i) acc[i] = 0;

  typedef typename std::conditional<PACKED, LhsStep<PACKED ? LHS_G * ROWS : 4>, piece_t>::type lhs_t;
  auto load_lhs = [&](lhs_t* l, int64_t block, bool second_kstep) {
#pragma unroll
    for (int m = 0; m < LHS_ROWS; ++m) {
      const uint8_t* p = lhs_row[m] + block * lhs_block;
      if constexpr (PACKED) l[m] = *(const lhs_t*)p;
      else if constexpr (TWO_KSTEPS) l[m] = make_uint2((uint32_t)p[0] | ((second_kstep ? p[lhs_kstep_bytes] : 0u) << 8), 0);
      else l[m] = load_lhs_piece<KIND, G>(p);
    }
  };
  auto multiply = [&](const uint4 v, const lhs_t* l) {
#pragma unroll
    for (int m = 0; m < ROWS; ++m) {
      if constexpr (PACKED) {
        const uint32_t* d = l[0].dwords;
        piece_t piece;
        if constexpr (G == 2) piece = make_uint2(m & 1 ? d[m / 2] >> 16 : d[m / 2] & 0xFFFFu, 0);
        else if constexpr (G == 4) piece = make_uint2(d[m], 0);
        else piece = make_uint2(d[2 * m], d[2 * m + 1]);
        multiply_piece<KIND, G>(v, piece, acc + m * R);
      } else {
        multiply_piece<KIND, G>(v, l[m], acc + m * R);
      }
    }
  };

  // The blocks are dealt to the wavefronts in turn. What is left behind the last whole one goes to the last wavefront:
  // lanes beyond the stream's end multiply zeros, whatever the lhs holds there.
  const int32_t full = (int32_t)(a.tile_bytes >> 10);
  const int32_t rest_bytes = (int32_t)(a.tile_bytes & 1023);
  const bool has_rest = wave == WAVES - 1 && rest_bytes != 0;
  uint4 rest_v = make_uint4(0, 0, 0, 0);
  lhs_t rest_l[LHS_ROWS] = {};
  if (has_rest && 16 * lane < rest_bytes) {
    const uint8_t* p = rhs + ((int64_t)full << 10);
    if (TWO_KSTEPS && 16 * lane + 16 > rest_bytes) {
      // An odd K: the stream ends after this lane's first k step.
      const uint2 half = *(const uint2*)p;
      rest_v.x = half.x;
      rest_v.y = half.y;
    } else {
      rest_v = *(const uint4*)p;
    }
    load_lhs(rest_l, full, 16 * lane + 16 <= rest_bytes);
  }

  uint4 v[UNROLL];
  lhs_t l[UNROLL][LHS_ROWS];
  int32_t left = (full + WAVES - 1 - wave) / WAVES;
  int64_t block = wave;
  auto load = [&](int u) {
    const uint8_t* p = rhs + ((block + u * WAVES) << 10);
    if constexpr (STREAMED) v[u] = __builtin_bit_cast(uint4, __builtin_nontemporal_load((const v4i32*)p));
    else v[u] = *(const uint4*)p;
    load_lhs(l[u], block + u * WAVES, true);
  };
  auto next_batch = [&] {
    left -= UNROLL;
    block += UNROLL * WAVES;
  };
  if (left >= UNROLL) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) load(u);
    next_batch();
    while (left >= UNROLL) {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        multiply(v[u], l[u]);
        load(u);
        __builtin_amdgcn_sched_barrier(0);  // (no load moves in front of the multiplication of what its registers hold)
      }
      next_batch();
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      multiply(v[u], l[u]);
      if (u < left) load(u);
    }
  } else {
#pragma unroll
    for (int u = 0; u < UNROLL - 1; ++u)
      if (u < left) load(u);
  }
#pragma unroll
  for (int u = 0; u < UNROLL - 1; ++u)
    if (u < left) multiply(v[u], l[u]);
  if (has_rest) multiply(rest_v, rest_l);

  // Lanes that are a multiple of lanes_per_kstep apart hold the same rhs rows.
  const int32_t lanes_per_kstep = 1 << log2_lanes_per_kstep;
  sum_lanes<32, ROWS * R>(acc, lane, lanes_per_kstep, 0, [&](int first, const acc_t* sums, int count) {
    for (int i = 0; i < count; ++i)
      partial[wave][(first + i) / R][R * (lane & (lanes_per_kstep - 1)) + (first + i) % R] = sums[i];
  });
  __syncthreads();
  const int t = threadIdx.x;
  const int slab_row = t >> a.log2_N0, j0 = t & (N0 - 1);
  const int m = a.row0 + slab_row;
  if (slab_row < ROWS && m < a.rows) {
    acc_t sum = partial[0][slab_row][j0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += partial[w][slab_row][j0];
    if constexpr (KIND == kI8I4) sum >>= 4;
    const int64_t index = (int64_t)(m >> a.log2_M0) * a.out_stride0 +
                          ((int64_t)blockIdx.x << (a.log2_M0 + a.log2_N0)) + ((m & (M0 - 1)) << a.log2_N0) + j0;
    if constexpr (NARROW) {
      constexpr int EBITS = KIND == kF16 ? 5 : 8;
      uint16_t* dst = (uint16_t*)a.out + index;
      if (a.accumulate) sum += widen16<EBITS>(*dst);
      *dst = narrow16<EBITS>(sum);
    } else {
      acc_t* dst = (acc_t*)a.out + index;
      if (a.accumulate) sum += *dst;
      *dst = sum;
    }
  }
}

int log2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1))) return -1;
  int l = 0;
  while ((1ll << l) < v) ++l;
  return l;
}

bool make_args(const Mmt4dArgs& a, bool probe_only, int* kind, int* piece_bytes, bool* narrow, SkinnyArgs* s) {
  int elem_bytes;
  *narrow = false;
  const bool skip_roundings = a.flags & IREE_UK_FLAG_MMT4D_SKIP_INTERMEDIATE_ROUNDINGS;
  switch (a.flags & IREE_UK_FLAG_MMT4D_TYPE_MASK) {
    case IREE_UK_FLAG_MMT4D_TYPE_S8S8S32: *kind = kI8; elem_bytes = 1; break;
    case IREE_UK_FLAG_MMT4D_TYPE_F16F16F32: *kind = kF16; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_BF16BF16F32: *kind = kBF16; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_F32F32F32: *kind = kF32; elem_bytes = 4; break;
    case IREE_UK_FLAG_MMT4D_TYPE_S16S16S32: *kind = kI16; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_S16U4S32: *kind = kI16U4; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_S8S4S32: *kind = kI8I4; elem_bytes = 1; break;
    case IREE_UK_FLAG_MMT4D_TYPE_S16S8S32: *kind = kI16I8; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_F16F16F16:
      if (!skip_roundings) return false;
      *kind = kF16; elem_bytes = 2; *narrow = true;
      break;
    case IREE_UK_FLAG_MMT4D_TYPE_BF16BF16BF16:
      if (!skip_roundings) return false;
      *kind = kBF16; elem_bytes = 2; *narrow = true;
      break;
    default: return false;
  }
  const bool u4 = *kind == kI16U4, i4 = *kind == kI8I4, i16i8 = *kind == kI16I8;
  if (u4 && a.K0 != 8) return false;
  if (i4 && a.K0 != 2 && a.K0 != 8 && a.K0 != 16) return false;
  const int g = u4 ? 4 : (i4 ? a.K0 / 2 : (i16i8 ? a.K0 : a.K0 * elem_bytes));  // bytes of an rhs row piece
  const int lhs_g = u4 ? 16 : (i4 ? a.K0 : (i16i8 ? 2 * a.K0 : g));
  // int8 Mx8x1 (8x8x1 goes to the matrix kernels first, see mmt4d_skinny_preferred, and comes here when they cannot
  // load it: K shorter than a chunk, misaligned lhs).
  const bool two_ksteps = *kind == kI8 && g == 1 && a.N0 == 8 && a.M0 <= 8;
  if (g != 2 && g != 4 && g != 8 && !(i4 && g == 1) && !two_ksteps) return false;
  const int lm0 = log2_exact(a.M0), ln0 = log2_exact(a.N0);
  // A k step of the rhs must be whole 16-byte vectors (or half of one, above).
  if (lm0 < 0 || ln0 < 0 || a.M0 > 16 || a.N0 > 32 || (a.N0 * g < 16 && !two_ksteps)) return false;
  *piece_bytes = g;
  // What no matrix kernel takes.
  if (probe_only) return a.M0 * lhs_g < 16 || *kind == kI16 || u4 || i16i8 || (i4 && a.K0 < 16);
  // 16x-scaled int4 accumulation must not overflow int32.
  if (i4 && (int64_t)a.K * a.K0 >= 131072) return false;
  if (a.M * a.M0 > 0x7FFFFFFF || a.M <= 0 || a.K <= 0 || a.N <= 0 || a.N > 0x7FFFFFFF) return false;
  if ((u4 || i4) && (a.rhs_stride0 & 1)) return false;
  const int64_t lhs_stride_bytes = a.lhs_stride0 * elem_bytes;
  const int64_t rhs_stride_bytes = (u4 || i4) ? a.rhs_stride0 / 2 : (i16i8 ? a.rhs_stride0 : a.rhs_stride0 * elem_bytes);
  if ((uintptr_t)a.rhs % 16 || (a.N > 1 && rhs_stride_bytes % 16)) return false;
  if ((uintptr_t)a.lhs % lhs_g || (a.M > 1 && lhs_stride_bytes % lhs_g)) return false;
  if ((uintptr_t)a.out % (*narrow ? 2 : 4)) return false;
  s->lhs = a.lhs; s->rhs = a.rhs; s->out = a.out;
  s->lhs_stride_bytes = lhs_stride_bytes;
  s->rhs_stride_bytes = rhs_stride_bytes;
  s->out_stride0 = a.out_stride0;
  s->tile_bytes = a.K * a.N0 * g;
  s->rows = (int32_t)(a.M * a.M0);
  s->row0 = 0;
  s->N = (int32_t)a.N;
  s->K = (int32_t)a.K;
  s->log2_M0 = lm0;
  s->log2_N0 = ln0;
  s->accumulate = (a.flags & IREE_UK_FLAG_MMT4D_ACCUMULATE) ? 1 : 0;
  return true;
}

// Whether the lhs is one tile of 2 or 4 rows that is aligned to its k steps.
bool lhs_is_packed(const SkinnyArgs& s, int piece_bytes) {
  const int kstep = piece_bytes * s.rows;
  return s.rows == 1 << s.log2_M0 && (s.rows == 2 || s.rows == 4) && (uintptr_t)s.lhs % (kstep < 16 ? kstep : 16) == 0;
}

// PACKED_UNROLL: UNROLL for an lhs tile of 2 or 4 rows that is aligned to its k steps. Other lhs have a load for each row
// beside one of the rhs, and more registers to each step (3 x 4096 x 4096 f32 of 8-byte pieces: 17.8 us with eight wavefronts
// of four blocks, 12.1 of two).
template <int KIND, int G, int WAVES, int PACKED_UNROLL, bool STREAMED, bool NARROW>
hipError_t launch_slabs(const SkinnyArgs& all_rows, hipStream_t stream) {
  void (*kernel)(const SkinnyArgs);
  SkinnyArgs s = all_rows;
  auto launch = [&](int waves = WAVES) { return launch_kernel(kernel, (unsigned)all_rows.N, 64 * waves, 0, stream, s); };
  if constexpr (kPackedLhs<KIND, G>) {
    if (lhs_is_packed(s, G)) {
      kernel = s.rows == 2 ? mmt4d_skinny_kernel<KIND, G, 2, WAVES, PACKED_UNROLL, STREAMED, NARROW, true>
                           : mmt4d_skinny_kernel<KIND, G, 4, WAVES, PACKED_UNROLL, STREAMED, NARROW, true>;
      return launch();
    }
  }
  // More than 8 rows: one launch per slab of 8. Five rows and more have a ring of two blocks (8 x 4096 x 4096 s16u4 9.9 us, of
  // four 19.7, s16s8 10.8 and 11.4, int8 in 4x16x2 tiles 8.0 and 9.1, f32 in 2x16x1 12.6 and 13.8), but s16 in 4-byte pieces
  // from HBM, which needs the bytes in flight, one of four (16 x 14336 x 4096 64.2 -> 57.4, 8 x 14336 x 4096 24.8 -> 23.1). int4
  // in 1-byte pieces, 32 sums a row, does not fit the registers that eight wavefronts leave (31 spilled) and has four (8 x
  // 4096 x 4096 9.6 -> 8.0, 8 x 1024 x 1024 5.7 -> 4.8).
  constexpr int WAVES_8_ROWS = KIND == kI8I4 && G == 1 ? 4 : WAVES, UNROLL_8_ROWS = KIND == kI16 && G == 4 && STREAMED ? 4 : 2;
  for (s.row0 = 0; s.row0 < s.rows; s.row0 += 8) {
    const int left = s.rows - s.row0;
    if (left <= 1) kernel = mmt4d_skinny_kernel<KIND, G, 1, WAVES, 4, STREAMED, NARROW, false>;
    else if (left <= 2) kernel = mmt4d_skinny_kernel<KIND, G, 2, WAVES, 4, STREAMED, NARROW, false>;
    else if (left <= 4) kernel = mmt4d_skinny_kernel<KIND, G, 4, WAVES, G == 8 && WAVES == 8 ? 2 : 4, STREAMED, NARROW, false>;
    else kernel = mmt4d_skinny_kernel<KIND, G, 8, WAVES_8_ROWS, UNROLL_8_ROWS, STREAMED, NARROW, false>;
    const hipError_t e = launch(left <= 4 ? WAVES : WAVES_8_ROWS);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int KIND, int G, bool NARROW>
hipError_t launch_piece(const SkinnyArgs& s, hipStream_t stream) {
  const int64_t bytes = s.tile_bytes * s.N;
  // No more tile rows than compute units: eight wavefronts, 4 KiB in flight each (1 x 880 x 8918 bf16 9.3 -> 6.5 us, with 8
  // KiB in each of four 7.3; 2 x 1984 x 4991 f16 7.1 -> 5.5, 6.1).
  // int8, up to two rows and tiles of 128 KiB and more: 8 KiB each (2 x 592 x 9334 4.7, 4.8 with four, 1 x 816 x 9740 4.4, 4.7;
  // near 256 tile rows 2 to 7 % behind four: 2 x 4096 x 14336 10.7, 10.3).
  if constexpr (KIND == kI8 && G > 1) {
    if (s.N <= 256 && s.rows <= 2 && s.tile_bytes >= 128 * 1024) {
      if (s.rows == 1) return launch_kernel<SkinnyArgs>(mmt4d_skinny_kernel<KIND, G, 1, 8, 8, false, NARROW, false>, (unsigned)s.N, 512, 0, stream, s);
      if (lhs_is_packed(s, G)) return launch_kernel<SkinnyArgs>(mmt4d_skinny_kernel<KIND, G, 2, 8, 8, false, NARROW, true>, (unsigned)s.N, 512, 0, stream, s);
    }
  }
  if (s.N <= 256) return launch_slabs<KIND, G, 8, 4, false, NARROW>(s, stream);
  // One byte or less per rhs element against more than two rows is slowed down by streaming: 4 x 14336 x 4096 int8 17.6 us,
  // streamed 20.6, from HBM 20.9 both; only beyond what the caches can hold it gains (235 MB: 60.8 -> 56.8).
  const bool one_byte = KIND == kI8 || KIND == kI8I4 || KIND == kI16U4 || KIND == kI16I8;
  const bool streamed = one_byte && s.rows > 2 ? bytes > (128ll << 20) : comes_from_hbm(bytes);
  // One row and more than two tile rows a unit, from HBM: 12 KiB in flight in each of four wavefronts (1 x 24320 x 3664 int8
  // 15.4 -> 14.3, 1 x 16816 x 7722 23.4 -> 22.7). Their rings take 48 KiB of a tile and eight wavefronts' 32 KiB, and what is
  // left of the tile is read with fewer loads in flight: tiles of 64 to 96 and of 128 to 144 KiB leave less to eight (290
  // problems, 32 to 560 KiB: 2.5 % faster in the mean there, 1 x 14336 x 4096 bf16 20.6 -> 19.4 and x 4160 21.5 -> 20.8, 1 x
  // 16352 x 2964 f16 17.8 -> 16.4, 1 x 20000 x 5120 int8 17.6 -> 16.4); elsewhere eight are 1.2 % slower, at 256 KiB 4.5 %.
  // From the caches eight for tiles of 64 KiB and more.
  if (s.rows == 1 && s.N > 512) {
    const int64_t kib = s.tile_bytes >> 10;
    const bool eight = streamed ? (kib >= 64 && kib < 96) || (kib >= 128 && kib < 144) : kib >= 64;
    if (streamed)
      return eight ? launch_kernel<SkinnyArgs>(mmt4d_skinny_kernel<KIND, G, 1, 8, 4, true, NARROW, false>, (unsigned)s.N, 512, 0, stream, s)
                   : launch_kernel<SkinnyArgs>(mmt4d_skinny_kernel<KIND, G, 1, 4, 12, true, NARROW, false>, (unsigned)s.N, 256, 0, stream, s);
    if (eight) return launch_slabs<KIND, G, 8, 4, false, NARROW>(s, stream);
  }
  // Several rows and more than two tile rows a unit: 8 KiB in flight (4 x 9616 x 6381 f16 23.7, with 4 KiB 25.1; 4 x 5312 x
  // 6146 int8, two to a unit, 8.9 and 8.1).
  if (s.rows > 1 && s.N > 512)
    return streamed ? launch_slabs<KIND, G, 4, 8, true, NARROW>(s, stream) : launch_slabs<KIND, G, 4, 8, false, NARROW>(s, stream);
  return streamed ? launch_slabs<KIND, G, 4, 4, true, NARROW>(s, stream) : launch_slabs<KIND, G, 4, 4, false, NARROW>(s, stream);
}

template <int KIND, bool NARROW>
hipError_t launch_kind(const SkinnyArgs& s, int piece_bytes, hipStream_t stream) {
  if (piece_bytes == 4) return launch_piece<KIND, 4, NARROW>(s, stream);
  if (piece_bytes == 8) return launch_piece<KIND, 8, NARROW>(s, stream);
  if constexpr (KIND == kI8) {
    if (piece_bytes == 1) return launch_piece<KIND, 1, NARROW>(s, stream);
  }
  if constexpr (KIND != kF32) return launch_piece<KIND, 2, NARROW>(s, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_skinny(const Mmt4dArgs& a, hipStream_t stream, const char** name) {
  int kind, piece_bytes;
  bool narrow;
  SkinnyArgs s;
  if (!make_args(a, false, &kind, &piece_bytes, &narrow, &s)) return hipErrorInvalidValue;
  *name = "mmt4d_skinny";
  switch (kind) {
    case kI8: return launch_kind<kI8, false>(s, piece_bytes, stream);
    case kF16:
      return narrow ? launch_kind<kF16, true>(s, piece_bytes, stream) : launch_kind<kF16, false>(s, piece_bytes, stream);
    case kBF16:
      return narrow ? launch_kind<kBF16, true>(s, piece_bytes, stream) : launch_kind<kBF16, false>(s, piece_bytes, stream);
    case kI16: return launch_kind<kI16, false>(s, piece_bytes, stream);
    case kI16U4: return launch_piece<kI16U4, 4, false>(s, stream);
    case kI8I4:
      if (piece_bytes == 1) return launch_piece<kI8I4, 1, false>(s, stream);
      return piece_bytes == 4 ? launch_piece<kI8I4, 4, false>(s, stream) : launch_piece<kI8I4, 8, false>(s, stream);
    case kI16I8: return launch_kind<kI16I8, false>(s, piece_bytes, stream);
    default: return launch_kind<kF32, false>(s, piece_bytes, stream);
  }
}

}  // namespace

// Measured on 1 x 14336 x 4096 problems: with up to 4 lhs rows this kernel is
// at the HBM rate (bf16 1x16x2 18 us, int8 1x16x2 10 us) and level with the
// 64x64 matrix kernel where that applies; with 8 rows it is VALU bound (int8
// 8x16x2 41 us against 23 us, bf16 8x16x2 32 against 23 us).
bool mmt4d_skinny_preferred(const Mmt4dArgs& a) {
  int lhs_bits, rhs_bits, out_bits;
  if (!mmt4d_type_bits(a.flags, &lhs_bits, &rhs_bits, &out_bits)) return false;
  // (8-row tiles of one-byte pieces are 8 bytes per k step, but the matrix kernels load them k-major.)
  const bool k_major_for_mfma = a.K0 * lhs_bits == 8 && a.M0 >= 8;
  return a.M * a.M0 <= 4 || (a.M0 * a.K0 * lhs_bits / 8 < 16 && !k_major_for_mfma);
}

Mmt4dLauncher select_mmt4d_skinny(const Mmt4dArgs& a, bool probe_only) {
  int kind, piece_bytes;
  bool narrow;
  SkinnyArgs s;
  return make_args(a, probe_only, &kind, &piece_bytes, &narrow, &s) ? launch_skinny : nullptr;
}

}  // namespace uk
