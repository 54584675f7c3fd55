// MFMA mmt4d for gfx950: s8s8s32, s8s4s32, f16f16f32 and bf16bf16f32.
//
// One workgroup of 256 threads (4 wavefronts in a 2x2 arrangement) computes a
// block of (64*AM) lhs rows x (64*BN) rhs rows of the logical matrix; each
// wavefront owns a (32*AM) x (32*BN) sub-block as AM x BN accumulator
// fragments of one 32x32 MFMA each (v_mfma_i32_32x32x32_i8,
// v_mfma_f32_32x32x16_f16/bf16: a single wavefront per SIMD keeps the matrix
// pipe busy with these, which it cannot with the 16x16 shapes). The K dimension
// is walked in chunks of 64 BYTES per operand row (64 int8 or 32 f16/bf16
// values = two MFMA K-steps).
//
// Two kernels share this tiling and the epilogue:
//   mmt4d_mfma_direct_kernel (the fast path): operands go global memory ->
//     LDS directly, 16 contiguous bytes per lane, through a ring of LDS stages
//     filled several chunks ahead; needs 16-byte aligned operand rows and at
//     least one full chunk of K (where K ends inside a chunk, chunk 1 begins
//     inside chunk 0, which has what they share zeroed: mmt4d_chunk_walk.h).
//   mmt4d_mfma_kernel (everything else the plan admits: 4-byte aligned
//     operands, narrow tiles, less than a chunk of K, an int4 rhs of 8-byte row
//     pieces): global -> registers (issued two chunks ahead) -> LDS -> registers (read one chunk ahead) -> MFMA.
// In both, LDS holds the operands fragment-major, so that a wavefront fetches
// a 32-row x 32-byte MFMA operand with conflict-free reads that are linear in
// the lane number.
//
// Operand layouts. An mmt4d operand row (one i0 of one tile) is not contiguous
// in memory: its K0 values of consecutive k are M0*K0 elements apart
// (mmt4d_tile_generic.c:70-71). With RB = bytes of one (k, i0) row piece:
//   RB multiple of 16: a lane's 16 operand bytes are contiguous in memory;
//   RB == 4 (the 8x8x4 int8 tiles): a lane's 16 bytes come from 4 different k
//     steps. K is permuted inside a chunk, identically for lhs and rhs, which
//     leaves every integer sum unchanged (and reorders a float sum).
// The int4 rhs of s8s4s32 is widened in registers: nibble n becomes the int8
// value 16*n (sign in bit 7, no sign-extension step), the accumulators
// therefore hold 16x the result and are shifted right by 4 at the end, which
// is exact while 16*128*8*depth < 2^31.
//
// The MFMA is issued with the rhs fragment as its row operand and the lhs
// fragment as its column operand, so a lane ends up with 4 consecutive j0 of
// one output row: one 128-bit store per fragment into the [M0][N0] tile.
#ifndef IREE_AMD_CSRC_MMT4D_MFMA_KERNELS_H_
#define IREE_AMD_CSRC_MMT4D_MFMA_KERNELS_H_

#include <type_traits>

#include "mmt4d_chunk_walk.h"
#include "uk_device.h"
#include "uk_internal.h"

namespace uk {

enum MfmaKind { kI8 = 0, kF16 = 1, kBF16 = 2, kF32 = 3 };

struct MfmaArgs {
  const uint8_t* lhs;
  const uint8_t* rhs;
  uint8_t* out;
  int64_t lhs_stride_bytes;  // between consecutive lhs tiles rows (i)
  int64_t rhs_stride_bytes;
  int64_t out_stride0;       // elements
  int32_t M, N, K;           // tile counts
  int32_t log2_M0, log2_N0;
  int32_t lhs_rb, rhs_rb;    // bytes of one (k, i0) row piece
  int32_t log2_lhs_rb, log2_rhs_rb;
  int32_t chunks;            // ceil(K * lhs_rb / 64)
  int32_t tile_rows, tile_cols;  // grid of block tiles (set_tile_grid)
  uint32_t band_reciprocal;      // of tile_cols, see uk_device.h
  int32_t accumulate;
};

// One entry per translation unit of kernel instantiations (they are split by
// type so that they compile side by side). `gather` is 16 or 4 (bytes of one
// contiguous row piece that a lane's 16 operand bytes are made of); `narrow`:
// the output is the 16-bit type of the operands (one rounding at the end).
hipError_t launch_mfma_i8(const MfmaArgs& m, int gather, bool rhs_i4, hipStream_t stream, const char** name);
hipError_t launch_mfma_f16(const MfmaArgs& m, int gather, bool narrow, hipStream_t stream, const char** name);
hipError_t launch_mfma_bf16(const MfmaArgs& m, int gather, bool narrow, hipStream_t stream, const char** name);
hipError_t launch_mfma_f32(const MfmaArgs& m, int gather, hipStream_t stream, const char** name);
hipError_t launch_mfma_f16_narrow(const MfmaArgs& m, int gather, hipStream_t stream, const char** name);
hipError_t launch_mfma_bf16_narrow(const MfmaArgs& m, int gather, hipStream_t stream, const char** name);

// Whether the direct-to-LDS kernel covers the problem with row pieces of
// `gather` bytes (2 and 8 have no other MFMA kernel).
bool mfma_direct_covers(const MfmaArgs& m, int gather, bool rhs_i4);

// The kernel that splits K over a workgroup's wavefronts (mmt4d_wave_k_kernels.h): its tiles, smallest first, and its
// entry per translation unit. `shape` numbers the tiles; `streamed`: read the rhs with non-temporal loads.
struct WaveKShape {
  int fa, fb;  // 16-row fragments of the lhs and of the rhs
  const char* name;
};
constexpr WaveKShape kWaveKShapes[] = {{1, 1, "mmt4d_mfma_wave_k_16x16"}, {1, 2, "mmt4d_mfma_wave_k_16x32"}, {2, 2, "mmt4d_mfma_wave_k_32x32"},
                                       {2, 4, "mmt4d_mfma_wave_k_32x64"}, {4, 2, "mmt4d_mfma_wave_k_64x32"}, {4, 4, "mmt4d_mfma_wave_k_64x64"}};
// f32 is bound by the matrix pipe whatever the tile, and what counts is how evenly the tiles fill the compute units: there is
// one for every size up to 20 fragments (what the LDS holds of partial sums) that has a use. 80 x 10240 x 3648 takes 108 us
// in 32x32 tiles and 55 in 80x48 ones (a library product 64), 2704 x 208 x 4032 69 in 64x64 and 41 in 32x80.
constexpr WaveKShape kWaveKShapesF32[] = {
    {1, 1, "mmt4d_mfma_wave_k_16x16"}, {1, 2, "mmt4d_mfma_wave_k_16x32"}, {2, 2, "mmt4d_mfma_wave_k_32x32"},
    {2, 3, "mmt4d_mfma_wave_k_32x48"}, {3, 2, "mmt4d_mfma_wave_k_48x32"}, {2, 4, "mmt4d_mfma_wave_k_32x64"},
    {4, 2, "mmt4d_mfma_wave_k_64x32"}, {3, 3, "mmt4d_mfma_wave_k_48x48"}, {2, 5, "mmt4d_mfma_wave_k_32x80"},
    {5, 2, "mmt4d_mfma_wave_k_80x32"}, {3, 4, "mmt4d_mfma_wave_k_48x64"}, {4, 3, "mmt4d_mfma_wave_k_64x48"},
    {3, 5, "mmt4d_mfma_wave_k_48x80"}, {5, 3, "mmt4d_mfma_wave_k_80x48"}, {4, 4, "mmt4d_mfma_wave_k_64x64"},
    {4, 5, "mmt4d_mfma_wave_k_64x80"}, {5, 4, "mmt4d_mfma_wave_k_80x64"}};
// Whether it loads the 4-byte row pieces of a tile of fa x fb fragments one at a time rather than through LDS. An instruction
// then covers 16 rows at four k steps. Over 855 products of int8 and bf16 (operand tiles of 4, 8 and 16 rows, every tile of
// this kernel, K of 300 to 12280) that takes 7 % less time in the mean, 4 % with one fragment, 11 % with 16, whatever the
// tile shapes (bf16 16x16x2, 512 x 2048 x 8192 29.1 -> 23.9 us; int8 8x8x4, 32 x 1680 x 6784 6.8 -> 5.8), and f32, bound
// by the matrix pipe, gains 12 to 20 % (8x8x1, 128 x 4096 x 2048 26.5 -> 21.8). Only where the 16 rows are those of four
// tiles a multiple of 512 bytes apart, on the same memory channels, it is up to 25 % slower (int8 4x8x4, 64 x 4096 x 8192 in
// 64x32 tiles; at 108 x 3072 x 8552 15.4 -> 13.1 us); not for the lhs with rhs tiles of 16 rows and more
// fragments of those (4x16x4 and 4x16x2 2 to 9 % faster there too).
inline bool wave_k_loads_pieces(const MfmaArgs& m, int kind, int gather, int fa, int fb) {
  if (gather != 4) return false;
  if (kind == kF32) return true;
  if (m.log2_N0 <= 2 && m.N > 1 && m.rhs_stride_bytes % 512 == 0) return false;
  if (m.log2_M0 <= 2 && m.M > 1 && m.lhs_stride_bytes % 512 == 0) return m.log2_N0 == 4 && fb > fa;
  return true;
}
hipError_t launch_wave_k_i8(const MfmaArgs& m, int gather, bool rhs_i4, int shape, bool streamed, hipStream_t stream);
hipError_t launch_wave_k_f16(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream);
hipError_t launch_wave_k_bf16(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream);
hipError_t launch_wave_k_f32(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream);
hipError_t launch_wave_k_f16_narrow(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream);
hipError_t launch_wave_k_bf16_narrow(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream);

// The kernel whose wavefronts multiply the whole of a large tile each (mmt4d_wave_tile.hip): 128x128 for 16-bit operands,
// 64x128 for an int4 rhs.
hipError_t launch_wave_tile(const MfmaArgs& m, int kind, bool rhs_i4, bool narrow, hipStream_t stream);

// The block tiles of the block kernels. Larger ones move fewer operand bytes per multiply through L2 -> LDS and run the
// matrix pipe longer between barriers, smaller ones spread a problem over more compute units; those with a side of 192
// are there for the problems that leave a last round of 128- or 256-wide tiles nearly empty (bf16 752 x 10928 x 2272 has
// 516 tiles of 128x128 for 256 compute units: 56 us, and 228 of 192x192: 39 us).
struct TileChoice {
  int am, bn;
  bool direct_only;  // no register-staged instantiation of this shape
};

// The 128x64 tile with K split over its wavefronts (mmt4d_mfma_split_k_kernel): 65 to 128 lhs rows, one row of tiles.
// (bf16 128 x 14336 x 4096 27 -> 25 us, 96 rows 27 -> 23 us, 128 x 8192 x 8192 40 -> 36 us. Not with less K per
// row, where the prologue and the summing of the partial tiles cost what the steps gain; not with more tiles than
// compute units, where 128x128 tiles win: bf16 128 x 28672 x 4096 41 -> 49 us.)
inline bool split_k_covers(const MfmaArgs& m) {
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  const int64_t row_bytes = (int64_t)m.K * m.lhs_rb;
  return rows > 64 && rows <= 128 && cols <= 256 * 64 && row_bytes % 128 == 0 && row_bytes >= 8192;
}

constexpr TileChoice kBlockTiles[] = {{4, 4, false}, {4, 2, true}, {2, 2, false}, {2, 1, true}, {1, 1, false}, {1, 2, true},
                                      {3, 3, true},  {2, 3, true}, {3, 2, true},  {4, 3, true}, {3, 4, true}};

// One workgroup per compute unit at most, and K long enough: two groups of four wavefronts with a ring each multiply the tile
// over every other chunk of K, so that each SIMD has two wavefronts, one issuing while the other waits, and are summed at the
// end through LDS (1.4 us, and twice the first loads). 128x128 tiles, and 64x128 ones of an int4 rhs: bf16 512 x 5008 x 4000
// 31.0 -> 26.8 us, 1504^2 x 3008 24.4 -> 21.3, 784 x 4112 x 4096 in 8x8x4 tiles 32.4 -> 30.4, 2048^2 x 3712 34.0 -> 32.3, x
// 6144 53.3 -> 49.7; int8 8x8x8 3064 x 944 x 5232 23.7 -> 20.9; int4 576 x 5104 x 4704 21.6 -> 20.1, 256 x 8192 x 8192 25.9 ->
// 24.3. The fewer tiles there are the less K it takes, the clock being higher. 16-bit: 1 to 6 % slower at 24 to 35 chunks of K,
// 3 to 6 % faster at 40 to 50 with up to 220 tiles; with 231 of them up to 5 % slower at 64 and 2.5 % faster at 80, with 256 up
// to 4 % slower at 96 and 1.5 to 4 % faster at 112. (With row pieces of 16 and 32 bytes and four rows a tile or more 200 to 248
// tiles of 64 chunks and more go to mmt4d_wave_tile.hip before this is asked.) int8 and the 128x128 tile of int4: 3 to 8 %
// faster from 42 chunks on with up to 170 tiles, 11 % at 82 with 192; 2 % slower at 64 with 231, 1 to 3 % faster at 96 with
// 256. int4 64x128: level at 36 to 48, 4 to 9 % faster at 54 with 140 tiles, 1 to 4 % at 64 with 256.
// (2-byte pieces: pairs of fragments, which a group's half does not have whole. f32 is bound by the matrix pipe. Operands from
// HBM: a ring of ten stages is as fast or faster, 784 x 4112 x 8192 60.2 and 62.8, see streams_operands.)
inline bool two_groups(const MfmaArgs& m, int kind, bool rhs_i4, int gather, bool direct, const TileChoice& t) {
  if (!direct || gather == 2 || kind == kF32 || t.bn != 2 || t.am != (rhs_i4 && t.am == 1 ? 1 : 2)) return false;
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  const int64_t tiles = ((rows + 64 * t.am - 1) / (64 * t.am)) * ((cols + 127) / 128);
  if (tiles > 256 || m.chunks < 44 || comes_from_hbm((rows * m.lhs_rb + cols * m.rhs_rb) * m.K)) return false;
  if (t.am == 1) return 2 * (int64_t)m.chunks >= tiles - 128;
  return kind == kI8 ? 10 * (int64_t)m.chunks >= 7 * (tiles - 100) : 2 * (int64_t)m.chunks >= tiles - 32;
}

// The tile that a problem takes: the least time for 64 bytes of K per row over all of its workgroups, from the time that
// one workgroup per compute unit takes and, where two fit a compute unit (LDS: up to 128x192), two beside each other; less
// with two groups of wavefronts (two_groups).
// Microseconds on the direct-to-LDS kernel, fitted to 24 shapes (M 160..4096, N 464..13952, K 700..8192) with every tile
// for bf16 / f16 16x16x16, bf16 8x8x4, int8 8x8x4 and 16x16x64, f16 16x16x1 and int8 16x16x2 (2-byte pieces: fragments
// come in pairs, which an odd number of them does not have), int4 16x16x32. Over 200 problems of those ranges, timed since the
// loops got shorter, the tile picked is slower than the best one in the mean by 0.3 to 0.5 % (16-bit), 0.1 to 0.6 (int8), 1.6
// (int4) and, of 2-byte pieces, 0.2 (int8) and 2.5 (f16: 464 x 1792 x 8041 60.3 us in 64x64 tiles, 54.3 in 128x64); without
// the 192-wide ones and one efficiency per tile it was 4 to 7 %. f32 is bound by the
// matrix pipe whatever the tile, which leaves the number of rounds (in units of a 128x128 tile; the large tiles, which
// move fewer bytes, are favoured by 10 %).
// `us_per_chunk`: that least time.
inline int choose_tile(const MfmaArgs& m, int kind, bool rhs_i4, int gather, bool direct, double* us_per_chunk) {
  constexpr int kCount = sizeof kBlockTiles / sizeof kBlockTiles[0];
  // Per class of operands and tile, 0: no such instantiation.
  enum { kSixteenBit, kInt8, kTwoBytePieces, kInt4, kFloat32 };
  static const float kOne[][kCount] = {{.51f, .33f, .222f, .148f, .129f, 0, .342f, .25f, .25f, .40f, .405f},
                                       {.50f, .35f, .249f, .170f, .125f, 0, .352f, .28f, .28f, .40f, .405f},
                                       {.61f, .40f, .285f, .251f, .25f, 0, 0, 0, 0, .52f, .523f},
                                       {.62f, .324f, .237f, 0, .129f, .172f, 0, 0, .26f, 0, 0},
                                       {3.45f, 1.87f, 1.0f, .53f, .27f, 0, 0, 0, 0, 0, 0}};
  static const float kTwo[][kCount] = {{0, 0, .345f, .31f, .195f, 0, 0, .43f, .43f}, {0, 0, .44f, .345f, .23f, 0, 0, .41f, .41f},
                                       {0, 0, .48f, .52f, .35f},
                                       {0, 0, .345f, 0, .195f, .263f}, {0, 0, 2.0f, 1.06f, .54f}};
  const int what = kind == kF32 ? kFloat32 : rhs_i4 ? kInt4 : gather == 2 ? kTwoBytePieces : kind == kI8 ? kInt8 : kSixteenBit;
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  int best = -1;
  double best_cost = 0;
  for (int i = 0; i < kCount; ++i) {
    const TileChoice& t = kBlockTiles[i];
    if (kOne[what][i] == 0 || (t.direct_only && !direct)) continue;
    if (gather == 1 && (t.am == 3 || t.bn == 3)) continue;
    // The int4 64x64 tile exists only register-staged, at less than half the
    // rate of the direct 64x128 one on the same problem.
    if (rhs_i4 && direct && t.am == 1 && t.bn == 1) continue;
    const int64_t br = 64 * t.am, bc = 64 * t.bn;
    const int64_t rounds = (((rows + br - 1) / br) * ((cols + bc - 1) / bc) + 255) / 256;
    const double one = kOne[what][i], two = kTwo[what][i];
    double cost = two > 0 ? (rounds & 1) * one + (rounds >> 1) * two : rounds * one;
    if (two_groups(m, kind, rhs_i4, gather, direct, t))
      cost = t.am == 1 ? .84 * one + 1.0 / m.chunks : .78 * one + 1.4 / m.chunks;
    if (best < 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  *us_per_chunk = best_cost;
  return best;
}

#ifdef UK_MFMA_KERNEL_BODIES
namespace {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v16i32 __attribute__((ext_vector_type(16)));
typedef float v16f32 __attribute__((ext_vector_type(16)));
typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf16 __attribute__((ext_vector_type(8)));

template <int KIND>
struct AccType { typedef v16i32 type; typedef int scalar; };
template <> struct AccType<kF16> { typedef v16f32 type; typedef float scalar; };
template <> struct AccType<kBF16> { typedef v16f32 type; typedef float scalar; };
template <> struct AccType<kF32> { typedef v16f32 type; typedef float scalar; };

// MFMAs that one pair of 16-byte operand fragments feeds: f32 has only the
// 32x32x2 shape (one float per lane), so its 4 floats take 4 instructions.
template <int KIND> struct SubSteps { static constexpr int value = KIND == kF32 ? 4 : 1; };

// Sub-step `sub` (< SubSteps<KIND>::value) of the product of two 16-byte
// operand fragments.
template <int KIND>
__device__ __forceinline__ typename AccType<KIND>::type mfma(uint4 row_operand, uint4 col_operand,
                                                             typename AccType<KIND>::type acc, int sub = 0) {
  if constexpr (KIND == kI8) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(v4i32, row_operand),
                                                 __builtin_bit_cast(v4i32, col_operand), acc, 0, 0, 0);
  } else if constexpr (KIND == kF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8f16, row_operand),
                                                  __builtin_bit_cast(v8f16, col_operand), acc, 0, 0, 0);
  } else if constexpr (KIND == kBF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf16, row_operand),
                                                   __builtin_bit_cast(v8bf16, col_operand), acc, 0, 0, 0);
  } else {
    const uint32_t r = sub == 0 ? row_operand.x : sub == 1 ? row_operand.y : sub == 2 ? row_operand.z : row_operand.w;
    const uint32_t c = sub == 0 ? col_operand.x : sub == 1 ? col_operand.y : sub == 2 ? col_operand.z : col_operand.w;
    return __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(r), __uint_as_float(c), acc, 0, 0, 0);
  }
}

// All sub-steps of one fragment pair.
template <int KIND>
__device__ __forceinline__ typename AccType<KIND>::type mfma_all(uint4 row_operand, uint4 col_operand,
                                                                 typename AccType<KIND>::type acc) {
#pragma unroll
  for (int sub = 0; sub < SubSteps<KIND>::value; ++sub) acc = mfma<KIND>(row_operand, col_operand, acc, sub);
  return acc;
}

// 16 int4 values (two dwords, element 2b in the low nibble of byte b) to 16
// int8 values equal to 16x the signed nibbles, in element order: the even and
// the odd elements of a dword are isolated in the high nibbles of two dwords,
// whose bytes are then interleaved.
__device__ __forceinline__ uint4 widen_i4_times16(uint2 w) {
  const uint32_t even0 = (w.x << 4) & 0xF0F0F0F0u, odd0 = w.x & 0xF0F0F0F0u;
  const uint32_t even1 = (w.y << 4) & 0xF0F0F0F0u, odd1 = w.y & 0xF0F0F0F0u;
  uint4 r;
  r.x = __builtin_amdgcn_perm(odd0, even0, 0x05010400u);
  r.y = __builtin_amdgcn_perm(odd0, even0, 0x07030602u);
  r.z = __builtin_amdgcn_perm(odd1, even1, 0x05010400u);
  r.w = __builtin_amdgcn_perm(odd1, even1, 0x07030602u);
  return r;
}

// k step (relative to its chunk's first) that the 16-byte column `c` of an
// operand row starts at.
template <int G, bool I4>
__device__ __forceinline__ int32_t piece_kstep(int c, int32_t log2_rb) {
  if constexpr (I4) return (8 * c) >> log2_rb;
  if constexpr (G == 16) return (16 * c) >> log2_rb;
  return 4 * c;
}

// One 16-byte operand piece for LDS. `p` points at the piece's first byte for
// the current chunk. G is the contiguous run in memory: 16 (one vector load),
// 4 (gather one dword from each of 4 consecutive k steps, `kstep` bytes apart)
// or, for I4, 8 bytes of nibbles widened to 16. With CHECKED, parts whose k
// step `k1 (+d)` is not below K read as zero.
template <int G, bool I4, bool CHECKED>
__device__ __forceinline__ uint4 load_piece(const uint8_t* p, int64_t kstep, int32_t k1, int32_t K) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if constexpr (I4) {
    if (!CHECKED || k1 < K) v = widen_i4_times16(*(const uint2*)p);
  } else if constexpr (G == 16) {
    if (!CHECKED || k1 < K) v = *(const uint4*)p;
  } else {
    if (!CHECKED || k1 + 0 < K) v.x = *(const uint32_t*)(p);
    if (!CHECKED || k1 + 1 < K) v.y = *(const uint32_t*)(p + kstep);
    if (!CHECKED || k1 + 2 < K) v.z = *(const uint32_t*)(p + 2 * kstep);
    if (!CHECKED || k1 + 3 < K) v.w = *(const uint32_t*)(p + 3 * kstep);
  }
  return v;
}

// Workgroup -> block tile. Consecutive workgroup ids go to different XCDs (8 of
// them, each with its own L2), so ids are first regrouped so that one XCD works
// on a contiguous range of tiles, then that range is walked in bands of 4 tile
// rows so that neighbours share lhs and rhs panels. False: nothing to do.
__device__ __forceinline__ bool locate_block(const MfmaArgs& a, int* tile_row, int* tile_col) {
  const uint32_t total_tiles = (uint32_t)a.tile_rows * a.tile_cols;
  const uint32_t per_xcd = (total_tiles + 7) >> 3;
  const uint32_t linear = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (linear >= total_tiles) return false;
  tile_of_number(linear, (uint32_t)a.tile_rows, (uint32_t)a.tile_cols, a.band_reciprocal, tile_row, tile_col);
  return true;
}

// What runs in front of a workgroup's first load counts on every launch. The kernel arguments lie in two cache lines that
// nothing has fetched yet, 560 cycles away: needed here together they are fetched together, where as their uses came up the
// second line was fetched behind the first. An instruction takes 4 to 5 cycles, branches to code not yet fetched more. With
// this, tile_of_number, offsets in 32 bits and no branches, 160 to 220 instructions are left of 230 to 320, and a launch is
// 0.3 to 0.45 us shorter: int8 8x8x4 1024^3 5.39 -> 4.99 us, 1024 x 2048 x 512 5.8 -> 5.44, f32 256 x 512 x 512 3.69 -> 3.27,
// bf16 64 x 4096 x 4096 8.25 -> 7.91, int4 512 x 11008 x 4096 30.2 -> 29.9.
__device__ __forceinline__ void fetch_arguments(const MfmaArgs& a) {
  asm volatile("" ::"s"(a.lhs), "s"(a.rhs), "s"(a.lhs_stride_bytes), "s"(a.rhs_stride_bytes), "s"(a.M), "s"(a.N), "s"(a.K),
               "s"(a.log2_M0), "s"(a.log2_N0), "s"(a.lhs_rb), "s"(a.rhs_rb), "s"(a.log2_lhs_rb), "s"(a.log2_rhs_rb),
               "s"(a.chunks), "s"(a.tile_rows), "s"(a.tile_cols), "s"(a.band_reciprocal));
  __builtin_amdgcn_sched_barrier(0);
}

// Whether a kernel is for calls that accumulate, for those that do not, or finds out at run time. Apart, a call that does not
// accumulate has none of the registers and instructions of the other kind: with both in one kernel and the destination read ahead (see
// store_block), plain calls of a 32-bit output were 0.5 % slower over 250 problems, 256x256 tiles 2 to 3 (32 register moves a step
// for want of registers), int4 256x128 ones 14 where one workgroup fitted a unit instead of two (3744 x 6032 x 768 29.3 -> 33.4
// us, apart 29.3). Apart they are 0.3 to 1.3 % faster than with one kernel that asks for every fragment, 320 problems.
enum Accumulate { kNever, kAlways, kAsked };

// Writes one wavefront's accumulators. Lane l holds, for fragment (i, j): lhs
// row 32*i + (l & 31) and, in accumulator registers 4*q .. 4*q+3, rhs rows
// 32*j + 8*q + 4*(l >> 5) + {0..3} of the wavefront's sub-block, which starts at
// (wave_row, wave_col) of the logical matrix: four consecutive j0 of one output
// row, one 128-bit store (64-bit for a NARROW, i.e. 16-bit, output, rounded to
// nearest even the way common.h:701-770 does).
//
// PAIR_A / PAIR_B: the fragments of that operand were fed in interleaved pairs
// (2-byte row pieces, see the direct-to-LDS kernel): lane row r of fragments
// 2p and 2p + 1 is row 64*p + 2*r resp. 64*p + 2*r + 1 of the sub-block. For
// the columns this means that accumulators e and e + 1 of fragment 2p and of
// fragment 2p + 1 together are four consecutive j0, so two fragments are
// written at a time.
template <int KIND, bool RHS_I4, bool NARROW, int AM, int BN, bool PAIR_A = false, bool PAIR_B = false, int ACCUMULATE = kAsked>
__device__ __forceinline__ void store_block(const MfmaArgs& a, typename AccType<KIND>::type (&acc)[AM][BN],
                                            int64_t wave_row, int64_t wave_col, int lane) {
  typedef typename AccType<KIND>::scalar scalar_t;
  typedef scalar_t quad_t __attribute__((ext_vector_type(4)));
  typedef typename std::conditional<NARROW, uint2, quad_t>::type stored_t;
  constexpr int OUT_BYTES = NARROW ? 2 : 4;
  constexpr int EBITS = KIND == kF16 ? 5 : 8;
  static_assert(!NARROW || KIND == kF16 || KIND == kBF16, "16-bit outputs are floats");
  const int32_t M0 = 1 << a.log2_M0, N0 = 1 << a.log2_N0;
  const int64_t total_rows = (int64_t)a.M << a.log2_M0;
  const int64_t total_cols = (int64_t)a.N << a.log2_N0;
  static_assert((!PAIR_A || AM % 2 == 0) && (!PAIR_B || BN % 2 == 0), "pairs of fragments");
  constexpr int JS = PAIR_B ? 2 : 1;  // rhs fragments written together
  // Byte offset of quad (j, q) from the sub-block's first column tile (the same
  // for every row, and small) and whether the quad lies inside the matrix.
  const int64_t first_col_tile = wave_col >> a.log2_N0;
  uint8_t* wave_out = a.out + OUT_BYTES * (first_col_tile << (a.log2_M0 + a.log2_N0));
  uint32_t col_off[BN][4];
  uint32_t col_inside = 0;
#pragma unroll
  for (int j = 0; j < BN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t col = PAIR_B ? wave_col + 8 * (lane >> 5) + 64 * (j >> 1) + 16 * q + 4 * (j & 1)
                                 : wave_col + 4 * (lane >> 5) + 32 * j + 8 * q;
      col_off[j][q] = (uint32_t)(OUT_BYTES * ((((col >> a.log2_N0) - first_col_tile) << (a.log2_M0 + a.log2_N0)) +
                                              (col & (N0 - 1))));
      if (col < total_cols) col_inside |= 1u << (4 * j + q);
    }
  auto to_float = [](stored_t w) -> quad_t {
    if constexpr (NARROW) {
      return quad_t{widen16_first<EBITS>(w.x), widen16_second<EBITS>(w.x), widen16_first<EBITS>(w.y), widen16_second<EBITS>(w.y)};
    } else {
      return w;
    }
  };
  auto to_stored = [](quad_t v) -> stored_t {
    if constexpr (NARROW) {
      return make_uint2(narrow16_pair<EBITS>(v.x, v.y), narrow16_pair<EBITS>(v.z, v.w));
    } else {
      return v;
    }
  };
  static_assert(ACCUMULATE != kAlways || (!PAIR_A && !PAIR_B), "pairs are for calls of both kinds");
  if constexpr (ACCUMULATE == kAlways) {
    // What the destination holds is asked for ahead of the fragments that it is added to, as much as 16 registers hold. Asked
    // for when a fragment's turn came it was waited for once a fragment, with a 16-bit output, each converted as it
    // arrived, four times: int8 8x8x4 344 x 6576 x 336 8.9 -> 6.8 us, 856 x 4480 x 580 10.9 -> 9.4, bf16 8x8x4 1024 x 4096 x 1024
    // 15.6 -> 13.9, 256x256 tiles 3072 x 5024 x 1264 48.0 -> 46.7, bf16 output 74.8 -> 43.5 (with the conversions of uk_device.h).
    // 32 and 64 registers of it are as fast in small tiles and slower in large ones (int4 192x128 tiles, 13 problems, against
    // none ahead: 1.07 times as fast with 16, 1.04 with 32, 0.99 with 64; 128x128 1.09, 1.06, 1.04). Pairs of fragments, 32 registers
    // at the least, gain nothing from it and are up to 8 % slower.
    // (Without conditions: rows and columns behind the last ones read others of the sub-block.)
    if (wave_row >= total_rows || wave_col >= total_cols) return;
    uint8_t* row_out[AM];
    bool row_inside[AM];
#pragma unroll
    for (int i = 0; i < AM; ++i) {
      const int64_t this_row = wave_row + 32 * i + (lane & 31), row = min(this_row, total_rows - 1);
      row_inside[i] = this_row < total_rows;
      row_out[i] = wave_out + OUT_BYTES * ((row >> a.log2_M0) * a.out_stride0 + ((row & (M0 - 1)) << a.log2_N0));
    }
    constexpr int FIT = 16 / (int)sizeof(stored_t), AHEAD = FIT < AM * BN ? FIT : AM * BN;
    stored_t old[AHEAD][4];
    auto fetch = [&](int f) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t off = col_inside >> (4 * (f % BN) + q) & 1 ? col_off[f % BN][q] : 0;
        old[f % AHEAD][q] = *(const stored_t*)(row_out[f / BN] + off);
      }
    };
#pragma unroll
    for (int f = 0; f < AHEAD; ++f) fetch(f);
#pragma unroll
    for (int f = 0; f < AM * BN; ++f) {
      typename AccType<KIND>::type frag = acc[f / BN][f % BN];
      asm volatile("" : "+a"(frag));  // (pinned until its turn, see below)
      quad_t v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = quad_t{frag[4 * q], frag[4 * q + 1], frag[4 * q + 2], frag[4 * q + 3]};
        if constexpr (RHS_I4) v[q] = v[q] >> 4;
        v[q] += to_float(old[f % AHEAD][q]);
      }
      if (f + AHEAD < AM * BN) fetch(f + AHEAD);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (row_inside[f / BN] && (col_inside >> (4 * (f % BN) + q) & 1))
          *(stored_t*)(row_out[f / BN] + col_off[f % BN][q]) = to_stored(v[q]);
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  // With paired lhs fragments, fragments 2p and 2p + 1 hold the even and the odd
  // rows of the same 64: they are written together, so that the stores which
  // make up a cache line of the output (two rows of a 16-wide int32 tile, say)
  // follow each other directly. Written a fragment at a time, each line was
  // sent to memory in pieces (2.6x the output size in write traffic).
  constexpr int IS = PAIR_A ? 2 : 1;  // lhs fragments written together
#pragma unroll
  for (int i0 = 0; i0 < AM; i0 += IS) {
    bool row_inside[IS];
    uint8_t* row_out[IS];
#pragma unroll
    for (int t = 0; t < IS; ++t) {
      const int i = i0 + t;
      const int64_t this_row =
          wave_row + (PAIR_A ? 64 * (i >> 1) + 2 * (lane & 31) + (i & 1) : 32 * i + (lane & 31));
      const int64_t row = min(this_row, total_rows - 1);
      row_inside[t] = this_row < total_rows;
      row_out[t] = wave_out + OUT_BYTES * ((row >> a.log2_M0) * a.out_stride0 + ((row & (M0 - 1)) << a.log2_N0));
    }
#pragma unroll
    for (int j0 = 0; j0 < BN; j0 += JS) {
      // Pin the fragment(s) where they are until their turn: left alone, the
      // compiler moves all 256 accumulators to ordinary registers right after
      // the main loop, and there are not that many.
      typename AccType<KIND>::type frag[IS][JS];
#pragma unroll
      for (int t = 0; t < IS; ++t)
#pragma unroll
        for (int s = 0; s < JS; ++s) {
          frag[t][s] = acc[i0 + t][j0 + s];
          asm volatile("" : "+a"(frag[t][s]));
        }
      quad_t v[IS][JS][4];
#pragma unroll
      for (int t = 0; t < IS; ++t)
#pragma unroll
        for (int s = 0; s < JS; ++s)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if constexpr (PAIR_B) {
              v[t][s][q] = quad_t{frag[t][0][4 * q + 2 * s], frag[t][1][4 * q + 2 * s], frag[t][0][4 * q + 2 * s + 1],
                                  frag[t][1][4 * q + 2 * s + 1]};
            } else {
              v[t][s][q] = quad_t{frag[t][s][4 * q], frag[t][s][4 * q + 1], frag[t][s][4 * q + 2], frag[t][s][4 * q + 3]};
            }
            if constexpr (RHS_I4) v[t][s][q] = v[t][s][q] >> 4;
          }
      if (ACCUMULATE == kAsked && a.accumulate) {
        stored_t old[IS][JS][4];
#pragma unroll
        for (int t = 0; t < IS; ++t)
#pragma unroll
          for (int s = 0; s < JS; ++s)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              old[t][s][q] = stored_t{};
              if (row_inside[t] && (col_inside >> (4 * (j0 + s) + q) & 1))
                old[t][s][q] = *(const stored_t*)(row_out[t] + col_off[j0 + s][q]);
            }
#pragma unroll
        for (int t = 0; t < IS; ++t)
#pragma unroll
          for (int s = 0; s < JS; ++s)
#pragma unroll
            for (int q = 0; q < 4; ++q) v[t][s][q] += to_float(old[t][s][q]);
      }
      // Store order: the pieces of one row right after each other (with paired
      // rhs fragments v[.][0][q] and v[.][1][q] are the two halves of 32
      // contiguous bytes), then the neighbouring row of the other lhs fragment.
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int t = 0; t < IS; ++t)
#pragma unroll
          for (int s = 0; s < JS; ++s)
            if (row_inside[t] && (col_inside >> (4 * (j0 + s) + q) & 1))
              *(stored_t*)(row_out[t] + col_off[j0 + s][q]) = to_stored(v[t][s][q]);
      // Keep the fragments apart: hoisting all address arithmetic and
      // accumulator reads to the top costs more registers than there are.
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int KIND, bool RHS_I4, bool NARROW, int G, int AM, int BN, int MIN_BLOCKS, bool TAIL>
__global__ __launch_bounds__(256, MIN_BLOCKS) void mmt4d_mfma_kernel(const MfmaArgs a) {
  typedef typename AccType<KIND>::type acc_t;
  constexpr int BLOCK_ROWS = 64 * AM;  // lhs rows per workgroup
  constexpr int BLOCK_COLS = 64 * BN;  // rhs rows per workgroup
  constexpr int A_PIECES = BLOCK_ROWS * 4;  // 16-byte pieces per chunk
  constexpr int B_PIECES = BLOCK_COLS * 4;
  constexpr int A_PER_THREAD = (A_PIECES + 255) / 256;
  constexpr int B_PER_THREAD = (B_PIECES + 255) / 256;
  static_assert(A_PIECES % 256 == 0 && B_PIECES % 256 == 0, "block tile too small");
  __shared__ uint4 lds_a[2][A_PIECES];
  __shared__ uint4 lds_b[2][B_PIECES];

  int tile_row, tile_col;
  if (!locate_block(a, &tile_row, &tile_col)) return;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wave_m = wave >> 1, wave_n = wave & 1;

  const int32_t M0 = 1 << a.log2_M0, N0 = 1 << a.log2_N0;
  const int64_t total_rows = (int64_t)a.M << a.log2_M0;
  const int64_t total_cols = (int64_t)a.N << a.log2_N0;
  const int64_t lhs_kstep = (int64_t)a.lhs_rb << a.log2_M0;
  const int64_t rhs_kstep = (int64_t)a.rhs_rb << a.log2_N0;
  // k steps covered by one chunk (64 bytes of an lhs row).
  const int32_t ksteps_per_chunk = 64 >> a.log2_lhs_rb;

  // Workgroup-uniform bases and 32-bit per-piece offsets from them. Piece
  // p = tid + 256*s lands at LDS slot p: fragment (p >> 7), 16-byte column
  // (p >> 5) & 3, row p & 31 of the fragment (column c is K-step c >> 1, lane
  // half c & 1 of the MFMA operand). Rows past the end of the matrix
  // are redirected to its last row: their products are computed, never stored.
  const int64_t first_row = (int64_t)tile_row * BLOCK_ROWS;
  const int64_t first_col = (int64_t)tile_col * BLOCK_COLS;
  const uint8_t* lhs_base = a.lhs + (first_row >> a.log2_M0) * a.lhs_stride_bytes;
  const uint8_t* rhs_base = a.rhs + (first_col >> a.log2_N0) * a.rhs_stride_bytes;
  uint32_t a_off[A_PER_THREAD], b_off[B_PER_THREAD];
#pragma unroll
  for (int s = 0; s < A_PER_THREAD; ++s) {
    const int p = tid + 256 * s;
    const int c = (p >> 5) & 3;
    const int64_t row = min(first_row + (p >> 7) * 32 + (p & 31), total_rows - 1);
    const int64_t tile = (row >> a.log2_M0) - (first_row >> a.log2_M0);
    const int32_t col_byte = G == 16 ? 16 * c : 0;
    const int32_t k1 = piece_kstep<G, false>(c, a.log2_lhs_rb);
    a_off[s] = (uint32_t)(tile * a.lhs_stride_bytes + (row & (M0 - 1)) * a.lhs_rb +
                          k1 * lhs_kstep + (col_byte & (a.lhs_rb - 1)));
  }
#pragma unroll
  for (int s = 0; s < B_PER_THREAD; ++s) {
    const int p = tid + 256 * s;
    const int c = (p >> 5) & 3;
    const int64_t row = min(first_col + (p >> 7) * 32 + (p & 31), total_cols - 1);
    const int64_t tile = (row >> a.log2_N0) - (first_col >> a.log2_N0);
    const int32_t col_byte = RHS_I4 ? 8 * c : (G == 16 ? 16 * c : 0);
    const int32_t k1 = piece_kstep<G, RHS_I4>(c, a.log2_rhs_rb);
    b_off[s] = (uint32_t)(tile * a.rhs_stride_bytes + (row & (N0 - 1)) * a.rhs_rb +
                          k1 * rhs_kstep + (col_byte & (a.rhs_rb - 1)));
  }

  acc_t acc[AM][BN];
#pragma unroll
  for (int i = 0; i < AM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

  // Global -> register prefetch of one chunk, two chunks deep: while chunk kc
  // is multiplied, chunk kc + 1 moves from registers to LDS and chunks kc + 2
  // and kc + 3 are in flight from memory (a load takes longer than one chunk
  // of MFMAs, so a single chunk of lookahead would stall every iteration).
  uint4 a_pre[2][A_PER_THREAD], b_pre[2][B_PER_THREAD];
  auto fetch = [&](int kc, uint4* a_next, uint4* b_next) {
    const int32_t k1_0 = kc * ksteps_per_chunk;
    const uint8_t* la = lhs_base + (int64_t)k1_0 * lhs_kstep;
    const uint8_t* lb = rhs_base + (int64_t)k1_0 * rhs_kstep;
#pragma unroll
    for (int s = 0; s < A_PER_THREAD; ++s)
      a_next[s] = load_piece<G, false, false>(la + a_off[s], lhs_kstep, 0, 0);
#pragma unroll
    for (int s = 0; s < B_PER_THREAD; ++s)
      b_next[s] = load_piece<G, RHS_I4, false>(lb + b_off[s], rhs_kstep, 0, 0);
  };
  // Same for a chunk that K ends inside of: missing k steps read as zero.
  auto fetch_checked = [&](int kc, uint4* a_next, uint4* b_next) {
    const int32_t k1_0 = kc * ksteps_per_chunk;
    const uint8_t* la = lhs_base + (int64_t)k1_0 * lhs_kstep;
    const uint8_t* lb = rhs_base + (int64_t)k1_0 * rhs_kstep;
#pragma unroll
    for (int s = 0; s < A_PER_THREAD; ++s)
      a_next[s] = load_piece<G, false, true>(
          la + a_off[s], lhs_kstep,
          k1_0 + piece_kstep<G, false>(((tid + 256 * s) >> 5) & 3, a.log2_lhs_rb), a.K);
#pragma unroll
    for (int s = 0; s < B_PER_THREAD; ++s)
      b_next[s] = load_piece<G, RHS_I4, true>(
          lb + b_off[s], rhs_kstep,
          k1_0 + piece_kstep<G, RHS_I4>(((tid + 256 * s) >> 5) & 3, a.log2_rhs_rb), a.K);
  };
  auto stash = [&](int stage, const uint4* a_next, const uint4* b_next) {
#pragma unroll
    for (int s = 0; s < A_PER_THREAD; ++s) lds_a[stage][tid + 256 * s] = a_next[s];
#pragma unroll
    for (int s = 0; s < B_PER_THREAD; ++s) lds_b[stage][tid + 256 * s] = b_next[s];
  };

  // Fragment registers, double buffered: while the MFMAs of chunk kc run from
  // one set, the fragments of chunk kc + 1 are read from LDS into the other.
  // The loop is unrolled by two so the sets swap roles without copies, and its
  // body is branch-free (the prefetch index is clamped instead) so that LDS
  // reads, global loads and MFMAs can be scheduled against each other.
  uint4 pa[AM][2], pb[BN][2], qa[AM][2], qb[BN][2];
  auto read_frags = [&](int stage, uint4 (*fa)[2], uint4 (*fb)[2]) {
    const uint4* frag_a = &lds_a[stage][(wave_m * AM) * 128 + lane];
    const uint4* frag_b = &lds_b[stage][(wave_n * BN) * 128 + lane];
    // K-step 0 first: it is what the next step's first MFMAs consume.
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int j = 0; j < BN; ++j) fb[j][kk] = frag_b[j * 128 + kk * 64];
#pragma unroll
      for (int i = 0; i < AM; ++i) fa[i][kk] = frag_a[i * 128 + kk * 64];
    }
  };
  auto multiply = [&](const uint4 (*fa)[2], const uint4 (*fb)[2], int kk) {
#pragma unroll
    for (int i = 0; i < AM; ++i)
#pragma unroll
      for (int j = 0; j < BN; ++j) acc[i][j] = mfma_all<KIND>(fb[j][kk], fa[i][kk], acc[i][j]);
  };
  // Chunks that lie entirely inside K run through the pipeline; a trailing
  // partial chunk is handled after it, unpipelined.
  const int full_chunks = a.K / ksteps_per_chunk;
  const int last_chunk = full_chunks - 1;
  // One pipeline step for chunk kc, whose fragments are in `cur`:
  //   registers(kc + 1) -> LDS stage, first half of the MFMAs (covers the LDS
  //   write latency), barrier, global loads of chunk kc + 3 into the register
  //   set just freed, LDS reads of the fragments of chunk kc + 1, second half
  //   of the MFMAs (covers the LDS read latency). Prefetch indices are clamped
  //   to the last full chunk, so the body is branch-free.
  auto step = [&](int kc, int stage, const uint4 (*cur_a)[2], const uint4 (*cur_b)[2],
                  uint4 (*nxt_a)[2], uint4 (*nxt_b)[2]) {
    // A wavefront issues in order, so memory instructions only overlap with
    // the matrix pipe if they sit between MFMAs in program order: the two
    // halves below are interleaved one MFMA at a time with the LDS writes and
    // global loads (first half) and with the LDS reads (second half).
    constexpr int MFMAS = AM * BN;  // per half
    constexpr int WRITES = A_PER_THREAD + B_PER_THREAD;
    constexpr int LOADS = (G == 4 ? 4 : 1) * A_PER_THREAD + ((G == 4 && !RHS_I4) ? 4 : 1) * B_PER_THREAD;
    constexpr int READS = 2 * (AM + BN);
    stash(stage, a_pre[stage], b_pre[stage]);
    fetch(min(kc + 3, last_chunk), a_pre[stage], b_pre[stage]);
    multiply(cur_a, cur_b, 0);
#pragma unroll
    for (int m = 0; m < MFMAS; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      if (m < WRITES) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // one LDS write
      constexpr int LOADS_PER = (LOADS + MFMAS - 1) / MFMAS;
      if (m * LOADS_PER < LOADS) {
        __builtin_amdgcn_sched_group_barrier(0x002, 2 * LOADS_PER, 0);  // address arithmetic
        __builtin_amdgcn_sched_group_barrier(0x020, LOADS_PER, 0);      // global loads
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    read_frags(stage, nxt_a, nxt_b);
    multiply(cur_a, cur_b, 1);
#pragma unroll
    for (int m = 0; m < MFMAS; ++m) {
      constexpr int READS_PER = (READS + MFMAS - 1) / MFMAS;
      if (m * READS_PER < READS) __builtin_amdgcn_sched_group_barrier(0x100, READS_PER, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  if (full_chunks > 0) {
    // Chunk c travels through register set c & 1 and LDS stage c & 1.
    fetch(0, a_pre[0], b_pre[0]);
    fetch(min(1, last_chunk), a_pre[1], b_pre[1]);
    stash(0, a_pre[0], b_pre[0]);
    fetch(min(2, last_chunk), a_pre[0], b_pre[0]);
    __syncthreads();
    read_frags(0, pa, pb);
    int kc = 0;
    for (; kc + 1 < full_chunks; kc += 2) {
      step(kc, 1, pa, pb, qa, qb);
      step(kc + 1, 0, qa, qb, pa, pb);
    }
    if (kc < full_chunks) {
      multiply(pa, pb, 0);
      multiply(pa, pb, 1);
    }
  }
  if constexpr (TAIL) {
    fetch_checked(full_chunks, a_pre[0], b_pre[0]);
    __syncthreads();  // every wavefront is done reading LDS stage 0
    stash(0, a_pre[0], b_pre[0]);
    __syncthreads();
    read_frags(0, pa, pb);
    multiply(pa, pb, 0);
    multiply(pa, pb, 1);
  }

  store_block<KIND, RHS_I4, NARROW, AM, BN>(a, acc, first_row + wave_m * (32 * AM),
                                            first_col + wave_n * (32 * BN), lane);
}

// ---------------------------------------------------------------------------
// Direct-to-LDS variant: the same block tiling, but operand pieces travel
// global memory -> LDS without passing through registers
// (global_load_lds_dwordx4: lane l of a wavefront writes its 16 bytes at
// M0 + 16*l), through a ring of 4 LDS stages filled three chunks ahead of the
// MFMAs. It needs no register prefetch buffers, no LDS writes and no
// data-dependent waits other than one counter wait per chunk. (direct_covers
// says what it takes; everything else uses the kernel above.)
//
// Every load moves 16 contiguous bytes per lane, also for the 4-byte row
// pieces of e.g. the 8x8x4 int8 tiles (G == 4), where 16 contiguous bytes are
// 4 consecutive rows of one k step: there the transposition to "one row, 16
// bytes of K" happens on the way out of LDS, with four 32-bit reads per
// fragment instead of one 128-bit read, and the loads are arranged so that
// those reads are linear in the lane number (conflict-free).
//
// A wavefront alone on its SIMD issues an instruction every four to six cycles, and a step of the smaller tiles takes as long
// as its instructions: 46 for 4 MFMAs on the 128x64 tile (57 before the first chunk took what is odd about K, see below, and
// loads came in pairs). bf16 512 x 4096 x 4096 23.0 -> 21.6 us, 304 x 5008 x 3008 16.4 -> 15.5, int8 8x8x4 512 x 4096 x 4096
// 13.7 -> 12.9; int4 512 x 11008 x 4096 (256x128) 29.2 -> 27.4, 784 x 4112 x 4096 (128x128) 21.5 -> 20.1; 192-wide tiles 2
// to 5 %, 256x256 up to 2 % (2-byte pieces: int8 16x16x2 3072 x 4096 x 4096 57.4 -> 56.1, 4096^2 x 4094 69.8 -> 69.5, but with all
// units busy and K a power of two 1.4 to 1.7 % slower: 4096^3 69.1 -> 70.3, x 2048 44.1 -> 44.7).
//
// The loads are issued from inline assembly: the compiler cannot see that they
// write LDS, so it does not serialise the LDS reads against them; ordering is
// enforced by hand with s_waitcnt vmcnt + a workgroup barrier once per chunk.
extern __shared__ uint4 ring[];

// Measuring aid, compiled in only by the benchmark's probe library (csrc/bench/probe_mmt4d_timeline.hip):
// wavefront 0 of each of the first 256 workgroups leaves five readings of the constant-rate 100 MHz
// counter (start, main loop begins, main loop ends, last MFMA issued, stores acknowledged).
#ifdef UK_KERNEL_TIMELINE
#define UK_TIMELINE(...) __VA_ARGS__
__device__ unsigned long long uk_timeline[256 * 8];
#else
#define UK_TIMELINE(...)
#endif

// One wavefront-wide load of 64 x 16 bytes to LDS byte offset `lds_off` + FURTHER (wavefront-uniform) from `base`
// (uniform) + per-lane byte offset `voff`.
template <uint32_t FURTHER = 0>
__device__ __forceinline__ void load_to_lds(uint32_t lds_off, uint32_t voff, const uint8_t* base) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_off), "v"(voff), "s"(base), "n"(FURTHER)
               : "memory", "scc");
}
// Two, the second to LDS 1 KiB further on. The instruction's offset is added to both addresses: the caller has taken the
// 1 KiB off `voff1`.
template <uint32_t FURTHER>
__device__ __forceinline__ void load_two_to_lds(uint32_t lds_off, uint32_t voff0, uint32_t voff1, const uint8_t* base) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024"
               :
               : "s"(lds_off), "v"(voff0), "v"(voff1), "s"(base), "n"(FURTHER)
               : "memory", "scc");
}

// 8 bytes per lane from LDS, transposed within each group of 16 lanes
// (ds_read_b64_tr_b8): the 16 lanes' 8-byte chunks are taken as 8 rows of 16
// bytes (chunks 2j and 2j + 1 make row j), and lane i of the group receives
// byte i of every row. With a k-major operand ("16 matrix rows at k, then the
// same rows at k + 1, ...") lane i thus gets 8 consecutive k of matrix row i.
__device__ __forceinline__ uint2 lds_read_transposed(const uint8_t* p) {
  typedef int v2i32 __attribute__((ext_vector_type(2)));
  const v2i32 v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i32*)(p));
  return make_uint2((uint32_t)v.x, (uint32_t)v.y);
}

// A wavefront-uniform pointer, said to be so: the loads above take their base from scalar registers, and whether
// the compiler keeps a uniform 64-bit address computation on the scalar unit depends on what else uses its inputs.
__device__ __forceinline__ const uint8_t* uniform_pointer(const uint8_t* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const uint8_t*)(((uint64_t)hi << 32) | lo);
}

// (Overloads on scalars rather than a bit cast of a vector element.)
__device__ __forceinline__ uint32_t value_bits(int32_t v) { return (uint32_t)v; }
__device__ __forceinline__ uint32_t value_bits(float v) { return __float_as_uint(v); }
__device__ __forceinline__ void set_from_bits(int32_t& v, uint32_t bits) { v = (int32_t)bits; }
__device__ __forceinline__ void set_from_bits(float& v, uint32_t bits) { v = __uint_as_float(bits); }

// What a step of the kernel below takes its place from.
template <typename Read, typename Load, typename Advance>
struct StepPlace {
  Read read_from;
  Load load;
  Advance advance;
};

// f(0), .. f(N - 1), each number a type of its own.
template <int N, typename F>
__device__ __forceinline__ void each_of(F f) {
  if constexpr (N > 0) {
    each_of<N - 1>(f);
    f(std::integral_constant<int, N - 1>());
  }
}

template <int N>
__device__ __forceinline__ void wait_loads_but() {
  static_assert(N >= 0 && N <= 63, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// (The 256x256 tile needs all 512 registers of a lane for one wavefront; said
// explicitly, because left to its occupancy heuristics the compiler may keep
// the accumulators in scratch memory instead.)
// STAGGER: 0 = every accumulator stored after the last MFMA; 1 = staggered tail (see below); 2 = the same for
// an accumulating call, the destination read in the tail; 3 = accumulating call with the destination read and
// added during the main loop (needs enough steps), tail as in 1.
template <int KIND, bool RHS_I4, bool NARROW, int G, int AM, int BN, int STAGES, int STAGGER = 0, int GROUPS = 1, int ACCUMULATE = kAsked>
__global__ __launch_bounds__(256 * GROUPS) __attribute__((amdgpu_waves_per_eu(GROUPS, AM * BN >= 9 ? 1 : (AM * BN >= 4 ? 2 : 4))))
void mmt4d_mfma_direct_kernel(const MfmaArgs a) {
  typedef typename AccType<KIND>::type acc_t;
  static_assert(!RHS_I4 || (G == 16 && BN >= 2), "int4 rhs: 16-byte pieces, at least one fragment per wavefront");
  constexpr int BLOCK_ROWS = 64 * AM, BLOCK_COLS = 64 * BN;
  // 16-byte pieces per chunk: 64 bytes of K per row, 32 bytes for an int4 rhs.
  constexpr int A_PIECES = BLOCK_ROWS * 4, B_PIECES = BLOCK_COLS * (RHS_I4 ? 2 : 4);
  constexpr int STAGE_PIECES = A_PIECES + B_PIECES;
  constexpr int AHEAD = STAGES - 1;  // chunks in flight ahead of the one being multiplied
  static_assert(STAGES >= 4, "ring depth");
  // 2-byte row pieces: an operand with an even number of fragments per
  // wavefront is fed in interleaved pairs of fragments (see the layouts below).
  constexpr bool PAIR_A = G == 2 && AM % 2 == 0, PAIR_B = G == 2 && BN % 2 == 0;
  // Load instructions per wavefront and chunk (64 lanes x 16 bytes each), each
  // with its own per-lane offset.
  constexpr int A_LOADS = A_PIECES / 256, B_LOADS = B_PIECES / 256;
  constexpr int LOADS = A_LOADS + B_LOADS;
  static_assert(A_PIECES % 256 == 0 && B_PIECES % 256 == 0, "block tile too small");
  static_assert((AHEAD - 1) * LOADS <= 63, "the loads in flight must fit the 6-bit counter");

  UK_TIMELINE(const unsigned long long tl_start = __builtin_amdgcn_s_memrealtime(); unsigned long long tl_loop = 0,
              tl_loop_end = 0;)
  fetch_arguments(a);
  int tile_row, tile_col;
  if (!locate_block(a, &tile_row, &tile_col)) return;

  const int lane = threadIdx.x & 63;
  const int wave_of_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = GROUPS == 1 ? 0 : wave_of_all >> 2, wave = GROUPS == 1 ? wave_of_all : wave_of_all & 3;
  const int wave_m = wave >> 1, wave_n = wave & 1;

  const int64_t total_rows = (int64_t)a.M << a.log2_M0;
  const int64_t total_cols = (int64_t)a.N << a.log2_N0;
  // Bytes of a k step and of a chunk.
  const int log2_lhs_kstep = a.log2_lhs_rb + a.log2_M0, log2_rhs_kstep = a.log2_rhs_rb + a.log2_N0;
  const int32_t lhs_chunk_bytes = 64 << a.log2_M0, rhs_chunk_bytes = (RHS_I4 ? 32 : 64) << a.log2_N0;

  const int64_t first_row = (int64_t)tile_row * BLOCK_ROWS;
  const int64_t first_col = (int64_t)tile_col * BLOCK_COLS;
  const uint8_t* lhs_base = uniform_pointer(a.lhs + (first_row >> a.log2_M0) * a.lhs_stride_bytes);
  const uint8_t* rhs_base = uniform_pointer(a.rhs + (first_col >> a.log2_N0) * a.rhs_stride_bytes);

  // Load t of wavefront w fills the 16-byte LDS slots 64*m .. 64*m + 63 of its
  // operand, lane l the slot 64*m + l; m = 4*t + w or, where an operand's loads are issued together, loads*w + t.
  // Together (one or two of them): on tiles whose steps are as long as their instructions take to issue, 64x64 and
  // 128x64 and those of an int4 rhs up to 128x128, and where the operands come from HBM (ten stages: bf16 384 x 8192 x
  // 4096 29.5 -> 29.1 us, 8x8x4 28.5 -> 28.0). The 128x128 tile of four stages, bound by the LDS, is 1 % faster one by one.
  constexpr bool TOGETHER = AM * BN <= 2 || (AM * BN <= 4 && (RHS_I4 || STAGES == 10));
  auto a_number = [&](int t) { return TOGETHER ? A_LOADS * wave + t : 4 * t + wave; };
  auto b_number = [&](int t) { return TOGETHER ? B_LOADS * wave + t : 4 * t + wave; };
  //   G == 16: slot p holds fragment p >> 7, rows 16*((p >> 6) & 1) + (p & 15),
  //     16-byte column c = (p >> 4) & 3 (K-step c >> 1, lane half c & 1 of the
  //     MFMA operand): one load covers 16 rows x 64 bytes, which for 64-byte row
  //     pieces is 1 KiB of contiguous memory (with "32 rows x 32 bytes" every
  //     cache line was touched by two loads: 7 % slower). Lane 32*h + r reads
  //     slot 128*f + 64*(r >> 4) + 16*(2*kk + h) + (r & 15), one 128-bit read;
  //     every group of 16 lanes reads 256 contiguous bytes: no bank conflicts.
  //     (With an int4 rhs the lhs keeps the older arrangement: slot p holds row
  //     p & 31, column slot (p >> 5) & 3, read at slot 128*f + 64*kk + lane.)
  //   G == 2, 8 (bytes of a row piece; R = 16 / G rows share 16 contiguous
  //     bytes, a chunk is 64 / G k steps): slot 64*m + l holds rows R*g ..
  //     R*g + R - 1 (g = l % (2*G)) of fragment m >> 1 at k step
  //     (32/G)*(m & 1) + (16/G)*h + d of the chunk (h = (l / (2*G)) & 1,
  //     d = l / (4*G)). The G-byte element number 64*((2*f + kk)*(16/G) + d) +
  //     32*h + r of the operand is then row r of fragment f at that k step: the
  //     MFMA operand of lane 32*h + r for K-step kk is elements d = 0 .. 16/G - 1,
  //     each read linear in the lane number (8-byte pieces: two 64-bit reads; 2-byte: eight reads of the dword the
  //     element shares with its neighbour row, and a byte permute that picks
  //     the lane's half). K is permuted inside a chunk, identically for lhs
  //     and rhs.
  //   G == 4 (four rows share 16 contiguous bytes, a chunk is 16 k steps): load m of
  //     an operand holds k steps 8*(m & 1) + 2*d + h of fragment m >> 1, its slot
  //     16*d + s the rows 4*g .. 4*g + 3 at (d, h), where s is
  //       8*h + g                                      M0 = 16 or 4
  //       4*(g >> 1) + ((2*h + (g & 1)) ^ 2*(g >> 2))  M0 = 8,
  //     so that four consecutive lanes load 64 contiguous bytes (M0 = 16: the rows
  //     of one k step, 8: those of two), and the 32 lanes of a half find their
  //     dwords in 32 different banks. Lane 32*h + r reads dword r & 3 of the slots
  //     of g = r >> 2, 256 bytes from one d to the next: two paired dword reads.
  //   G == 2, fragments in pairs (an even number of them per wavefront): 16-bit
  //     reads deliver half of what the LDS can, so a lane reads dwords, i.e. two
  //     adjacent rows of one k step, and gives the low half to fragment 2p, the
  //     high half to fragment 2p + 1: row r of those fragments is row 2*r resp.
  //     2*r + 1 of the pair's 64 rows (the epilogue undoes it). Slot 64*m + l
  //     holds rows 8*g .. 8*g + 7 (g = l & 7) of pair m >> 2 at k step
  //     16*kk + 8*h + 4*(m & 1) + (l >> 4) of the chunk (kk = (m >> 1) & 1,
  //     h = (l >> 3) & 1), the same k steps per (K-step, lane half) as in the
  //     unpaired layout, so the two can be mixed between lhs and rhs. Dword
  //     64*d + 32*h + r of a (pair, K-step) is then rows 2*r, 2*r + 1 at the
  //     lane's d-th k step: eight dword reads linear in the lane number (four
  //     two-address instructions) and eight byte permutes per two fragments.
  //     (These loads touch two stretches of 64 bytes per four lanes with M0 = 16, four with M0 = 8. With one
  //     resp. two, laid out like the 4-byte pieces, nothing is gained, the reads and permutes being what the step waits
  //     for: int8 16x16x2 777 x 4100 x 4096 23.4 us both, 512 x 4096 x 4096 19.7 -> 20.1.)
  //   What the lanes of a load have to do with each other: the memory pipeline takes four of them at a time, and takes
  //   those twice that touch two lines of 128 bytes: 105 bytes a nanosecond and compute unit with one, 70 with two, in a loop
  //   of nothing but these loads. Tiles of up to 128x128 come close to the latter. 4-byte pieces with M0 = 8 and 64-byte
  //   pieces (below) had the rows first: int8 512 x 4096 x 4096 16x16x64 16.2 -> 13.8 us, 8x8x4 15.6 -> 13.6, 777 x 4100 x
  //   4096 22.3 -> 20.1 and 21.0 -> 19.4, 3072^3 (192x192 tiles) 32.2 -> 31.2 and 30.3 -> 29.4; 256x256 tiles are bound by the
  //   matrix pipe, level. Four rows of 32-byte pieces are one line as they are.
  //   int4 rhs: slot 64*f + 32*h + r holds nibbles 32*h .. 32*h + 31 of row r of
  //     fragment f: lane 32*h + r reads that slot once per chunk and widens its
  //     first 8 bytes for K-step 0, its last 8 for K-step 1. The lhs columns are
  //     assigned to match: (K-step kk, lane half h) gets 16-byte column kk + 2*h.
  // Rows past the end of the matrix are redirected to its last row (group):
  // their products are computed, never stored.
  // (In 32 bits, counted from the workgroup's first row, which is the first of a tile: this is code that runs once, in front
  // of the first load.)
  const int32_t rows_left = (int32_t)min(total_rows - first_row, (int64_t)BLOCK_ROWS);
  const int32_t cols_left = (int32_t)min(total_cols - first_col, (int64_t)BLOCK_COLS);
  auto row_offset = [&](int32_t row, int32_t last, int log2_t0, int64_t stride_bytes, int log2_rb) -> uint32_t {
    row = min(row, last);
    return (uint32_t)(row >> log2_t0) * (uint32_t)stride_bytes + ((uint32_t)(row & ((1 << log2_t0) - 1)) << log2_rb);
  };
  //   G == 16, a row's 64 bytes of a chunk contiguous (64-byte row pieces; lhs tiles
  //     one row tall, i.e. a row-major matrix): with the arrangement above four
  //     consecutive lanes would load from four rows. Here lane l of a load takes row
  //     l >> 2 of the load's 16 and the
  //     16-byte column (l & 3) ^ ((l >> 4) & 3), so four consecutive lanes cover
  //     one row's 64 bytes; lane 32*h + r reads slot 128*f + 64*(r >> 4) + 4*r' +
  //     ((2*kk + h) ^ ((r' >> 2) & 3)), r' = r & 15: the xor spreads the sixteen
  //     rows of a group of lanes over all banks. The slot for K-step 1 is the one
  //     for K-step 0 with bit 1 flipped, a per-lane distance (lhs_kk1_step, rhs_kk1_step).
  constexpr bool ROWS16 = G == 16 && !RHS_I4;
  const bool lhs_by_rows = ROWS16 && (a.log2_M0 == 0 || a.lhs_rb == 64);
  const bool rhs_by_rows = ROWS16 && a.rhs_rb == 64;
  uint32_t a_off[A_LOADS], b_off[B_LOADS];
  if constexpr (G == 16) {
#pragma unroll
    for (int t = 0; t < A_LOADS; ++t) {
      const int p = 64 * a_number(t) + lane;
      int c = RHS_I4 ? ((p >> 6) & 1) + 2 * ((p >> 5) & 1) : (p >> 4) & 3;
      int row = RHS_I4 ? (p >> 7) * 32 + (p & 31) : (p >> 7) * 32 + 16 * ((p >> 6) & 1) + (p & 15);
      if (lhs_by_rows) {
        c = (p & 3) ^ ((p >> 4) & 3);
        row = (p >> 7) * 32 + 16 * ((p >> 6) & 1) + ((p >> 2) & 15);
      }
      a_off[t] = row_offset(row, rows_left - 1, a.log2_M0, a.lhs_stride_bytes, a.log2_lhs_rb) +
                 ((16 * c) >> a.log2_lhs_rb << log2_lhs_kstep) + ((16 * c) & (a.lhs_rb - 1));
    }
#pragma unroll
    for (int t = 0; t < B_LOADS; ++t) {
      const int p = 64 * b_number(t) + lane;
      int c = RHS_I4 ? (p >> 5) & 1 : (p >> 4) & 3;
      int row = RHS_I4 ? (p >> 6) * 32 + (p & 31) : (p >> 7) * 32 + 16 * ((p >> 6) & 1) + (p & 15);
      if (rhs_by_rows) {
        c = (p & 3) ^ ((p >> 4) & 3);
        row = (p >> 7) * 32 + 16 * ((p >> 6) & 1) + ((p >> 2) & 15);
      }
      b_off[t] = row_offset(row, cols_left - 1, a.log2_N0, a.rhs_stride_bytes, a.log2_rhs_rb) +
                 ((16 * c) >> a.log2_rhs_rb << log2_rhs_kstep) + ((16 * c) & (a.rhs_rb - 1));
    }
  } else if constexpr (G == 1) {
    // One-byte row pieces (K0 = 1 int8: the operand is k-major, M0 bytes per k
    // step). A load brings one group of 16 rows x 64 k steps = 1 KiB, group
    // m of the operand (fragment m >> 1), into slots 64*m .. 64*m + 63:
    // 16-row tiles: lane l the 16 rows at k step l; 8-row tiles: lane l the 8
    // rows of tile l & 1 of the group at k steps 2*(l >> 1) and + 1. Either
    // way a k step's 16 rows lie within 32 bytes of LDS and the transposing
    // read (lds_read_transposed) hands lane (r, h) 8 consecutive k of row r; two
    // of them make a K-step's 16 bytes, in ascending k like every layout here.
    auto piece_of = [&](int log2_t0, int group, int* row, int* k1) {
      *row = 16 * group + (log2_t0 == 4 ? 0 : 8 * (lane & 1));
      *k1 = log2_t0 == 4 ? lane : 2 * (lane >> 1);
    };
#pragma unroll
    for (int t = 0; t < A_LOADS; ++t) {
      int row, k1;
      piece_of(a.log2_M0, a_number(t), &row, &k1);
      a_off[t] = row_offset(row, rows_left - (1 << a.log2_M0), a.log2_M0, a.lhs_stride_bytes, a.log2_lhs_rb) +
                 (k1 << log2_lhs_kstep);
    }
#pragma unroll
    for (int t = 0; t < B_LOADS; ++t) {
      int row, k1;
      piece_of(a.log2_N0, b_number(t), &row, &k1);
      b_off[t] = row_offset(row, cols_left - (1 << a.log2_N0), a.log2_N0, a.rhs_stride_bytes, a.log2_rhs_rb) +
                 (k1 << log2_rhs_kstep);
    }
  } else {
    constexpr int R = 16 / G;  // rows per 16-byte piece
    // Row group and k step of the chunk of this lane's piece in load m.
    auto piece_of = [&](int log2_t0, bool paired, int m, int* row, int* k1) {
      if (paired) {
        *row = 64 * (m >> 2) + 8 * (lane & 7);
        *k1 = 16 * ((m >> 1) & 1) + 8 * ((lane >> 3) & 1) + 4 * (m & 1) + (lane >> 4);
      } else if constexpr (G == 4) {
        // (Selected by masks, which the compiler does not make branches of.)
        const int eight = -(int)(log2_t0 == 3), x = (lane & 3) ^ ((lane >> 2) & 2);
        const int g = ((2 * ((lane >> 2) & 3) + (x & 1)) & eight) | (lane & 7 & ~eight);
        const int h = ((x >> 1) & eight) | ((lane >> 3) & 1 & ~eight);
        *row = 32 * (m >> 1) + 4 * g;
        *k1 = 8 * (m & 1) + 2 * (lane >> 4) + h;
      } else {
        *row = 32 * (m >> 1) + R * (lane % (2 * G));
        *k1 = (32 / G) * (m & 1) + (16 / G) * ((lane / (2 * G)) & 1) + lane / (4 * G);
      }
    };
#pragma unroll
    for (int t = 0; t < A_LOADS; ++t) {
      int row, k1;
      piece_of(a.log2_M0, PAIR_A, a_number(t), &row, &k1);
      a_off[t] = row_offset(row, rows_left - R, a.log2_M0, a.lhs_stride_bytes, a.log2_lhs_rb) + (k1 << log2_lhs_kstep);
    }
#pragma unroll
    for (int t = 0; t < B_LOADS; ++t) {
      int row, k1;
      piece_of(a.log2_N0, PAIR_B, b_number(t), &row, &k1);
      b_off[t] = row_offset(row, cols_left - R, a.log2_N0, a.rhs_stride_bytes, a.log2_rhs_rb) + (k1 << log2_rhs_kstep);
    }
  }

  acc_t acc[AM][BN];
#pragma unroll
  for (int i = 0; i < AM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

  const GroupChunks<GROUPS> own_chunks(a.chunks, a.K, a.log2_lhs_rb, group);
  const int chunks = own_chunks.count, last_chunk = own_chunks.last;
  const int32_t lhs_cut = own_chunks.cut_of_row << a.log2_M0;
  const int32_t rhs_cut = own_chunks.cut_of_row << a.log2_N0 >> (RHS_I4 ? 1 : 0);
  const int32_t cut_bytes = own_chunks.cut_bytes;

  // Loads number `n` (compile-time after unrolling) of the chunk whose operand bases are la / lb, into the stage at LDS byte
  // offset `stage_off`, the wavefront's first slots included.
  constexpr int A_ISSUES = TOGETHER ? 1 : A_LOADS, ISSUES = A_ISSUES + (TOGETHER ? 1 : B_LOADS);
  const int32_t b_from_a = 16 * A_PIECES + 1024 * (b_number(0) - a_number(0));
  if constexpr (TOGETHER) {
    static_assert(A_LOADS <= 2 && B_LOADS <= 2, "one pair");
    if constexpr (A_LOADS == 2) a_off[0] += 1024;  // (see load_two_to_lds; the bases are 1 KiB lower)
    if constexpr (B_LOADS == 2) b_off[0] += 1024;
  }
  // (`further`: bytes from that stage to the one meant; a, b: per-lane offsets.)
  auto issue_load_to = [&](auto number, auto further, uint32_t stage_off, uint32_t b_stage_off, const uint32_t* a, const uint32_t* b,
                           const uint8_t* la, const uint8_t* lb) {
    constexpr int n = decltype(number)::value;
    constexpr uint32_t FURTHER = decltype(further)::value;
    if constexpr (TOGETHER) {
      if constexpr (n == 0) {
        if constexpr (A_LOADS == 2) load_two_to_lds<FURTHER>(stage_off, a[0], a[1], la);
        else load_to_lds<FURTHER>(stage_off, a[0], la);
      } else {
        if constexpr (B_LOADS == 2) load_two_to_lds<FURTHER>(b_stage_off, b[0], b[1], lb);
        else load_to_lds<FURTHER>(b_stage_off, b[0], lb);
      }
    } else {
      if constexpr (n < A_LOADS) load_to_lds<FURTHER + 4096 * n>(stage_off, a[n], la);
      else load_to_lds<FURTHER + 16 * A_PIECES + 4096 * (n - A_LOADS)>(stage_off, b[n - A_LOADS], lb);
    }
  };
  auto issue_load = [&](auto number, uint32_t stage_off, const uint8_t* la, const uint8_t* lb) {
    issue_load_to(number, std::integral_constant<uint32_t, 0>(), stage_off, stage_off + b_from_a, a_off, b_off, la, lb);
  };
  const uint8_t* lhs_from = lhs_base - (TOGETHER && A_LOADS == 2 ? 1024 : 0);
  const uint8_t* rhs_from = rhs_base - (TOGETHER && B_LOADS == 2 ? 1024 : 0);
  auto lhs_near = [&](int kc) { return lhs_from + own_chunks.offset(kc, lhs_chunk_bytes, lhs_cut); };
  auto rhs_near = [&](int kc) { return rhs_from + own_chunks.offset(kc, rhs_chunk_bytes, rhs_cut); };
  // The group's ring.
  const uint32_t ring_off = (uint32_t)group * (STAGES * STAGE_PIECES * 16);
  const uint4* const own_ring = ring + ring_off / 16;
  // (Chunk c lies in stage c - 1 modulo their number.)
  const uint4* const first_stage = own_ring + (STAGES - 1) * STAGE_PIECES;
  auto issue_chunk = [&](int kc) {
    const uint32_t stage_off = ring_off + (uint32_t)((kc + STAGES - 1) % STAGES) * (STAGE_PIECES * 16) + 1024 * a_number(0);
    const uint8_t* la = lhs_near(kc);
    const uint8_t* lb = rhs_near(kc);
    each_of<ISSUES>([&](auto n) { issue_load(n, stage_off, la, lb); });
  };

  uint4 pa[AM][2], pb[BN][2], qa[AM][2], qb[BN][2];
  // G == 4: byte offset of a lane's first dword inside a fragment's K-step, see the layouts above.
  auto dwords_lane_offset = [&](int log2_t0) -> int32_t {
    const int h = lane >> 5, r = lane & 31, g = r >> 2, eight = -(int)(log2_t0 == 3);
    const int s = ((4 * (g >> 1) + ((2 * h + (g & 1)) ^ (2 * (g >> 2)))) & eight) | ((8 * h + g) & ~eight);
    return 16 * s + 4 * (r & 3);
  };
  // G < 16: dword `part` (0..3) of a lane's operand for one (fragment, K-step),
  // whose first element is at `first` (already including the lane's offset):
  // the elements are 64*G bytes apart.
  auto gather_dword = [](const uint8_t* first, int part) -> uint32_t {
    if constexpr (G == 2) {
      const uint32_t lo = *(const uint16_t*)(first + (2 * part) * 128);
      const uint32_t hi = *(const uint16_t*)(first + (2 * part + 1) * 128);
      return lo | (hi << 16);
    } else if constexpr (G == 4) {
      return *(const uint32_t*)(first + part * 256);
    } else {
      return *(const uint32_t*)(first + (part >> 1) * 512 + 4 * (part & 1));
    }
  };
  // G == 1: byte offset of lane (r, h)'s transposing reads inside a fragment's
  // 2 KiB (two 16-row groups of 1 KiB, k-major): group r >> 4, k steps from 16*h,
  // and the lane's chunk c = r & 15 of the 16 that one read transposes: the 8
  // rows 8*(c & 1) .. + 7 at k step c >> 1.
  auto transposed_lane_offset = [&](int log2_t0) -> int32_t {
    const int c = lane & 15;
    const int chunk = log2_t0 == 4 ? 8 * c : 32 * (c >> 2) + 16 * (c & 1) + 8 * ((c >> 1) & 1);
    return 1024 * ((lane & 31) >> 4) + 256 * (lane >> 5) + chunk;
  };
  // Fragment f of an operand at 16-byte slot `operand` of the ring, K-step kk.
  auto read_frag = [&](int operand, int f, int kk) -> uint4 {
    if (RHS_I4 && operand >= A_PIECES) {
      const uint4 raw = first_stage[operand + 64 * f + lane];
      return widen_i4_times16(kk ? make_uint2(raw.z, raw.w) : make_uint2(raw.x, raw.y));
    }
    if constexpr (G == 16) {
      if (!RHS_I4 && (operand == 0 ? lhs_by_rows : rhs_by_rows))
        return first_stage[operand + 128 * f + 64 * ((lane & 31) >> 4) + 4 * (lane & 15) + ((2 * kk + (lane >> 5)) ^ ((lane >> 2) & 3))];
      if (!RHS_I4) return first_stage[operand + 128 * f + 32 * kk + 64 * ((lane & 31) >> 4) + 16 * (lane >> 5) + (lane & 15)];
      return first_stage[operand + 128 * f + 64 * kk + lane];
    } else if constexpr (G == 1) {
      const uint8_t* first = (const uint8_t*)(first_stage + operand) + 2048 * f + 512 * kk +
                             transposed_lane_offset(operand >= A_PIECES ? a.log2_N0 : a.log2_M0);
      const uint2 lo = lds_read_transposed(first), hi = lds_read_transposed(first + 128);
      return make_uint4(lo.x, lo.y, hi.x, hi.y);
    } else {
      const uint8_t* first = (const uint8_t*)(first_stage + operand) + 1024 * (2 * f + kk) +
                             (G == 4 ? dwords_lane_offset(operand >= A_PIECES ? a.log2_N0 : a.log2_M0) : G * lane);
      return make_uint4(gather_dword(first, 0), gather_dword(first, 1), gather_dword(first, 2), gather_dword(first, 3));
    }
  };
  // Paired fragments: dwords 2*part and 2*part + 1 of the lane's eight for
  // (pair, K-step), split into dword `part` of the even and of the odd fragment.
  auto set_dword = [](uint4& v, int part, uint32_t w) {
    if (part == 0) v.x = w; else if (part == 1) v.y = w; else if (part == 2) v.z = w; else v.w = w;
  };
  auto read_pair_part = [](const uint8_t* first, int part) -> uint2 {
    return make_uint2(*(const uint32_t*)(first + 512 * part), *(const uint32_t*)(first + 512 * part + 256));
  };
  auto split_pair_part = [&](uint2 w, int part, uint4& even, uint4& odd) {
    set_dword(even, part, __builtin_amdgcn_perm(w.y, w.x, 0x05040100u));
    set_dword(odd, part, __builtin_amdgcn_perm(w.y, w.x, 0x07060302u));
  };
  const int frag_a0 = wave_m * AM, frag_b0 = wave_n * BN;

  // Loop-carried, wavefront-uniform state.
  constexpr uint32_t STAGE_BYTES = STAGE_PIECES * 16, RING_BYTES = STAGES * STAGE_BYTES;
  RingPlace<STAGES, GROUPS, STAGE_BYTES> at(lhs_near(AHEAD), rhs_near(AHEAD), ring_off + 1024 * a_number(0));
  const uint32_t frag_a_off = (uint32_t)((wave_m * AM) * 128) * 16;
  const uint32_t frag_b_off = (uint32_t)(A_PIECES + (wave_n * BN) * (RHS_I4 ? 64 : 128)) * 16;
  // Lane 32*h + r's byte offset into a fragment, and the slots from one K-step
  // of a fragment to the next (see the layouts above).
  const uint8_t* ring_bytes =
      (const uint8_t*)own_ring + (ROWS16 ? 16 * (64 * ((lane & 31) >> 4) + 16 * (lane >> 5) + (lane & 15))
                                     : (G == 1 || G == 4 ? 0 : G * lane));
  // What a lane's reads of either operand add to that. G == 1: the transposing reads' offset. G == 4: the dword reads'. G == 2: lanes address
  // dwords, not 16-bit elements. Paired: dword number
  // lane; unpaired: the dword that holds the lane's element (two lanes share
  // it), from which `own_half` then picks the low or the high half. (16-bit
  // reads that fill the halves of a register one after the other made these
  // tiles 1.8x slower than the 4-byte ones: the second read of a register has
  // to wait for the first.) G == 16, by rows: the distance to the by-rows slot for K-step 0.
  const int32_t by_rows_slot0 = 4 * (lane & 15) + ((lane >> 5) ^ ((lane >> 2) & 3));
  auto lane_offset = [&](int log2_t0, bool paired, bool by_rows) -> int32_t {
    if constexpr (G == 1) return transposed_lane_offset(log2_t0);
    if constexpr (G == 2) return paired ? 2 * lane : -2 * (lane & 1);
    if constexpr (G == 4) return dwords_lane_offset(log2_t0);
    return by_rows ? 16 * (by_rows_slot0 - (16 * (lane >> 5) + (lane & 15))) : 0;
  };
  const int32_t pair_a_lane = lane_offset(a.log2_M0, PAIR_A, lhs_by_rows);
  const int32_t pair_b_lane = lane_offset(a.log2_N0, PAIR_B, rhs_by_rows);
  // Bytes from a fragment's K-step 0 to its K-step 1 in this lane's reads (16-byte pieces).
  const int32_t lhs_kk1_step = lhs_by_rows ? 16 * ((by_rows_slot0 ^ 2) - by_rows_slot0) : 16 * (ROWS16 ? 32 : 64);
  const int32_t rhs_kk1_step = rhs_by_rows ? 16 * ((by_rows_slot0 ^ 2) - by_rows_slot0) : 16 * 32;
  const uint32_t own_half = (lane & 1) ? 0x07060302u : 0x05040100u;

  // Zeroes what chunk 0 shares with chunk 1. Lane half h of K-step kk holds bytes 32*kk + 16*h .. + 15 of
  // the chunk's 64 bytes per row, in ascending order of k; with an int4 rhs bytes 16*kk + 32*h .. + 15; of 4-byte
  // pieces every other one of bytes 32*kk .. + 31, from the h-th on.
  auto cut_fragments = [&](uint4 (*fa)[2], uint4 (*fb)[2]) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int first_byte = RHS_I4 ? 16 * kk + 32 * (lane >> 5) : 32 * kk + 16 * (lane >> 5);
      const int kept = min(max(64 - cut_bytes - first_byte, 0), 16);
      uint32_t keep[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if constexpr (G == 4) {
          keep[w] = 32 * kk + 8 * w + 4 * (lane >> 5) < 64 - cut_bytes ? 0xFFFFFFFFu : 0u;
          continue;
        }
        keep[w] = kept >= 4 * w + 4 ? 0xFFFFFFFFu : (kept <= 4 * w ? 0u : (1u << (8 * (kept - 4 * w))) - 1);
      }
#pragma unroll
      for (int i = 0; i < AM; ++i) {
        fa[i][kk].x &= keep[0]; fa[i][kk].y &= keep[1]; fa[i][kk].z &= keep[2]; fa[i][kk].w &= keep[3];
      }
      if constexpr (!RHS_I4) {
#pragma unroll
        for (int j = 0; j < BN; ++j) {
          fb[j][kk].x &= keep[0]; fb[j][kk].y &= keep[1]; fb[j][kk].z &= keep[2]; fb[j][kk].w &= keep[3];
        }
      }
    }
  };
  // One pipeline step for the chunk whose fragments are in `cur`:
  //   a few MFMAs first (they only need registers, and keep the matrix pipe
  //   fed across the barrier); wait until this wavefront's loads of the next
  //   chunk have landed; barrier (now everyone's have, and everyone is done
  //   reading the stage of the previous chunk); then the remaining MFMAs with,
  //   between them, the loads of the chunk three ahead into the stage just
  //   freed and the LDS reads of the next chunk's fragments.
  // A wavefront issues in order and a memory instruction takes several cycles
  // to issue, so more than one or two of them between two MFMAs lets the
  // matrix pipe run dry: they are dealt out one (half) fragment and at most one
  // load per MFMA. The reads end a quarter of the step before its end, so that
  // the last of them has returned when the next step starts; fragments are
  // read in the order the next step consumes them.
  // (`held_loads_behind`: the eight loads of destination values that variant 3 issues at the start of a phase
  // are younger than the chunk this step waits for, and may stay in flight with it.)
  // `between_mfmas(m)`: extra work placed behind MFMA m of the step (variant 3 adds destination values there).
  // `place`: where this step's loads go and its fragments come from, and what follows it.
  auto step_at = [&](const uint4 (*cur_a)[2], const uint4 (*cur_b)[2], uint4 (*nxt_a)[2], uint4 (*nxt_b)[2],
                     bool held_loads_behind, auto between_mfmas, auto place) {
    constexpr int SUB = SubSteps<KIND>::value;
    constexpr int MFMAS = 2 * AM * BN * SUB;
    // Units a fragment's LDS reads are dealt out in: a 128-bit read; two pairs of
    // dwords; two 64-bit reads; four pairs of dwords holding 16-bit elements.
    constexpr int PARTS = G == 16 ? 1 : (G == 2 ? 4 : 2);
    // Read units, in the order the next step consumes them: per K-step the rhs
    // fragments, then the lhs fragments. An int4 rhs fragment is read once, raw,
    // for both K-steps (first), and widened after the last read has been issued.
    constexpr int B_UNITS = RHS_I4 ? BN : 0;
    constexpr int UNITS_A = AM * (PAIR_A ? 2 : PARTS), UNITS_B = BN * (PAIR_B ? 2 : PARTS);  // per K-step
    constexpr int READS = RHS_I4 ? BN + 2 * AM : 2 * (UNITS_A + UNITS_B);
    constexpr int LEAD = MFMAS >= 16 ? 4 : (MFMAS >= 8 ? 2 : 0);   // MFMAs ahead of the barrier
    // MFMAs after the last read. (On the 128x64 tile 2-byte pieces get one, so that their reads are not split
    // right behind their issue: 128 x 14336 x 4096 int8 16x16x2 27 -> 24 us, f16 16x16x1 49 -> 42 us; on the
    // 64x64 tile it changed nothing.)
    constexpr int TAIL_FREE = MFMAS >= 8 ? MFMAS / 4 : ((RHS_I4 || (G == 2 && MFMAS >= 4)) ? 1 : 0);
    constexpr int SLOTS = MFMAS - LEAD - TAIL_FREE;                // MFMAs that carry memory work
    static_assert(SLOTS >= 1, "no room for the memory instructions");
    static_assert(!RHS_I4 || TAIL_FREE >= 1, "nowhere to widen");
    // Paired fragments: the dwords of a read unit are split this many MFMAs
    // after the read was issued (a wavefront issues in order: splitting right
    // away would stall it, MFMAs included, for the LDS latency of every unit).
    // (3 MFMAs: int8 16x16x2 at 4096^3 86 us; 5: 81 us; 8, all there are on the 256x256 tile: 79 us.)
    constexpr int SPLIT_DELAY = TAIL_FREE;
    uint2 raw_pair[G == 2 ? READS : 1];
    // Where read unit u of the next step's fragments goes.
    auto unit_of = [&](int u, bool* is_b, bool* paired, int* kk, int* y) {
      *kk = u / (UNITS_A + UNITS_B);
      const int x = u % (UNITS_A + UNITS_B);
      *is_b = x < UNITS_B;
      *paired = *is_b ? PAIR_B : PAIR_A;
      *y = *is_b ? x : x - UNITS_B;
    };
    auto split_units_of = [&](int read_slot) {
      if constexpr (G == 2) {
        if (read_slot < 0 || read_slot >= SLOTS) return;
#pragma unroll
        for (int u = read_slot * READS / SLOTS; u < (read_slot + 1) * READS / SLOTS; ++u) {
          bool is_b, paired;
          int kk, y;
          unit_of(u, &is_b, &paired, &kk, &y);
          uint4(*nxt)[2] = is_b ? nxt_b : nxt_a;
          if (paired) {
            split_pair_part(raw_pair[u], y % 4, nxt[2 * (y / 4)][kk], nxt[2 * (y / 4) + 1][kk]);
          } else {
            set_dword(nxt[y / 4][kk], y % 4, __builtin_amdgcn_perm(raw_pair[u].y, raw_pair[u].x, own_half));
          }
        }
      }
    };
    auto multiply = [&](int m) {
      const int kk = m / (AM * BN * SUB), sub = (m / (AM * BN)) % SUB, i = (m % (AM * BN)) / BN, j = m % BN;
      acc[i][j] = mfma<KIND>(cur_b[j][kk], cur_a[i][kk], acc[i][j], sub);
    };
#pragma unroll
    for (int m = 0; m < LEAD; ++m) {
      multiply(m);
      between_mfmas(m);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (STAGGER == 3) {
      if (held_loads_behind) wait_loads_but<LOADS*(AHEAD - 2) + 8>(); else wait_loads_but<LOADS*(AHEAD - 2)>();
    } else {
      wait_loads_but<LOADS*(AHEAD - 2)>();
    }
    __builtin_amdgcn_s_barrier();
    // (K-step 1 of either: used where it has 16-byte pieces)
    const uint8_t *read_a, *read_a_kk1, *read_b, *read_b_kk1;
    place.read_from(&read_a, &read_a_kk1, &read_b, &read_b_kk1);
    uint4 raw_b[RHS_I4 ? BN : 1];
#pragma unroll
    for (int m = LEAD; m < MFMAS; ++m) {
      const int slot = m - LEAD;
      if (slot < SLOTS) {
        each_of<ISSUES>([&](auto n) {
          if (n.value >= slot * ISSUES / SLOTS && n.value < (slot + 1) * ISSUES / SLOTS)
            place.load(n);
        });
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = slot * READS / SLOTS; u < (slot + 1) * READS / SLOTS; ++u) {
          if constexpr (RHS_I4) {
            if (u < B_UNITS) {
              raw_b[u] = *(const uint4*)(read_b + (64 * u) * 16);
            } else {
              const int kk = (u - B_UNITS) / AM, i = (u - B_UNITS) % AM;
              nxt_a[i][kk] = *(const uint4*)((kk ? read_a_kk1 : read_a) + 128 * i * 16);
            }
          } else {
            bool is_b, paired;
            int kk, y;
            unit_of(u, &is_b, &paired, &kk, &y);
            const uint8_t* src = is_b ? read_b : read_a;
            uint4(*nxt)[2] = is_b ? nxt_b : nxt_a;
            if (paired) {
              raw_pair[u] = read_pair_part(src + 4096 * (y / 4) + 2048 * kk, y % 4);
              continue;
            }
            const int frag = y / PARTS, part = y % PARTS;
            uint4& dst = nxt[frag][kk];
            if constexpr (G == 16) {
              if (is_b) dst = *(const uint4*)((kk ? read_b_kk1 : read_b) + 128 * frag * 16);
              else dst = *(const uint4*)((kk ? read_a_kk1 : read_a) + 128 * frag * 16);
            } else {
              const uint8_t* first = src + 1024 * (2 * frag + kk);
              if constexpr (G == 1) {
                // One transposing read: 8 consecutive k of the lane's row.
                const uint2 w = lds_read_transposed(src + 2048 * frag + 512 * kk + 128 * part);
                if (part == 0) { dst.x = w.x; dst.y = w.y; } else { dst.z = w.x; dst.w = w.y; }
              } else if constexpr (G == 2) {
                // Elements 2*part and 2*part + 1 of the lane's eight, 128 bytes apart, each with its neighbour.
                raw_pair[u] = make_uint2(*(const uint32_t*)(first + 256 * part), *(const uint32_t*)(first + 256 * part + 128));
                (void)dst;
              } else if constexpr (G == 8) {
                // One 64-bit read (two dword reads of adjacent addresses, which
                // is what the compiler makes of 4-byte aligned accesses, collide
                // on the banks: lanes are 8 bytes apart).
                const uint2 w = *(const uint2*)(first + part * 512);
                if (part == 0) { dst.x = w.x; dst.y = w.y; } else { dst.z = w.x; dst.w = w.y; }
              } else {
                if (part == 0) { dst.x = gather_dword(first, 0); dst.y = gather_dword(first, 1); }
                else { dst.z = gather_dword(first, 2); dst.w = gather_dword(first, 3); }
              }
            }
          }
        }
      } else if constexpr (RHS_I4) {
        // Widening, dealt out over the MFMAs that carry no memory work.
        const int tail = slot - SLOTS;
#pragma unroll
        for (int w = tail * 2 * BN / TAIL_FREE; w < (tail + 1) * 2 * BN / TAIL_FREE; ++w) {
          const int kk = w / BN, j = w % BN;
          nxt_b[j][kk] = widen_i4_times16(kk ? make_uint2(raw_b[j].z, raw_b[j].w) : make_uint2(raw_b[j].x, raw_b[j].y));
        }
      }
      split_units_of(slot - SPLIT_DELAY);
      multiply(m);
      between_mfmas(m);
      if (m == MFMAS - 1) place.advance();
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // A step anywhere: all of that is running state, advanced by the step.
  auto running_read = [&](const uint8_t** read_a, const uint8_t** read_a_kk1, const uint8_t** read_b, const uint8_t** read_b_kk1) {
    *read_a = ring_bytes + at.read_off + frag_a_off + pair_a_lane;
    *read_a_kk1 = *read_a + lhs_kk1_step;
    *read_b = ring_bytes + at.read_off + frag_b_off + pair_b_lane;
    *read_b_kk1 = *read_b + rhs_kk1_step;
  };
  auto running_load = [&](auto n) { issue_load(n, at.load_off, at.load_a, at.load_b); };
  auto running_advance = [&]() { at.advance(last_chunk, lhs_chunk_bytes, rhs_chunk_bytes); };
  auto step_with = [&](const uint4 (*cur_a)[2], const uint4 (*cur_b)[2], uint4 (*nxt_a)[2], uint4 (*nxt_b)[2],
                       bool held_loads_behind, auto between_mfmas) {
    step_at(cur_a, cur_b, nxt_a, nxt_b, held_loads_behind, between_mfmas,
            StepPlace<decltype(running_read), decltype(running_load), decltype(running_advance)>{running_read, running_load, running_advance});
  };
  auto step = [&](const uint4 (*cur_a)[2], const uint4 (*cur_b)[2], uint4 (*nxt_a)[2], uint4 (*nxt_b)[2],
                  bool held_loads_behind = false) {
    step_with(cur_a, cur_b, nxt_a, nxt_b, held_loads_behind, [](int) {});
  };

  // The last AHEAD chunks, for the 256x256 tile. At the end of the loop above
  // every accumulator becomes final at the same moment, and the whole tile (256
  // KiB per workgroup, the whole output of the launch in one burst) is stored
  // with the matrix pipe idle. Here the loop stops AHEAD chunks early, when
  // their operands are all in the workgroup already (one chunk's fragments in
  // registers, the others in the ring), and those chunks are multiplied in
  // another order: first the register chunk as usual, during which the loads
  // still in flight are awaited and the ring chunks' rhs fragments and the first
  // row's lhs fragments are read; then fragment by fragment, two fragments of a
  // row at a time, each pair running through the ring chunks and being stored
  // while the next pair is multiplied (one 128-bit store per MFMA, the first
  // behind the pair's last MFMA by a few instructions so that it does not wait
  // for it). Only the last pair's stores come after the last MFMA. The stores of
  // the launch are thereby spread over the last two and a half steps.
  // K in whole chunks, unpaired fragment layouts.
  constexpr bool TAILED = STAGGER != 0;
  static_assert(!TAILED || (AM == 4 && BN == 4 && !RHS_I4 && !PAIR_A && !PAIR_B && KIND != kF32), "staggered tail");
  // Output addressing of this wavefront's fragments, as in store_block: the byte offset of quad (j, q) from the
  // sub-block's first column tile, whether it lies inside the matrix, and the pointer of a fragment row's line.
  typedef typename AccType<KIND>::scalar out_scalar_t;
  typedef out_scalar_t out_quad_t __attribute__((ext_vector_type(4)));
  typedef typename std::conditional<NARROW, uint2, out_quad_t>::type out_stored_t;
  constexpr int OUT_BYTES = NARROW ? 2 : 4;
  struct OutAddressing {
    uint8_t* wave_out;
    uint32_t col_off[BN][4];
    uint32_t col_inside;
  };
  auto out_addressing = [&]() -> OutAddressing {
    OutAddressing o;
    const int32_t N0 = 1 << a.log2_N0;
    const int64_t wave_col = first_col + wave_n * (32 * BN);
    const int64_t first_col_tile = wave_col >> a.log2_N0;
    o.wave_out = a.out + OUT_BYTES * (first_col_tile << (a.log2_M0 + a.log2_N0));
    o.col_inside = 0;
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t col = wave_col + 4 * (lane >> 5) + 32 * j + 8 * q;
        o.col_off[j][q] = (uint32_t)(OUT_BYTES * ((((col >> a.log2_N0) - first_col_tile) << (a.log2_M0 + a.log2_N0)) +
                                                  (col & (N0 - 1))));
        if (col < total_cols) o.col_inside |= 1u << (4 * j + q);
      }
    return o;
  };
  auto out_row_pointer = [&](const OutAddressing& o, int i, bool* inside) -> uint8_t* {
    const int32_t M0 = 1 << a.log2_M0;
    const int64_t this_row = first_row + wave_m * (32 * AM) + 32 * i + (lane & 31);
    const int64_t row = min(this_row, total_rows - 1);
    *inside = this_row < total_rows;
    return o.wave_out + OUT_BYTES * ((row >> a.log2_M0) * a.out_stride0 + ((row & (M0 - 1)) << a.log2_N0));
  };
  constexpr int OUT_EBITS = KIND == kF16 ? 5 : 8;
  auto out_to_float = [](out_stored_t w) -> out_quad_t {
    if constexpr (NARROW) {
      return out_quad_t{widen16_first<OUT_EBITS>(w.x), widen16_second<OUT_EBITS>(w.x),
                        widen16_first<OUT_EBITS>(w.y), widen16_second<OUT_EBITS>(w.y)};
    } else {
      return w;
    }
  };
  auto out_to_stored = [](out_quad_t v) -> out_stored_t {
    if constexpr (NARROW) {
      return make_uint2(narrow16_pair<OUT_EBITS>(v.x, v.y), narrow16_pair<OUT_EBITS>(v.z, v.w));
    } else {
      return v;
    }
  };

  auto tail = [&](auto cur_a, auto cur_b) {  // (generic: only instantiated where it is called)
    constexpr int JR = AHEAD - 1;            // chunks in the ring
    constexpr int PAIR_MFMAS = 4 * JR;       // two fragments x JR chunks x two K-steps
    static_assert(PAIR_MFMAS >= 8, "a quad of the previous pair is stored with each MFMA");
    const OutAddressing o = out_addressing();

    // Fragment f of an operand, K-step kk, from the stage whose per-lane bases are given.
    auto read_fragment = [&](const uint8_t* base_a, const uint8_t* base_a_kk1, const uint8_t* base_b, bool is_b, int f,
                             int kk) -> uint4 {
      const uint8_t* src = is_b ? base_b : base_a;
      if constexpr (G == 16) {
        if (is_b) return *(const uint4*)(src + (kk ? rhs_kk1_step : 0) + 128 * f * 16);
        return *(const uint4*)((kk ? base_a_kk1 : base_a) + 128 * f * 16);
      } else if constexpr (G == 1) {
        const uint2 lo = lds_read_transposed(src + 2048 * f + 512 * kk);
        const uint2 hi = lds_read_transposed(src + 2048 * f + 512 * kk + 128);
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
      } else if constexpr (G == 8) {
        const uint8_t* first = src + 1024 * (2 * f + kk);
        const uint2 lo = *(const uint2*)first, hi = *(const uint2*)(first + 512);
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
      } else {
        const uint8_t* first = src + 1024 * (2 * f + kk);
        return make_uint4(gather_dword(first, 0), gather_dword(first, 1), gather_dword(first, 2), gather_dword(first, 3));
      }
    };
    // Per-lane bases of the ring chunks' stages.
    const uint8_t* base_a[JR];
    const uint8_t* base_a_kk1[JR];
    const uint8_t* base_b[JR];
    {
      uint32_t stage_off = at.read_off;
#pragma unroll
      for (int c = 0; c < JR; ++c) {
        base_a[c] = ring_bytes + stage_off + frag_a_off + pair_a_lane;
        base_a_kk1[c] = base_a[c] + lhs_kk1_step;
        base_b[c] = ring_bytes + stage_off + frag_b_off + pair_b_lane;
        stage_off = stage_off + STAGE_BYTES == RING_BYTES ? 0 : stage_off + STAGE_BYTES;
      }
    }
    uint4 tb[BN][JR][2], ta[2][JR][2];
    // The reads of the register phase, in the order the first pair needs them: per chunk and K-step the first
    // lhs row and the first two rhs fragments, then the other two rhs fragments.
    constexpr int EARLY_READS = 2 * JR * (1 + BN);
    auto early_read = [&](int n) {
      const int half = n / (2 * JR * 3);  // 0: lhs row 0 and rhs 0, 1; 1: rhs 2, 3
      if (half == 0) {
        const int c = n / 6, kk = (n / 3) % 2, what = n % 3;
        if (what == 0) ta[0][c][kk] = read_fragment(base_a[c], base_a_kk1[c], base_b[c], false, 0, kk);
        else tb[what - 1][c][kk] = read_fragment(base_a[c], base_a_kk1[c], base_b[c], true, what - 1, kk);
      } else {
        const int m = n - 2 * JR * 3, c = m / 4, kk = (m / 2) % 2, j = 2 + m % 2;
        tb[j][c][kk] = read_fragment(base_a[c], base_a_kk1[c], base_b[c], true, j, kk);
      }
    };

    // Register phase: the chunk whose fragments are in `cur`, in the usual order.
    constexpr int REG_MFMAS = 2 * AM * BN;
    constexpr int WAIT_AT = REG_MFMAS - 20 > 4 ? 12 : 4;  // MFMAs ahead of the wait for the ring chunks' loads
#pragma unroll
    for (int m = 0; m < REG_MFMAS; ++m) {
      if (m == WAIT_AT) {
        wait_loads_but<0>();
        __builtin_amdgcn_s_barrier();
      }
      if (m >= WAIT_AT) {
        constexpr int SLOTS = REG_MFMAS - WAIT_AT;
#pragma unroll
        for (int n = (m - WAIT_AT) * EARLY_READS / SLOTS; n < (m - WAIT_AT + 1) * EARLY_READS / SLOTS; ++n) early_read(n);
      }
      const int kk = m / (AM * BN), i = (m % (AM * BN)) / BN, j = m % BN;
      acc[i][j] = mfma<KIND>(cur_b[j][kk], cur_a[i][kk], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }

    // Fragment phase. (The accumulators are pinned where they are, here and again before each pair is stored:
    // left alone, the compiler moves them to ordinary registers ahead of the stores, and there are not that many.)
#pragma unroll
    for (int i = 0; i < AM; ++i)
#pragma unroll
      for (int j = 0; j < BN; ++j) asm volatile("" : "+a"(acc[i][j]));
    uint8_t* prev_row = nullptr;
    bool prev_row_inside = false;
    // Quad n (fragment n / 4 of the pair, quad n % 4) of pair (i, jp). An accumulating call adds what the
    // destination held, loaded while the pair was multiplied (one quad per MFMA, each into the register the
    // previous pair's quad of the same number has just been added from).
    constexpr bool ACCUMULATING = STAGGER == 2;
    out_quad_t old[2][4];
    auto store_quad = [&](int i, int jp, int n, uint8_t* row_out, bool row_inside) {
      const int t = n / 4, q = n % 4, j = 2 * jp + t;
      out_quad_t v = out_quad_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      if constexpr (ACCUMULATING) v += old[t][q];
      if (row_inside && (o.col_inside >> (4 * j + q) & 1)) *(out_stored_t*)(row_out + o.col_off[j][q]) = out_to_stored(v);
    };
    auto load_old = [&](int jp, int n, const uint8_t* row_out, bool row_inside) {
      const int t = n / 4, q = n % 4, j = 2 * jp + t;
      old[t][q] = out_quad_t{0, 0, 0, 0};
      if (row_inside && (o.col_inside >> (4 * j + q) & 1))
        old[t][q] = out_to_float(*(const out_stored_t*)(row_out + o.col_off[j][q]));
    };
#pragma unroll
    for (int i = 0; i < AM; ++i) {
      bool row_inside;
      uint8_t* row_out = out_row_pointer(o, i, &row_inside);
#pragma unroll
      for (int jp = 0; jp < BN / 2; ++jp) {
        const int pair = i * (BN / 2) + jp;
#pragma unroll
        for (int m = 0; m < PAIR_MFMAS; ++m) {
          // The previous pair's quads, from the third MFMA on (its last MFMA has left the pipe by then).
          constexpr int STORE_FROM = PAIR_MFMAS >= 10 ? 2 : 0;
          const int n = m - STORE_FROM;
          if (n >= 0 && n < 8) {
            if (pair > 0) {
              const int pi = (pair - 1) / (BN / 2), pjp = (pair - 1) % (BN / 2);
              if (n == 0) asm volatile("" : "+a"(acc[pi][2 * pjp]), "+a"(acc[pi][2 * pjp + 1]));
              store_quad(pi, pjp, n, pi == i ? row_out : prev_row, pi == i ? row_inside : prev_row_inside);
            }
            if constexpr (ACCUMULATING) load_old(jp, n, row_out, row_inside);
          }
          // The next row's lhs fragments, read under this row's second pair.
          if (jp == BN / 2 - 1 && i + 1 < AM && m < 2 * JR)
            ta[(i + 1) & 1][m / 2][m % 2] = read_fragment(base_a[m / 2], base_a_kk1[m / 2], base_b[m / 2], false, i + 1, m % 2);
          const int c = m / 4, kk = (m / 2) % 2, t = m % 2, j = 2 * jp + t;
          acc[i][j] = mfma<KIND>(tb[j][c][kk], ta[i & 1][c][kk], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      prev_row = row_out;
      prev_row_inside = row_inside;
    }
    // The last pair's quads.
    UK_TIMELINE(const unsigned long long tl_last_mfma = __builtin_amdgcn_s_memrealtime();)
    asm volatile("" : "+a"(acc[AM - 1][BN - 2]), "+a"(acc[AM - 1][BN - 1]));
#pragma unroll
    for (int n = 0; n < 8; ++n) store_quad(AM - 1, BN / 2 - 1, n, prev_row, prev_row_inside);
    UK_TIMELINE(asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (lane == 0 && wave == 0 && blockIdx.x < 256) {
                  unsigned long long* t = uk_timeline + blockIdx.x * 8;
                  t[0] = tl_start; t[1] = tl_loop; t[2] = tl_loop_end; t[3] = tl_last_mfma;
                  t[4] = __builtin_amdgcn_s_memrealtime();
                })
  };

#pragma unroll
  for (int c = 0; c < AHEAD; ++c) issue_chunk(c);
  wait_loads_but<(AHEAD - 1) * LOADS>();
  __syncthreads();
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int j = 0; j < BN; ++j) {
      if constexpr (PAIR_B) {
        if (j % 2 == 0) {
#pragma unroll
          for (int part = 0; part < 4; ++part)
            split_pair_part(
                read_pair_part((const uint8_t*)(first_stage + A_PIECES) + 2048 * (frag_b0 + j) + 2048 * kk + 4 * lane, part),
                part, pb[j][kk], pb[j + 1][kk]);
        }
      } else {
        pb[j][kk] = read_frag(A_PIECES, frag_b0 + j, kk);
      }
    }
#pragma unroll
    for (int i = 0; i < AM; ++i) {
      if constexpr (PAIR_A) {
        if (i % 2 == 0) {
#pragma unroll
          for (int part = 0; part < 4; ++part)
            split_pair_part(read_pair_part((const uint8_t*)first_stage + 2048 * (frag_a0 + i) + 2048 * kk + 4 * lane, part),
                            part, pa[i][kk], pa[i + 1][kk]);
        }
      } else {
        pa[i][kk] = read_frag(0, frag_a0 + i, kk);
      }
    }
  }
  if (!TAILED && cut_bytes != 0) cut_fragments(pa, pb);
  UK_TIMELINE(tl_loop = __builtin_amdgcn_s_memrealtime();)
  int kc = 0;
  if constexpr (TAILED) {
    // (The host launches this variant only for K in whole chunks, at least 2 * STAGES of them.)
    // An odd step first, so that the loop always ends with the next chunk's fragments in (pa, pb).
    const int main_steps = chunks - AHEAD;
    if (main_steps & 1) {
      step(pa, pb, qa, qb);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int i = 0; i < AM; ++i) pa[i][kk] = qa[i][kk];
#pragma unroll
        for (int j = 0; j < BN; ++j) pb[j][kk] = qb[j][kk];
      }
      kc = 1;
    }
    if constexpr (STAGGER == 3) {
      // An accumulating call: what the destination held is added to the accumulators on the way, so that the
      // tail only stores (read in the tail, the 256 KiB per workgroup come from HBM on top of the stores, with
      // three chunks of MFMAs to hide under). One phase per pair of fragments: its eight quads are loaded, an even
      // number of steps runs, and in the last of them the values are added, each fragment's behind its first
      // MFMA of that step, two registers per MFMA, done before its second. The loads are issued from assembly,
      // like those of the ring, so that the compiler does not wait for them (its waits would be for every load
      // in flight, the ring's youngest included): after three steps they have landed, because loads return in
      // order and the third step waits for a chunk that was requested after them. A lane outside the matrix loads
      // from the start of the destination; what it adds is never stored.
      static_assert(SubSteps<KIND>::value == 1, "one MFMA per fragment and K-step");
      const OutAddressing o = out_addressing();
      constexpr int PAIRS = AM * (BN / 2);
      // The workgroups of a launch run in step; were all of them to load a pair at the same moment, the 16 MiB
      // would take longer to arrive than the two steps the ring can wait. Each therefore starts its phases a
      // different number of steps into the loop (one phase's worth of steps is set aside for that).
      const int per_phase = ((main_steps - kc) / (PAIRS + 1)) & ~1;  // (the host sees to it that this is at least 4)
      for (int lead = 2 * ((int)((blockIdx.x >> 3) & 7) * (per_phase / 2) >> 3); lead > 0; lead -= 2, kc += 2) {
        step(pa, pb, qa, qb);
        step(qa, qb, pa, pb);
      }
#pragma unroll
      for (int pair = 0; pair < PAIRS; ++pair) {
        const int i = pair / (BN / 2), jp = pair % (BN / 2);
        bool row_inside;
        const uint8_t* row_out = out_row_pointer(o, i, &row_inside);
        out_stored_t held[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const int j = 2 * jp + n / 4, q = n % 4;
          const uint8_t* from = row_inside && (o.col_inside >> (4 * j + q) & 1) ? row_out + o.col_off[j][q] : a.out;
          if constexpr (NARROW) asm volatile("global_load_dwordx2 %0, %1, off" : "=v"(held[n]) : "v"(from) : "memory");
          else asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(held[n]) : "v"(from) : "memory");
        }
        int held_loads_behind = 1;
        for (int s = 0; s + 2 < per_phase; s += 2, kc += 2) {
          asm volatile("" : "+s"(held_loads_behind));  // (one copy of the loop body, not a peeled first pass)
          step(pa, pb, qa, qb, held_loads_behind != 0);
          step(qa, qb, pa, pb, held_loads_behind != 0);
          held_loads_behind = 0;
        }
        step(pa, pb, qa, qb);
        out_quad_t was[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          asm volatile("" : "+v"(held[n]));
          was[n] = out_to_float(held[n]);
        }
        step_with(qa, qb, pa, pb, false, [&](int m) {
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int j = 2 * jp + t, slot = m - (i * BN + j + 2);
            if (slot < 0 || slot >= 8) continue;
#pragma unroll
            for (int r = 2 * slot; r < 2 * slot + 2; ++r) acc[i][j][r] += was[4 * t + r / 4][r % 4];
          }
        });
        kc += 2;
      }
    }
    for (; kc + 1 < main_steps; kc += 2) {
      step(pa, pb, qa, qb);
      step(qa, qb, pa, pb);
    }
    UK_TIMELINE(tl_loop_end = __builtin_amdgcn_s_memrealtime();)
    tail(pa, pb);
    return;
  }
  // Four steps at a time while all of their loads are of chunks that exist: where a step reads and loads is then a constant
  // beyond one base each, and the four chunks' offsets are registers. 28 instructions a step of the 128x64 tile where a step
  // anywhere has 46, 21 of 38 for 64x64, 64 of 80 for 64x128 and an int4 rhs. bf16 8x8x4 512 x 4096 x 4096 24.3 -> 22.4 us,
  // 16x16x16 22.8 -> 22.0, int8 16x16x2 19.2 -> 18.2, int4 256 x 8000 x 3008 13.0 -> 12.4, 784 x 4112 x 4096 (128x128) 21.4 -> 21.0.
  // Not where it was level: int8 but for its 2-byte pieces (128x64
  // -4 to +4 %) and the 128x128 tile of others, bound by the LDS (-2 to +2 %).
  constexpr bool BY_FOUR = STAGES % 4 == 0 && KIND != kF32 && (RHS_I4 ? AM * BN <= 4 : AM * BN <= 2 && (KIND != kI8 || G == 2));
  typedef FourSteps<STAGES == 8 ? 8 : 4, GROUPS, STAGE_BYTES> Fours;
  if constexpr (BY_FOUR) if (Fours::pays(last_chunk)) {
    uint32_t fast_a[4][A_LOADS], fast_b[4][B_LOADS];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int t = 0; t < A_LOADS; ++t) fast_a[c][t] = a_off[t] + c * GROUPS * lhs_chunk_bytes;
#pragma unroll
      for (int t = 0; t < B_LOADS; ++t) fast_b[c][t] = b_off[t] + c * GROUPS * rhs_chunk_bytes;
    }
    Fours fours(at);
    const uint8_t* from_a = ring_bytes + frag_a_off + pair_a_lane;
    const uint8_t* from_b = ring_bytes + frag_b_off + pair_b_lane;
    while (Fours::fits(kc, last_chunk)) {
      const uint32_t read_off = fours.reads(at);
      const uint8_t* base_a = from_a + read_off;
      const uint8_t* base_b = from_b + read_off;
      const uint8_t *base_a_kk1 = base_a + lhs_kk1_step, *base_b_kk1 = base_b + rhs_kk1_step;
      each_of<4>([&](auto number) {
        constexpr int S = decltype(number)::value;
        auto read = [&](const uint8_t** read_a, const uint8_t** read_a_kk1, const uint8_t** read_b, const uint8_t** read_b_kk1) {
          *read_a = base_a + S * STAGE_BYTES;
          *read_a_kk1 = base_a_kk1 + S * STAGE_BYTES;
          *read_b = base_b + S * STAGE_BYTES;
          *read_b_kk1 = base_b_kk1 + S * STAGE_BYTES;
        };
        auto load = [&](auto n) {
          const uint32_t four = fours.loads(S);
          issue_load_to(n, std::integral_constant<uint32_t, Fours::loads_into(S) * STAGE_BYTES>(), four, four + b_from_a, fast_a[S],
                        fast_b[S], at.load_a, at.load_b);
        };
        auto advance = [] {};
        StepPlace<decltype(read), decltype(load), decltype(advance)> place{read, load, advance};
        if constexpr (S % 2 == 0) step_at(pa, pb, qa, qb, false, [](int) {}, place);
        else step_at(qa, qb, pa, pb, false, [](int) {}, place);
      });
      kc += 4;
      fours.advance(&at, lhs_chunk_bytes, rhs_chunk_bytes);
    }
    fours.leave(&at, kc, last_chunk, lhs_chunk_bytes, rhs_chunk_bytes);
  }
  for (; kc + 1 < chunks; kc += 2) {
    step(pa, pb, qa, qb);
    step(qa, qb, pa, pb);
  }
  if (kc < chunks) step(pa, pb, qa, qb);
  // No load may still be writing LDS when the workgroup's allocation is freed.
  wait_loads_but<0>();
  UK_TIMELINE(tl_loop_end = __builtin_amdgcn_s_memrealtime();)

  if constexpr (GROUPS == 2) {
    // Group g takes the wavefront's fragments (i, j) with half of the i (or, AM = 1, of the j) and adds what the other group
    // has of them, the first group's sum first. sums[wavefront of all][fragment][4 registers of 16][lane]
    constexpr bool BY_ROWS = AM == 2;
    static_assert((AM == 2 && BN <= 2) || (AM == 1 && BN == 2), "halves of one row or column of fragments");
    static_assert(!PAIR_A && !PAIR_B && STAGGER == 0, "fragments on their own");
    constexpr int HALF = AM * BN / 2;
    static_assert(8 * HALF * 4 * 64 * 16 <= 2 * STAGES * STAGE_PIECES * 16, "the rings take the sums");
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4* const sums = (u32x4*)ring;
    __syncthreads();  // nobody reads operands from the rings any more
    auto fragment = [&](int of_group, int f) -> acc_t& { return BY_ROWS ? acc[of_group][f] : acc[0][of_group]; };
#pragma unroll
    for (int f = 0; f < HALF; ++f) {
      acc_t other = fragment(1, f);
      if (group == 1) other = fragment(0, f);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sums[((wave_of_all * HALF + f) * 4 + v) * 64 + lane] =
            u32x4{value_bits(other[4 * v]), value_bits(other[4 * v + 1]), value_bits(other[4 * v + 2]), value_bits(other[4 * v + 3])};
    }
    __syncthreads();
    acc_t total[1][BY_ROWS ? BN : 1];
#pragma unroll
    for (int f = 0; f < HALF; ++f) {
      acc_t own = fragment(0, f), part;
      if (group == 1) own = fragment(1, f);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const u32x4 bits = sums[(((wave_of_all ^ 4) * HALF + f) * 4 + v) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          typename AccType<KIND>::scalar value;
          set_from_bits(value, bits[e]);
          part[4 * v + e] = value;
        }
      }
      total[0][f] = own + part;
    }
    store_block<KIND, RHS_I4, NARROW, 1, BY_ROWS ? BN : 1, false, false, ACCUMULATE>(
        a, total, first_row + wave_m * (32 * AM) + (BY_ROWS ? 32 * group : 0),
        first_col + wave_n * (32 * BN) + (BY_ROWS ? 0 : 32 * group), lane);
    return;
  }
  store_block<KIND, RHS_I4, NARROW, AM, BN, PAIR_A, PAIR_B, ACCUMULATE>(a, acc, first_row + wave_m * (32 * AM),
                                                                        first_col + wave_n * (32 * BN), lane);
  UK_TIMELINE(asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
              if (lane == 0 && wave == 0 && blockIdx.x < 256) {
                unsigned long long* t = uk_timeline + blockIdx.x * 8;
                t[0] = tl_start; t[1] = tl_loop; t[2] = tl_loop_end; t[3] = tl_loop_end;
                t[4] = __builtin_amdgcn_s_memrealtime();
              })
}

// ---------------------------------------------------------------------------
// A 128x64 block tile whose four wavefronts split K instead of the tile, for 65 to
// 128 lhs rows against a long K (one tile row). The kernel above is then bound by
// the latency of one pipeline step (counter wait, barrier, LDS reads; about 140
// ns) per 64 bytes of K per workgroup. Here every wavefront multiplies the whole
// tile (4 x 2 fragments) over its quarter of the step's K bytes (one MFMA K-step
// of the 128 bytes per row and step; ring of 6 stages of 24 KiB), so a workgroup
// streams more per step, and the four partial tiles are summed through LDS at the
// end, in wavefront order (deterministic). Row pieces of 16 bytes or more, f16 /
// bf16. What bounds it is what a compute unit's load path moves (a stage takes
// about 400 cycles). Problems with fewer tiles go to mmt4d_wave_k_kernels.h.
//
// LDS stage: per operand four slices (one per wavefront's share of K, 16*COLS
// bytes per row, COLS = 2 * K-steps per wavefront) of fragments in the layout
// of the kernel above (G == 16) with COLS 16-byte columns: slot p of a
// fragment holds rows 16*(p / (16*COLS)) + (p & 15), column (p >> 4) & (COLS-1).
// A load fills 64 consecutive slots of one slice.
template <int KIND, bool NARROW, int ACCUMULATE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mmt4d_mfma_split_k_kernel(const MfmaArgs a) {
  typedef typename AccType<KIND>::type acc_t;
  static_assert(KIND == kF16 || KIND == kBF16, "16-bit floats");
  constexpr int AMF = 4;                      // 32-row lhs fragments
  constexpr int KKW = 1;                      // MFMA K-steps per wavefront and step
  constexpr int COLS = 2 * KKW;               // 16-byte columns of a slice
  constexpr int CHUNK_BYTES = 4 * 16 * COLS;  // of K per row and step
  constexpr int STAGES = 6, AHEAD = STAGES - 1;
  constexpr int FRAG_SLOTS = 32 * COLS;
  constexpr int A_SLICE = AMF * FRAG_SLOTS, B_SLICE = 2 * FRAG_SLOTS;  // slots per slice
  constexpr int A_PIECES = 4 * A_SLICE, B_PIECES = 4 * B_SLICE;
  constexpr uint32_t STAGE_BYTES = (A_PIECES + B_PIECES) * 16, RING_BYTES = STAGES * STAGE_BYTES;
  constexpr int A_LOADS = A_PIECES / 256, B_LOADS = B_PIECES / 256, LOADS = A_LOADS + B_LOADS;  // per wavefront
  constexpr int READS = KKW * (AMF + 2);      // 128-bit LDS reads per wavefront and step
  constexpr int MFMAS = KKW * AMF * 2;
  static_assert(MFMAS == 8 && LOADS <= 8 && READS <= 8, "the step below deals memory work over four of eight MFMAs");

  fetch_arguments(a);
  int tile_row, tile_col;
  if (!locate_block(a, &tile_row, &tile_col)) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int64_t total_rows = (int64_t)a.M << a.log2_M0;
  const int64_t total_cols = (int64_t)a.N << a.log2_N0;
  const int64_t lhs_kstep = (int64_t)a.lhs_rb << a.log2_M0;
  const int64_t rhs_kstep = (int64_t)a.rhs_rb << a.log2_N0;
  const int64_t lhs_chunk_bytes = (CHUNK_BYTES >> a.log2_lhs_rb) * lhs_kstep;
  const int64_t rhs_chunk_bytes = (CHUNK_BYTES >> a.log2_rhs_rb) * rhs_kstep;
  const int64_t first_row = (int64_t)tile_row * (32 * AMF), first_col = (int64_t)tile_col * 64;
  const uint8_t* lhs_base = a.lhs + (first_row >> a.log2_M0) * a.lhs_stride_bytes;
  const uint8_t* rhs_base = a.rhs + (first_col >> a.log2_N0) * a.rhs_stride_bytes;

  // Rows past the end of the matrix are redirected to its last row: computed, never stored.
  auto piece_offset = [&](int64_t row, int64_t last, int64_t first, int log2_t0, int64_t stride_bytes, int32_t rb,
                          int log2_rb, int64_t kstep, int byte_in_chunk) -> uint32_t {
    row = min(row, last);
    const int64_t tile = (row >> log2_t0) - (first >> log2_t0);
    return (uint32_t)(tile * stride_bytes + (row & ((1 << log2_t0) - 1)) * rb + (byte_in_chunk >> log2_rb) * kstep +
                      (byte_in_chunk & (rb - 1)));
  };
  // Load t of wavefront w is group 4*t + w of its operand's groups of 64 slots, slice by slice.
  auto group_of = [&](int t, int slice_slots, int* slice, int* row, int* byte_in_chunk) {
    const int group = 4 * t + wave, per_slice = slice_slots / 64;
    *slice = group / per_slice;
    const int p = 64 * (group % per_slice) + lane;  // slot within the slice
    *row = 32 * (p / FRAG_SLOTS) + 16 * ((p / (16 * COLS)) & 1) + (p & 15);
    *byte_in_chunk = 16 * COLS * *slice + 16 * ((p >> 4) & (COLS - 1));
  };
  uint32_t a_off[A_LOADS], b_off[B_LOADS], a_lds[A_LOADS], b_lds[B_LOADS];
#pragma unroll
  for (int t = 0; t < A_LOADS; ++t) {
    int slice, row, byte_in_chunk;
    group_of(t, A_SLICE, &slice, &row, &byte_in_chunk);
    a_off[t] = piece_offset(first_row + row, total_rows - 1, first_row, a.log2_M0, a.lhs_stride_bytes, a.lhs_rb,
                            a.log2_lhs_rb, lhs_kstep, byte_in_chunk);
    a_lds[t] = (uint32_t)(64 * (4 * t + wave)) * 16;
  }
#pragma unroll
  for (int t = 0; t < B_LOADS; ++t) {
    int slice, row, byte_in_chunk;
    group_of(t, B_SLICE, &slice, &row, &byte_in_chunk);
    b_off[t] = piece_offset(first_col + row, total_cols - 1, first_col, a.log2_N0, a.rhs_stride_bytes, a.rhs_rb,
                            a.log2_rhs_rb, rhs_kstep, byte_in_chunk);
    b_lds[t] = (uint32_t)(A_PIECES + 64 * (4 * t + wave)) * 16;
  }

  acc_t acc[AMF][2];
#pragma unroll
  for (int i = 0; i < AMF; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

  const int chunks = (int)(((int64_t)a.K << a.log2_lhs_rb) / CHUNK_BYTES);  // K is whole steps
  const int last_chunk = chunks - 1;

  auto issue_load = [&](int n, uint32_t stage_off, const uint8_t* la, const uint8_t* lb) {
    if (n < A_LOADS) load_to_lds(stage_off + a_lds[n], a_off[n], la);
    else load_to_lds(stage_off + b_lds[n - A_LOADS], b_off[n - A_LOADS], lb);
  };
  // This wavefront's operand registers for one chunk: fragment f, K-step kk.
  uint4 pa[AMF][KKW], pb[2][KKW], qa[AMF][KKW], qb[2][KKW];
  // Lane 32*h + r reads slot 16*COLS*(r >> 4) + 16*(2*kk + h) + (r & 15) of a fragment.
  const uint8_t* lane_a = (const uint8_t*)ring +
                          16 * (A_SLICE * wave + 16 * COLS * ((lane & 31) >> 4) + 16 * (lane >> 5) + (lane & 15));
  const uint8_t* lane_b = lane_a + 16 * (A_PIECES + (B_SLICE - A_SLICE) * wave);
  // Read number u of a step, in the order the next step consumes them: per K-step the rhs fragments, then the lhs.
  auto read_unit = [&](int u, const uint8_t* stage, uint4 (*fa)[KKW], uint4 (*fb)[KKW]) {
    const int kk = u / (AMF + 2), e = u % (AMF + 2);
    if (e < 2) fb[e][kk] = *(const uint4*)(stage + (lane_b - (const uint8_t*)ring) + (FRAG_SLOTS * e + 32 * kk) * 16);
    else fa[e - 2][kk] = *(const uint4*)(stage + (lane_a - (const uint8_t*)ring) + (FRAG_SLOTS * (e - 2) + 32 * kk) * 16);
  };

  const uint8_t* load_a = lhs_base + min(AHEAD, last_chunk) * lhs_chunk_bytes;
  const uint8_t* load_b = rhs_base + min(AHEAD, last_chunk) * rhs_chunk_bytes;
  int load_chunk = AHEAD;
  uint32_t load_stage_off = AHEAD * STAGE_BYTES % RING_BYTES;
  uint32_t read_stage_off = STAGE_BYTES;

  // One step, as in the kernel above: two MFMAs ahead of the wait and the barrier, then the loads of the chunk
  // AHEAD ahead and the LDS reads of the next chunk dealt out over four MFMAs, two MFMAs without memory work.
  auto step = [&](const uint4 (*cur_a)[KKW], const uint4 (*cur_b)[KKW], uint4 (*nxt_a)[KKW], uint4 (*nxt_b)[KKW]) {
    auto multiply = [&](int m) {
      const int kk = m / (AMF * 2), i = (m % (AMF * 2)) >> 1, j = m & 1;
      acc[i][j] = mfma<KIND>(cur_b[j][kk], cur_a[i][kk], acc[i][j]);
    };
    multiply(0);
    multiply(1);
    __builtin_amdgcn_sched_barrier(0);
    wait_loads_but<LOADS*(AHEAD - 2)>();
    __builtin_amdgcn_s_barrier();
    const uint8_t* stage = (const uint8_t*)ring + read_stage_off;
#pragma unroll
    for (int m = 2; m < 8; ++m) {
      const int slot = m - 2;
      if (slot < 4) {
#pragma unroll
        for (int n = slot * LOADS / 4; n < (slot + 1) * LOADS / 4; ++n) issue_load(n, load_stage_off, load_a, load_b);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = slot * READS / 4; u < (slot + 1) * READS / 4; ++u) read_unit(u, stage, nxt_a, nxt_b);
      }
      multiply(m);
      if (m == 7) {
        const bool more = load_chunk < last_chunk;
        load_a += more ? lhs_chunk_bytes : 0;
        load_b += more ? rhs_chunk_bytes : 0;
        ++load_chunk;
        load_stage_off = load_stage_off + STAGE_BYTES == RING_BYTES ? 0 : load_stage_off + STAGE_BYTES;
        read_stage_off = read_stage_off + STAGE_BYTES == RING_BYTES ? 0 : read_stage_off + STAGE_BYTES;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int c = 0; c < AHEAD; ++c) {
    const int idx = min(c, last_chunk);
#pragma unroll
    for (int n = 0; n < LOADS; ++n)
      issue_load(n, (uint32_t)c * STAGE_BYTES, lhs_base + idx * lhs_chunk_bytes, rhs_base + idx * rhs_chunk_bytes);
  }
  wait_loads_but<(AHEAD - 1) * LOADS>();
  __syncthreads();
#pragma unroll
  for (int u = 0; u < READS; ++u) read_unit(u, (const uint8_t*)ring, pa, pb);
  int kc = 0;
  for (; kc + 1 < chunks; kc += 2) {
    step(pa, pb, qa, qb);
    step(qa, qb, pa, pb);
  }
  if (kc < chunks) step(pa, pb, qa, qb);
  wait_loads_but<0>();
  __syncthreads();  // nobody reads operands from the ring any more

  // The four partial tiles, summed in wavefront order. Wavefront w ends up with the fragments
  // (OWN*(w >> 1) + o, w & 1), o < OWN: a block of (32*OWN) x 32 outputs. partial[((f*4 + w)*16 + v)][lane] is
  // accumulator register v of wavefront w's fragment f = 2*i + j.
  constexpr int OWN = AMF / 2;
  uint32_t* partial = (uint32_t*)ring;
#pragma unroll
  for (int f = 0; f < 2 * AMF; ++f) {
    const int i = f >> 1, j = f & 1;
    if (2 * (i / OWN) + j != wave) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const typename AccType<KIND>::scalar value = acc[i][j][v];
        partial[((f * 4 + wave) * 16 + v) * 64 + lane] = value_bits(value);
      }
    }
  }
  __syncthreads();
  acc_t total[OWN][1];
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    // (the wavefront's own partial, selected without indexing the accumulator array by a run-time value)
    acc_t own = acc[o][0];
#pragma unroll
    for (int w = 1; w < 4; ++w)
      if (wave == w) own = acc[OWN * (w >> 1) + o][w & 1];
    const int f = 2 * (OWN * (wave >> 1) + o) + (wave & 1);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      acc_t part;
      if (w == wave) {
        part = own;
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          typename AccType<KIND>::scalar value;
          set_from_bits(value, partial[((f * 4 + w) * 16 + v) * 64 + lane]);
          part[v] = value;
        }
      }
      if (w == 0) total[o][0] = part; else total[o][0] += part;
    }
  }
  store_block<KIND, false, NARROW, OWN, 1, false, false, ACCUMULATE>(a, total, first_row + 32 * OWN * (wave >> 1), first_col + 32 * (wave & 1), lane);
}

// Whether the direct-to-LDS kernel covers the problem: every lane can load 16
// contiguous bytes (4-byte row pieces 4 rows at a time, an int4 rhs in pieces
// of 32 nibbles), and K is long enough.
template <bool RHS_I4, int G>
bool direct_covers(const MfmaArgs& m) {
  // K ending inside a chunk: one full chunk at least.
  const int64_t row_bytes = (int64_t)m.K * m.lhs_rb;
  if (row_bytes % 64 != 0 && row_bytes < 64) return false;
  if (RHS_I4) return m.rhs_rb >= 16 && (uintptr_t)m.rhs % 16 == 0 && m.rhs_stride_bytes % 16 == 0;
  if (G == 16) return true;
  // One-byte pieces: tiles of 8 or 16 rows (a 16-byte piece is one or two k steps of a whole tile).
  if (G == 1)
    return m.log2_M0 >= 3 && m.log2_N0 >= 3 && (uintptr_t)m.lhs % 16 == 0 && (uintptr_t)m.rhs % 16 == 0 &&
           m.lhs_stride_bytes % 16 == 0 && m.rhs_stride_bytes % 16 == 0;
  // 16 / G rows of one k step make up a lane's 16 bytes: tiles at least that tall.
  return (G << m.log2_M0) >= 16 && (G << m.log2_N0) >= 16 && (uintptr_t)m.lhs % 16 == 0 &&
         (uintptr_t)m.rhs % 16 == 0 && m.lhs_stride_bytes % 16 == 0 && m.rhs_stride_bytes % 16 == 0;
}

void set_tile_grid(MfmaArgs* m, int block_rows, int block_cols, unsigned* grid) {
  const int64_t rows = (int64_t)m->M << m->log2_M0, cols = (int64_t)m->N << m->log2_N0;
  m->tile_rows = (int32_t)((rows + block_rows - 1) / block_rows);
  m->tile_cols = (int32_t)((cols + block_cols - 1) / block_cols);
  const int64_t tiles = (int64_t)m->tile_rows * m->tile_cols;
  m->band_reciprocal = band_reciprocal((uint32_t)m->tile_cols);
  *grid = (unsigned)(((tiles + 7) / 8) * 8);
}

// Direct-to-LDS kernel on (64*AM) x (64*BN) block tiles with a ring of STAGES stages.
// GROUPS: of four wavefronts, that share K.
template <int KIND, bool RHS_I4, bool NARROW, int G, int AM, int BN, int STAGES, int GROUPS = 1>
hipError_t launch_direct(MfmaArgs m, hipStream_t stream, bool staggered_tail = true) {
  unsigned grid;
  set_tile_grid(&m, 64 * AM, 64 * BN, &grid);
  constexpr int stage_pieces = 256 * AM + (RHS_I4 ? 128 : 256) * BN;
  constexpr size_t lds_bytes = (size_t)GROUPS * STAGES * 16 * stage_pieces;
  static_assert(lds_bytes <= 160 * 1024, "ring does not fit the LDS");
  constexpr bool PAIRS = G == 2 && (AM % 2 == 0 || BN % 2 == 0);  // (see store_block)
  void (*kernel)(const MfmaArgs) = mmt4d_mfma_direct_kernel<KIND, RHS_I4, NARROW, G, AM, BN, STAGES, 0, GROUPS, PAIRS ? kAsked : kNever>;
  if constexpr (!PAIRS) {
    if (m.accumulate) kernel = mmt4d_mfma_direct_kernel<KIND, RHS_I4, NARROW, G, AM, BN, STAGES, 0, GROUPS, kAlways>;
  }
  // The 256x256 tile with the staggered tail: K in whole chunks, enough of them.
  if constexpr (AM == 4 && BN == 4 && !RHS_I4 && G != 2 && KIND != kF32) {
    if (staggered_tail && ((int64_t)m.K * m.lhs_rb) % 64 == 0 && m.chunks >= 2 * STAGES) {
      // (Accumulating: read the destination during the loop where every one of the eight phases gets four steps.)
      if (m.accumulate && m.chunks >= STAGES + 9 * 4) kernel = mmt4d_mfma_direct_kernel<KIND, RHS_I4, NARROW, G, AM, BN, STAGES, 3>;
      else if (m.accumulate) kernel = mmt4d_mfma_direct_kernel<KIND, RHS_I4, NARROW, G, AM, BN, STAGES, 2>;
      else kernel = mmt4d_mfma_direct_kernel<KIND, RHS_I4, NARROW, G, AM, BN, STAGES, 1>;
    }
  }
  // Above 64 KiB of dynamic LDS the limit has to be raised (per device, so it
  // is simply done on every launch: it only sets a field).
  if (lds_bytes > 65536) {
    const hipError_t attr =
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (attr != hipSuccess) return attr;
  }
  return launch_kernel<MfmaArgs>(kernel, grid, 256 * GROUPS, lds_bytes, stream, m);
}

template <int KIND, bool NARROW>
hipError_t launch_split_k(MfmaArgs m, hipStream_t stream) {
  unsigned grid;
  set_tile_grid(&m, 128, 64, &grid);
  constexpr int lds_bytes = 6 * 24576;
  auto kernel = m.accumulate ? mmt4d_mfma_split_k_kernel<KIND, NARROW, kAlways> : mmt4d_mfma_split_k_kernel<KIND, NARROW, kNever>;
  const hipError_t attr = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  if (attr != hipSuccess) return attr;
  return launch_kernel<MfmaArgs>(kernel, grid, 256, lds_bytes, stream, m);
}

// Register-staged kernel (any K, any alignment the plan admits).
template <int KIND, bool RHS_I4, bool NARROW, int G, int AM, int BN, int MIN_BLOCKS>
hipError_t launch_staged(MfmaArgs m, hipStream_t stream) {
  // 2- and 8-byte row pieces exist on the direct path only; the plan does not
  // admit problems that would need this kernel for them.
  if constexpr (G != 16 && G != 4) return hipErrorInvalidValue;
  else {
  unsigned grid;
  set_tile_grid(&m, 64 * AM, 64 * BN, &grid);
  // K ending inside a chunk needs the kernel variant with the zero-filling tail step.
  const bool tail = ((int64_t)m.K * m.lhs_rb) % 64 != 0;
  return launch_kernel<MfmaArgs>(tail ? mmt4d_mfma_kernel<KIND, RHS_I4, NARROW, G, AM, BN, MIN_BLOCKS, true>
                                      : mmt4d_mfma_kernel<KIND, RHS_I4, NARROW, G, AM, BN, MIN_BLOCKS, false>,
                                 grid, 256, 0, stream, m);
  }
}

// One workgroup per compute unit at most, and operands from HBM: what the workgroups have in flight then has to cover its
// latency, about 2 us under load, and the 24 KiB of either operand that four 128x128 stages hold ahead amount to 2.5 TB/s.
// Ten stages, all of the LDS, take from HBM bf16 512 x 5120 x 5120 (58 MB) from 56.7 to 48.4 us, 384 x 8192 x 4096 (70 MB)
// from 48.2 to 41.5, int8 192 x 14336 x 4096 (59 MB) from 28.3 to 25.7; with operands that a cache holds they cost nothing
// there (0.95 to 1.02, 2-byte pieces 1.02 to 1.06), below 48 MiB up to 10 %. Tiles of 64 columns have rings of eight
// stages and gained nothing from more.
inline bool streams_operands(const MfmaArgs& m, int block_rows, int block_cols) {
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  const int64_t tiles = ((rows + block_rows - 1) / block_rows) * ((cols + block_cols - 1) / block_cols);
  return tiles <= 256 && comes_from_hbm((rows * m.lhs_rb + cols * m.rhs_rb) * m.K);
}

template <int KIND, bool RHS_I4, int G, bool NARROW>
hipError_t launch_variant(const MfmaArgs& m, hipStream_t stream, const char** name) {
  const bool direct = direct_covers<RHS_I4, G>(m);
  if constexpr (G == 16 && (KIND == kF16 || KIND == kBF16)) {
    if (direct && split_k_covers(m)) {
      *name = "mmt4d_mfma_128x64_split_k";
      return launch_split_k<KIND, NARROW>(m, stream);
    }
  }
  constexpr bool kWide192 = KIND != kF32 && G != 1;
  double us_per_chunk;
  switch (choose_tile(m, KIND, RHS_I4, G, direct, &us_per_chunk)) {
    case 0:
      *name = "mmt4d_mfma_256x256";
#ifndef UK_STAGES_256
#define UK_STAGES_256 4
#endif
      if (direct) return launch_direct<KIND, RHS_I4, NARROW, G, 4, 4, UK_STAGES_256>(m, stream);
      return launch_staged<KIND, RHS_I4, NARROW, G, 4, 4, 1>(m, stream);
    case 1:
      *name = "mmt4d_mfma_256x128";
      return launch_direct<KIND, RHS_I4, NARROW, G, 4, 2, 4>(m, stream);
    case 2:
      *name = "mmt4d_mfma_128x128";
      if constexpr (!RHS_I4 && KIND != kF32) {
        if (direct && streams_operands(m, 128, 128)) return launch_direct<KIND, RHS_I4, NARROW, G, 2, 2, 10>(m, stream);
      }
      if constexpr (G != 2 && KIND != kF32) {
        if (two_groups(m, KIND, RHS_I4, G, direct, kBlockTiles[2]))
          return launch_direct<KIND, RHS_I4, NARROW, G, 2, 2, 4, 2>(m, stream);
      }
      if (direct) return launch_direct<KIND, RHS_I4, NARROW, G, 2, 2, 4>(m, stream);
      return launch_staged<KIND, RHS_I4, NARROW, G, 2, 2, 2>(m, stream);
    // (The conditions are choose_tile's: these shapes are not instantiated where it does not take them.)
    case 6:
      *name = "mmt4d_mfma_192x192";
      if constexpr (kWide192 && G != 2 && !RHS_I4) return launch_direct<KIND, RHS_I4, NARROW, G, 3, 3, 4>(m, stream);
      return hipErrorInvalidValue;
    case 7:
      *name = "mmt4d_mfma_128x192";
      if constexpr (kWide192 && G != 2 && !RHS_I4) return launch_direct<KIND, RHS_I4, NARROW, G, 2, 3, 4>(m, stream);
      return hipErrorInvalidValue;
    case 8:
      *name = "mmt4d_mfma_192x128";
      if constexpr (kWide192 && G != 2) return launch_direct<KIND, RHS_I4, NARROW, G, 3, 2, 4>(m, stream);
      return hipErrorInvalidValue;
    case 9:
      *name = "mmt4d_mfma_256x192";
      if constexpr (kWide192 && !RHS_I4) return launch_direct<KIND, RHS_I4, NARROW, G, 4, 3, 4>(m, stream);
      return hipErrorInvalidValue;
    case 10:
      *name = "mmt4d_mfma_192x256";
      if constexpr (kWide192 && !RHS_I4) return launch_direct<KIND, RHS_I4, NARROW, G, 3, 4, 4>(m, stream);
      return hipErrorInvalidValue;
    case 5:
      *name = "mmt4d_mfma_64x128";
      if constexpr (RHS_I4) {
        if (two_groups(m, KIND, RHS_I4, G, direct, kBlockTiles[5]))
          return launch_direct<KIND, RHS_I4, NARROW, G, 1, 2, 8, 2>(m, stream);
        return launch_direct<KIND, RHS_I4, NARROW, G, 1, 2, 8>(m, stream);
      }
      [[fallthrough]];
    case 3:
      *name = "mmt4d_mfma_128x64";
      if constexpr (!RHS_I4) return launch_direct<KIND, RHS_I4, NARROW, G, 2, 1, 8>(m, stream);
      [[fallthrough]];
    default:
      *name = "mmt4d_mfma_64x64";
      if constexpr (!RHS_I4) {
        if (direct) return launch_direct<KIND, RHS_I4, NARROW, G, 1, 1, 8>(m, stream);
      }
      return launch_staged<KIND, RHS_I4, NARROW, G, 1, 1, 2>(m, stream);
  }
}

}  // namespace
#endif  // UK_MFMA_KERNEL_BODIES

}  // namespace uk

#endif  // IREE_AMD_CSRC_MMT4D_MFMA_KERNELS_H_
