// Host side of the MFMA mmt4d kernels: which problems they cover, and the
// dispatch to the per-type translation units (mmt4d_mfma_kernels.h describes
// the kernels).
#include "mmt4d_mfma_kernels.h"

namespace uk {
namespace {

int log2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1))) return -1;
  int l = 0;
  while ((1ll << l) < v) ++l;
  return l;
}

const WaveKShape& wave_k_shape(int kind, int s) { return kind == kF32 ? kWaveKShapesF32[s] : kWaveKShapes[s]; }

struct Plan {
  int kind;
  bool rhs_i4;
  bool narrow;  // 16-bit output, rounded once at the end
  int gather;   // bytes of a row piece, 16 for 16 and more
  int wave_shape;  // tile of the kernel that splits K over wavefronts, or -1: a block kernel
  bool wave_tile;  // the kernel whose wavefronts have the whole of a large tile each, instead of either
  MfmaArgs args;
};

// Estimates in microseconds, to choose between the block kernels and the one that splits K over wavefronts. Both write
// the output at the same rate, which is left out. Measured over 741 problems (M 8..1100, N 64..28672, K 64..14336, every
// type and row piece) with operands from HBM (sets of 640 MB in turn, the condition of weights in a model's layers) and
// with operands that the last-level cache holds (150 MB), the coefficients fitted to the geometric mean of the two: the
// kernel picked is 0.5 % slower than the best one in the mean, 5 % and more on one problem in 31 (timed again since the kernels
// got shorter loops and prologues: 260 problems 0.6 %, one in 26; 200 of int4 0.3 %, one in 100). Fitted to repeated operands
// alone they would pick 32x64 tiles for bf16 96 x 14336 x 4096: 27.5 us held and 40.6 from HBM, where the 128x64 tile with
// K split takes 23.9 and 32.6; int4 96 x 14336 x 4096 19.1 from HBM against 16.3.
//
// f32: measured over 210 problems (M 17..4096, N 64..14336, K 64..8192, up to 8.6 GFLOP, 16- and 4-byte row pieces) with every
// tile, operands held: the terms below are off by 7 % (rms), the kernel picked is 0.5 % slower than the best one in the
// mean. The time to write the output is in both, per round of tiles.
double block_cost_f32(const MfmaArgs& m, int gather, bool direct) {
  // Microseconds per chunk of kBlockTiles' first five: one workgroup per compute unit, two beside each other.
  static const double kOne[] = {3.45, 1.83, .94, .494, .272}, kTwo[] = {6.9, 3.66, 1.763, .988, .47};
  double us_per_chunk;
  const int tile = choose_tile(m, kF32, false, gather, direct, &us_per_chunk);
  const TileChoice& t = kBlockTiles[tile];
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0, br = 64 * t.am, bc = 64 * t.bn;
  const int64_t rounds = (((rows + br - 1) / br) * ((cols + bc - 1) / bc) + 255) / 256;
  us_per_chunk = (rounds & 1) * kOne[tile] + (rounds >> 1) * kTwo[tile];
  if (!direct) us_per_chunk *= 2.2;  // staged through registers
  const double chunks_us = m.chunks * us_per_chunk + 1.2 * t.am * t.bn * rounds;
  const double memory_us = (double)(rows * m.lhs_rb + cols * m.rhs_rb) * m.K / 6.95e6;
  return 2.0 + (chunks_us > memory_us ? chunks_us : memory_us);
}

double wave_k_cost_f32(const MfmaArgs& m, const WaveKShape& s, int64_t tiles, bool staged) {
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  const double megabytes = 1e-6 * (double)(rows * m.lhs_rb + cols * m.rhs_rb) * m.K;
  const int fragments = s.fa * s.fb;
  // (The output is all there is, which the block kernels write faster: 2048 x 2048 x 16 8.3 us, in 32x64 tiles 12.8, 512 x 4096
  // x 48 6.9 and 8.1.)
  if (m.chunks < 4 && tiles > 256) return 1e30;
  // (Four steps a wavefront and less, four tiles a unit and more: summing and writing, which the block kernels do as they go
  // along, is most of it. One problem in 400 of K < 512 has another kernel for it; of 24 such, those kernels take 4 % less
  // in the mean: 464 x 13248 x 268 40.0 us with the block kernel, 46.8 in 80x64 tiles, 1008 x 6528 x 389 54.5 and 64.3, but 224
  // x 13136 x 496 34.7 and in 32x64 tiles 29.9.)
  if (m.chunks < 32 && tiles > 1024) return 1e30;
  // A chunk's multiplies at the pipe's rate, or its loads. Workgroups beside each other start and end beside each other too.
  const double multiplies = (staged ? 0.02 : 0.0142) * fragments, loads = (staged ? 0.0159 : 0.0107) * (s.fa + s.fb);
  const double us = 1.9 + (tiles > 256 ? tiles / 256.0 : 1.0) * (0.7 + 0.125 * fragments) +
                    (tiles + 255) / 256 * m.chunks * (multiplies > loads ? multiplies : loads) + 0.035 * megabytes;
  const double memory_us = 2.0 + megabytes / 6.95;
  return us > memory_us ? us : memory_us;
}

// A block kernel takes a fixed time per 64-byte chunk of K (choose_tile), or what its operands take from memory.
double block_cost(const MfmaArgs& m, int kind, bool rhs_i4, int gather) {
  const bool direct = mfma_direct_covers(m, gather, rhs_i4);
  if (kind == kF32) return block_cost_f32(m, gather, direct);
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  const double memory_us = (double)(rows * m.lhs_rb + cols * m.rhs_rb) * m.K / 6.95e6;
  double us_per_chunk, start_us = 3.52;
  if (gather == 16 && (kind == kF16 || kind == kBF16) && direct && split_k_covers(m)) {
    us_per_chunk = 0.163;
    start_us = 6.8;  // (and the summing of the partial tiles)
  } else {
    choose_tile(m, kind, rhs_i4, gather, direct, &us_per_chunk);
    // (int4, K ending inside a chunk, which is a mask in front of the loop: 0.2 us. With a few chunks of K this decides: 560 x 1760
    // x 288 5.0 us, 4.4 in 64x64 tiles of the other kernel; of 134 problems of up to 6 chunks that it alone gives to the other
    // kernel, the block kernel is 7 % slower in the mean. Of 40 such of 9 to 24 chunks it is 2 % faster in the mean and on 14 up to
    // 12 % slower, of 80 with more 14 % faster and on one 5 % slower: 144 x 6736 x 1568 7.9 us, 10.2 in 32x64 tiles.)
    if (rhs_i4 && m.chunks <= 24 && ((int64_t)m.K * m.lhs_rb) % 64 != 0) start_us += 0.4;
    if (!direct) us_per_chunk *= 2.2;       // staged through registers
    // Few rows and more 64x64 tiles than units: the unit's second tile, row pieces of 4 and 8 bytes, is dearer than the
    // table's (from 16-byte pieces, many rows): bf16 16 x 20720 x 7396, 16x16x2 tiles, 0.28 us and not 0.195. Without the
    // factor the block kernel was taken, 68 us, where a wave-K tile takes 60.
    if ((gather == 4 || gather == 8) && (kind == kF16 || kind == kBF16) && rows <= 16 && cols > 64 * 256) us_per_chunk *= 1.3;
    if (gather == 2) us_per_chunk *= 1.2;    // (the tiles that few rows take: wide ones, from HBM)
  }
  const double chunks_us = m.chunks * us_per_chunk;
  return start_us + (chunks_us > memory_us ? chunks_us : memory_us);
}

// The kernel that splits K over wavefronts is bound by the bytes a workgroup loads; workgroups beyond one per compute
// unit run beside each other where their registers and LDS allow it (not those of the 64x64 tile).
double wave_k_cost(const MfmaArgs& m, int kind, bool rhs_i4, int gather, const WaveKShape& s) {
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  // (In fragments, of which there are fewer than 2^31 either way: divisions of 32 bits.)
  const int64_t tiles = (int64_t)(((uint32_t)((rows + 15) / 16) + s.fa - 1) / s.fa) * (((uint32_t)((cols + 15) / 16) + s.fb - 1) / s.fb);
  const double row_kb = 1e-3 * m.K * m.lhs_rb, rhs_share = rhs_i4 ? 0.5 : 1.0;
  const bool narrow = gather < 16 && !wave_k_loads_pieces(m, kind, gather, s.fa, s.fb);  // row pieces that pass through LDS
  if (kind == kF32) return wave_k_cost_f32(m, s, tiles, narrow);
  // (Pieces of 2 and 8 bytes: chosen by what 255 problems lose to their best kernel. At 81.4 and a
  // start of 3.03, of before the end of K left the block kernels' steps, the pick was 1.9 % slower than the best one in the
  // mean, now 0.7: s8 208 x 5392 x 1480 in 16x16x2 tiles 13.4 -> 10.8 us, bf16 232 x 3504 x 1268 in 8x8x4 9.7 -> 8.5.)
  const bool narrow_2_8 = narrow && gather != 4;
  const double tile_us = 16 * (s.fa + s.fb * rhs_share) * row_kb / (narrow_2_8 ? 69.5 : narrow ? 81.4 : 92.5);
  double us = (narrow_2_8 ? 3.2 : narrow || rhs_i4 ? 3.03 : 2.63) + 0.067 * s.fa * s.fb + 4.6e-5 * (rows + cols * rhs_share) * row_kb;
  if (tiles <= 256) return us + tile_us;
  const double rounds = tiles / 256.0;
  if (tiles > (s.fa * s.fb >= 16 ? 256 : 1024)) us += 1e3 * rounds;
  // (int4, 106 problems: few tiles more than units cost more, many less; 320 x 1664 x 352 5.4 us in 260 tiles of 32x64, 4.3
  // in 130 of 64x64.)
  if (rhs_i4) return us + 0.4 + (rounds + 0.8) * tile_us + 0.402 * rounds;
  return us + (rounds + (narrow ? 0.941 : 0.922)) * tile_us + (narrow ? 0.467 : 0.402) * rounds;
}

// Whether the kernel that splits K over wavefronts covers the problem: 16-byte aligned operands whose 16 contiguous
// bytes belong to one k step.
bool wave_k_covers(const MfmaArgs& m, int gather, bool rhs_i4) {
  if (gather == 1 || (rhs_i4 && m.rhs_rb < 16)) return false;
  if (gather < 16 && ((gather << m.log2_M0) < 16 || (gather << m.log2_N0) < 16)) return false;
  return (uintptr_t)m.lhs % 16 == 0 && (uintptr_t)m.rhs % 16 == 0 && (m.M == 1 || m.lhs_stride_bytes % 16 == 0) &&
         (m.N == 1 || m.rhs_stride_bytes % 16 == 0);
}

// Whether the kernel whose wavefronts have a large tile each covers the problem: four lanes' 16-byte pieces, of four consecutive
// rows, in one 128-byte line; a whole chunk of K; offsets of a tile below its buffers' 2 GiB.
bool wave_tile_covers(const MfmaArgs& m, int kind, int gather, bool rhs_i4) {
  if (gather != 16 || kind == kF32 || (kind == kI8 && !rhs_i4) || !wave_k_covers(m, gather, rhs_i4)) return false;
  if (m.lhs_rb > 32 || m.log2_M0 < 2 || ((int64_t)m.K << m.log2_lhs_rb) < 64) return false;
  if (m.lhs_stride_bytes < 0 || m.rhs_stride_bytes < 0) return false;
  const int64_t lhs_reach = (128 >> m.log2_M0) * m.lhs_stride_bytes + (((int64_t)m.K + 8) << (m.log2_lhs_rb + m.log2_M0));
  const int64_t rhs_reach = (128 >> m.log2_N0) * m.rhs_stride_bytes + (((int64_t)m.K + 8) << (m.log2_rhs_rb + m.log2_N0));
  return lhs_reach < (1ll << 31) && rhs_reach < (1ll << 31);
}

// Whether it is the fastest, from 500 problems (M 17..4096, N 256..14336, K 256..8192, half a round of its tiles on the compute
// units to four) timed beside what was chosen for them, on three sets of operands in turn, which the last-level cache
// holds, and some on sets of 640 MB, from HBM.
// 16-bit operands, 128x128 tiles: 200 to 248 tiles and 64 chunks of K or more, 82 plain problems with a 32-bit output between 2.2 %
// slower and 10 % faster, 3.6 in the mean, from HBM 47 others 1 to 25 % faster, 8 in the mean. (249 to 256 tiles would gain
// too, 37 problems 0 to 10 %, from HBM 28 1 to 27: not taken so far.) With 22 to 48 chunks 2 to 14 % slower (the partial
// sums), with 140 to 199 tiles between 9 % slower and 7 % faster, a second round of tiles takes half as long again, and
// operands of more than 48 MiB (see streams_operands) -2 to +3 %.
// int4, 64x128 tiles: where 64x64 ones are more than a round of the compute units and these are not, and 32x64 ones would be taken
// and are more than two workgroups per unit: 120 problems 8 to 29 % faster, 18 in the mean, from HBM 120 others between 7 % slower
// and 16 % faster, 4.5 in the mean (from 94 chunks on 1.4). With up to 512 tiles of 32x64, which the units hold at once, 5 to 14 % slower
// (21 problems), from HBM 11 to 21 (12): 480 x 2144 x 7872 23.1 us, in 32x64 tiles 19.5. Where 32-high tiles
// have less padding, 160 rows and up to 160 that they divide, 3 to 14 % slower. (Where the block kernel's tile would be taken it
// is up to 5 % faster with 24 to 44 chunks, 17 with more, and from HBM 2 to 14 % slower. Near 256 tiles between 5 % slower and
// 6 % faster, beyond up to 30 % slower; with up to 256 tiles of 64x64 those take two thirds of the time.)
bool wave_tile_is_best(const MfmaArgs& m, bool rhs_i4, int wave_shape) {
  const int64_t rows = (int64_t)m.M << m.log2_M0, cols = (int64_t)m.N << m.log2_N0;
  const int64_t col_tiles = (cols + 127) / 128;
  if (rhs_i4) {
    const int64_t row_tiles = (rows + 63) / 64;
    const bool padded = 6 * 64 * row_tiles > 7 * 32 * ((rows + 31) / 32);  // (than 32-high tiles)
    return wave_shape >= 0 && row_tiles * ((cols + 63) / 64) > 256 && ((rows + 31) / 32) * ((cols + 63) / 64) > 512 &&
           row_tiles * col_tiles <= 240 && !padded && m.chunks >= 24;
  }
  const int64_t tiles = ((rows + 127) / 128) * col_tiles;
  return tiles >= 200 && tiles <= 248 && m.chunks >= 64 && wave_shape < 0 &&
         !comes_from_hbm((rows * m.lhs_rb + cols * m.rhs_rb) * m.K);
}

// Fills `plan` if the problem is covered. With `probe_only` only type and tile
// shape are looked at; without `choose` the kernel is left open.
bool make_plan(const Mmt4dArgs& a, bool probe_only, bool choose, Plan* plan) {
  int kind, elem_bytes;
  bool i4 = false, narrow = false;
  // With a 16-bit output the reference rounds the accumulator after every
  // multiply-add unless told to skip that (mmt4d_tile_generic.c:229-286,
  // 319-376): only the skipping variant (f32 accumulator, one rounding at the
  // end) is something a matrix pipe can compute.
  const bool skip_roundings = a.flags & IREE_UK_FLAG_MMT4D_SKIP_INTERMEDIATE_ROUNDINGS;
  switch (a.flags & IREE_UK_FLAG_MMT4D_TYPE_MASK) {
    case IREE_UK_FLAG_MMT4D_TYPE_S8S8S32: kind = kI8; elem_bytes = 1; break;
    case IREE_UK_FLAG_MMT4D_TYPE_S8S4S32: kind = kI8; elem_bytes = 1; i4 = true; break;
    case IREE_UK_FLAG_MMT4D_TYPE_F16F16F32: kind = kF16; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_BF16BF16F32: kind = kBF16; elem_bytes = 2; break;
    case IREE_UK_FLAG_MMT4D_TYPE_F32F32F32: kind = kF32; elem_bytes = 4; break;
    case IREE_UK_FLAG_MMT4D_TYPE_F16F16F16:
      if (!skip_roundings) return false;
      kind = kF16; elem_bytes = 2; narrow = true;
      break;
    case IREE_UK_FLAG_MMT4D_TYPE_BF16BF16BF16:
      if (!skip_roundings) return false;
      kind = kBF16; elem_bytes = 2; narrow = true;
      break;
    default: return false;
  }
  const int lm0 = log2_exact(a.M0), ln0 = log2_exact(a.N0);
  if (lm0 < 0 || ln0 < 0 || a.M0 > 16 || a.N0 > 16 || a.N0 < 4) return false;
  const int lhs_rb = a.K0 * elem_bytes;
  const int rhs_rb = i4 ? a.K0 / 2 : lhs_rb;
  const int llrb = log2_exact(lhs_rb), lrrb = log2_exact(rhs_rb);
  if (llrb < 0 || lrrb < 0) return false;
  int gather;
  if (i4) {
    if (lhs_rb < 16 || lhs_rb > 64) return false;
    gather = 16;
  } else if (lhs_rb >= 16 && lhs_rb <= 64) {
    gather = 16;
  } else if (lhs_rb == 1 && kind == kI8) {
    // int8 K0 = 1 (the Arm baseline tiles Mx8x1): k-major operands, transposed
    // on the way out of LDS; tiles of 8 or 16 rows, direct-to-LDS kernel only.
    if (lm0 < 3 || ln0 < 3) return false;
    gather = 1;
  } else if (lhs_rb == 4 || lhs_rb == 2 || lhs_rb == 8) {
    // 2 and 8 (e.g. the x86-64 int8 16x16x2 and f16 16x16x1 tiles, the Arm int8
    // 8x8x8 tiles) run on the direct-to-LDS kernel only: see below.
    gather = lhs_rb;
  } else {
    return false;
  }
  plan->kind = kind;
  plan->rhs_i4 = i4;
  plan->narrow = narrow;
  plan->gather = gather;
  if (probe_only) return true;

  const int64_t lhs_stride_bytes = a.lhs_stride0 * elem_bytes;
  const int64_t rhs_stride_bytes = i4 ? a.rhs_stride0 / 2 : a.rhs_stride0 * elem_bytes;
  // (four consecutive outputs per store: 16 bytes, 8 with a 16-bit output)
  if (((uintptr_t)a.out % (narrow ? 8 : 16)) || (a.M > 1 && a.out_stride0 % 4)) return false;
  // Per-piece offsets from a workgroup's first tile are kept in 32 bits.
  const int64_t lhs_reach = ((256 >> lm0) + 1) * lhs_stride_bytes + 80 * ((int64_t)lhs_rb << lm0);
  const int64_t rhs_reach = ((256 >> ln0) + 1) * rhs_stride_bytes + 80 * ((int64_t)rhs_rb << ln0);
  if (lhs_reach >= (1ll << 32) || rhs_reach >= (1ll << 32)) return false;
  // 16x-scaled int4 accumulation must not overflow int32.
  if (i4 && (int64_t)a.K * a.K0 >= 131072) return false;
  // K == 0 (zero fill) is left to the generic kernel.
  if (a.K == 0) return false;

  MfmaArgs& m = plan->args;
  m.lhs = a.lhs; m.rhs = a.rhs; m.out = a.out;
  m.lhs_stride_bytes = lhs_stride_bytes;
  m.rhs_stride_bytes = rhs_stride_bytes;
  m.out_stride0 = a.out_stride0;
  m.M = (int32_t)a.M; m.N = (int32_t)a.N; m.K = (int32_t)a.K;
  m.log2_M0 = lm0; m.log2_N0 = ln0;
  m.lhs_rb = lhs_rb; m.rhs_rb = rhs_rb;
  m.log2_lhs_rb = llrb; m.log2_rhs_rb = lrrb;
  m.chunks = (int32_t)(((int64_t)a.K * lhs_rb + 63) / 64);
  m.accumulate = (a.flags & IREE_UK_FLAG_MMT4D_ACCUMULATE) ? 1 : 0;

  // Alignment of every vector access the block kernels make.
  const int lhs_align = gather == 4 ? 4 : 16;  // (also for 1-, 2- and 8-byte pieces: 16 bytes per lane)
  const int rhs_align = i4 ? 8 : lhs_align;
  if (((uintptr_t)a.lhs % lhs_align) || (a.M > 1 && lhs_stride_bytes % lhs_align)) return false;
  if (((uintptr_t)a.rhs % rhs_align) || (a.N > 1 && rhs_stride_bytes % rhs_align)) return false;
  if ((gather == 1 || gather == 2 || gather == 8) && !mfma_direct_covers(m, gather, i4)) return false;
  plan->wave_shape = -1;
  plan->wave_tile = false;
  if (!choose || !wave_k_covers(m, gather, i4)) return true;
  double best = block_cost(m, kind, i4, gather);
  const int shapes = kind == kF32 ? sizeof kWaveKShapesF32 / sizeof(WaveKShape) : sizeof kWaveKShapes / sizeof(WaveKShape);
  for (int s = 0; s < shapes; ++s) {
    const double cost = wave_k_cost(m, kind, i4, gather, wave_k_shape(kind, s));
    if (cost < best) {
      best = cost;
      plan->wave_shape = s;
    }
  }
  plan->wave_tile = wave_tile_covers(m, kind, gather, i4) && wave_tile_is_best(m, i4, plan->wave_shape);
  return true;
}

hipError_t launch_wave_k(const Plan& plan, hipStream_t stream, const char** name) {
  const MfmaArgs& m = plan.args;
  const WaveKShape& shape = wave_k_shape(plan.kind, plan.wave_shape);
  *name = shape.name;
  // Weights that one row of tiles reads once are streamed past the caches like those of a matrix-vector product: bf16 64 x
  // 14336 x 4096 (117 MB) from HBM 28.1 -> 24.7 us, read again or just written 20.2 -> 24.3. With several rows of tiles
  // the caches serve the others: streamed 3 to 20 % slower from HBM too.
  const bool streamed = ((int64_t)m.M << m.log2_M0) <= 16 * shape.fa &&
                        comes_from_hbm(((int64_t)m.N * m.K * m.rhs_rb) << m.log2_N0);
  switch (plan.kind) {
    case kI8: return launch_wave_k_i8(m, plan.gather, plan.rhs_i4, plan.wave_shape, streamed, stream);
    case kF16:
      return plan.narrow ? launch_wave_k_f16_narrow(m, plan.gather, plan.wave_shape, streamed, stream)
                         : launch_wave_k_f16(m, plan.gather, plan.wave_shape, streamed, stream);
    case kBF16:
      return plan.narrow ? launch_wave_k_bf16_narrow(m, plan.gather, plan.wave_shape, streamed, stream)
                         : launch_wave_k_bf16(m, plan.gather, plan.wave_shape, streamed, stream);
    default: return launch_wave_k_f32(m, plan.gather, plan.wave_shape, streamed, stream);
  }
}

hipError_t launch_mfma(const Mmt4dArgs& a, hipStream_t stream, const char** name) {
  Plan plan;
  if (!make_plan(a, false, true, &plan)) return hipErrorInvalidValue;
  const MfmaArgs& m = plan.args;
  if (plan.wave_tile) {
    *name = "mmt4d_mfma_wave_tile";
    return launch_wave_tile(m, plan.kind, plan.rhs_i4, plan.narrow, stream);
  }
  if (plan.wave_shape >= 0) return launch_wave_k(plan, stream, name);
  switch (plan.kind) {
    case kI8: return launch_mfma_i8(m, plan.gather, plan.rhs_i4, stream, name);
    case kF16: return launch_mfma_f16(m, plan.gather, plan.narrow, stream, name);
    case kBF16: return launch_mfma_bf16(m, plan.gather, plan.narrow, stream, name);
    default: return launch_mfma_f32(m, plan.gather, stream, name);
  }
}

}  // namespace

Mmt4dLauncher select_mmt4d_mfma(const Mmt4dArgs& a, bool probe_only) {
  Plan plan;
  return make_plan(a, probe_only, false, &plan) ? launch_mfma : nullptr;
}

}  // namespace uk
