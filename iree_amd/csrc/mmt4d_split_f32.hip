// MFMA mmt4d for f32 on the bf16 matrix pipe: every value is split into three
// bf16 pieces, and a product is six products of pieces.
//
// The f32 MFMAs run at a sixteenth of the bf16 ones' rate, and f32 products are
// bound by them whatever the tile (mmt4d_wave_k_kernels.h). hi = x to the nearest
// bf16, mid = x - hi, lo = x - hi - mid are exact to 24 bits; of the nine
// products of two values' pieces lo*lo, lo*mid and mid*lo are below 2^-26 of the
// whole one and are left out. The other six are six MFMAs for 16 values of K
// where f32 takes eight of twice the time each: 2.7 times the rate, less the
// splitting. hi*hi has accumulators of its own, the five small ones others, so
// that a sum is rounded once in 16 values of K where the f32 MFMA rounds every
// two: against a 64-bit product the error is 1/3 to 2/3 of the f32 kernels' (N(0, 1),
// relative: K = 1000 8e-8 and 9.6e-8 in the two tiles, f32 2.1e-7; K = 4096
// 1.4e-7, 1.9e-7, 4.1e-7).
//
// What the pieces cannot hold is left to f32 MFMAs: a workgroup that finds a
// value other than zero below 2^-100, whose lo may be too small for bf16, or a
// sum that is no finite number (an infinity splits into infinity and NaN, a value
// above the largest bf16 rounds to one) computes its tile again with them. Such
// tiles take the time of both: with one such value in every tile 1024 x 2048 x 2048
// takes 115 us where the f32 kernel takes 64, 432 x 1936 x 3096 87 where it takes 45.
//
// The rest is mmt4d_wave_tile.hip's: wavefronts multiply the whole tile over
// K in turns of 64 bytes (16 values), operands straight from global memory in registers,
// buffer loads that read nothing where there is nothing, partial tiles summed by
// halves. A step multiplies the pieces of one turn while the next one's values are
// split, a pair of them every two or three MFMAs, and the values behind those
// are loaded. What bounds it is the vector unit: 14 instructions for a pair of
// values, 7 a value with everything, and an MFMA keeps it from issuing for 16 of its 32
// cycles; 64x128 takes 1.2 us a step of four turns of 64 bytes, 64x64 1.2 of
// eight. (The values less their pieces by v_dot2c_f32_bf16, 4 instructions fewer a pair: 10 to
// 20 % slower. Pieces cut off instead of rounded, 16 instructions of the plainest
// kind: 5 % slower. Everything in one accumulator, 96x128 tiles: error 1.2 times the f32
// kernels'.)
//
//   64x128, four wavefronts, one a SIMD: 512 x 4032 x 960 37.8 -> 28.4 us, 784 x 2304 x 2320 74.9 ->
//     55.0, 1472 x 3904 x 652 77.1 -> 62.6
//   64x64, eight wavefronts: 432 x 1936 x 3096 45.8 -> 36.8, 176 x 4864 x 2497 (4-byte pieces)
//     41.0 -> 34.0
#include <type_traits>

#define UK_MFMA_KERNEL_BODIES
#include "mmt4d_mfma_kernels.h"

namespace uk {
namespace {

typedef float v2f32 __attribute__((ext_vector_type(2)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef __bf16 v2bf16 __attribute__((ext_vector_type(2)));

// Two floats to bf16, to nearest even, the first in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f32{a, b}, v2bf16));
}
__device__ __forceinline__ float low_bf16(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_bf16(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }

// One operand of the workgroup's tile, F fragments of 32 rows.
template <int G, int F>
struct SplitOperand {
  static constexpr int LOADS = G == 16 ? 2 : 8;  // of a fragment and step
  const uint8_t* base;  // uniform: the tile's first row of tiles, k = 0
  uint32_t off[F];      // per lane, from base
  uint32_t step_bytes;  // from one step to the next
  uint32_t half_bytes;  // from a step's first half to its second
  uint32_t at;          // uniform: bytes from base to the step that is loaded next

  // Where `records` is 0 the loads read nothing and give zeros.
  __device__ __forceinline__ void load(int f, uint32_t from, int32_t records, float (&raw)[8]) const {
    const auto memory = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, records, 0x00020000);
    if constexpr (G == 16) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint4 v = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(memory, off[f], from + u * half_bytes, 0));
        raw[4 * u] = __uint_as_float(v.x);
        raw[4 * u + 1] = __uint_as_float(v.y);
        raw[4 * u + 2] = __uint_as_float(v.z);
        raw[4 * u + 3] = __uint_as_float(v.w);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t)
        raw[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(memory, off[f], from + t * (step_bytes >> 3), 0));
    }
  }
};

// Fragments of partial sums that the LDS holds: half of the tile from every wavefront, then half of that, and so on.
constexpr int partial_fragments(int fa, int fb, int waves) { return fb == 4 ? waves * fa * 3 : waves * 4; }

template <int G, int FA, int FB, int WAVES>
__device__ __forceinline__ void split_f32_tile(const MfmaArgs& a) {
  constexpr int F = FA + FB, LOG2_WAVES = WAVES == 8 ? 3 : 2;
  extern __shared__ uint4 partial[];

  fetch_arguments(a);
  int tile_row, tile_col;
  if (!locate_block(a, &tile_row, &tile_col)) return;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t total_rows = (int64_t)a.M << a.log2_M0, total_cols = (int64_t)a.N << a.log2_N0;
  const int64_t first_row = (int64_t)tile_row * (32 * FA), first_col = (int64_t)tile_col * (32 * FB);
  // Fragment j of the rhs is number j ^ swap of the tile.
  const int swap = FB == 4 ? wave & 3 : (wave >> 1) & 1;
  const int row_swap = FB == 4 ? 0 : wave >> 2;

  const int log2_ksteps = 6 - a.log2_lhs_rb;
  const int32_t cut = (a.chunks << log2_ksteps) - a.K;  // k steps that K lacks to whole steps

  auto set_up = [&](auto& op, const uint8_t* base, int64_t first, int32_t tiles, int log2_t0, int64_t stride, int log2_rb, int swap) {
    const int32_t first_tile = (int32_t)(first >> log2_t0), last_tile = tiles - 1 - first_tile;
    op.base = uniform_pointer(base + first_tile * stride);
    op.step_bytes = 64u << log2_t0;
    op.half_bytes = ((32u >> log2_rb) << (log2_rb + log2_t0)) + (32 & ((1 << log2_rb) - 1));
    op.at = wave * op.step_bytes - ((uint32_t)cut << (log2_rb + log2_t0));
    const uint32_t in_step = G * h;
    const uint32_t lane_off = ((in_step >> log2_rb) << (log2_rb + log2_t0)) + (in_step & ((1 << log2_rb) - 1));
#pragma unroll
    for (int f = 0; f < (int)(sizeof op.off / sizeof op.off[0]); ++f) {
      const int32_t row = 32 * (f ^ swap) + r, tile = row >> log2_t0;
      const uint32_t off = (uint32_t)tile * (uint32_t)stride + ((uint32_t)(row & ((1 << log2_t0) - 1)) << log2_rb) + lane_off;
      op.off[f] = tile <= last_tile ? off : 0x80000000u;
    }
  };
  SplitOperand<G, FA> lhs;
  SplitOperand<G, FB> rhs;
  set_up(lhs, a.lhs, first_row, a.M, a.log2_M0, a.lhs_stride_bytes, a.log2_lhs_rb, row_swap);
  set_up(rhs, a.rhs, first_col, a.N, a.log2_N0, a.rhs_stride_bytes, a.log2_rhs_rb, swap);
  const uint32_t lhs_start = lhs.at, rhs_start = rhs.at;

  const int32_t count = (a.chunks - wave + WAVES - 1) >> LOG2_WAVES;
  int32_t left;  // steps of the wavefront that are not loaded
  float raw[F][8];
  // Loads fragment f of the step at lhs.at, rhs.at, or nothing when none is left.
  auto load = [&](int f, uint32_t lhs_at, uint32_t rhs_at) {
    int32_t records = -left;
    asm("s_ashr_i32 %0, %0, 31\n\ts_and_b32 %0, %0, 0x80000000" : "+s"(records) : : "scc");
    if (f < FA) lhs.load(f, lhs_at, records, raw[f]);
    else rhs.load(f - FA, rhs_at, records, raw[f]);
  };
  auto next_step = [&]() {
    lhs.at += WAVES * lhs.step_bytes;
    rhs.at += WAVES * rhs.step_bytes;
    --left;
  };
  auto load_first = [&]() {
    left = count;
    lhs.at = lhs_start;
    rhs.at = rhs_start;
#pragma unroll
    for (int f = 0; f < F; ++f) load(f, wave == 0 ? 0 : lhs.at, wave == 0 ? 0 : rhs.at);
    next_step();
    if (wave == 0 && cut != 0) {
      const int32_t whole = (1 << log2_ksteps) - cut;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const bool keep = (G == 16 ? (32 * (t >> 2) + 16 * h) >> a.log2_lhs_rb : 2 * t + h) < whole;
#pragma unroll
        for (int f = 0; f < F; ++f) raw[f][t] = keep ? raw[f][t] : 0.0f;
      }
    }
  };

  v16f32 acc[FA][FB], rest[FA][FB];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < FB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = rest[i][j][e] = 0;
  };

  uint32_t smallest = 0xFFFFFFFFu;
  struct Pieces {
    uint32_t p[F][3][4];
  };
  auto split_pair = [&](int f, int t, Pieces& to) {
    const float x0 = raw[f][2 * t], x1 = raw[f][2 * t + 1];
    const uint32_t hi = pack_bf16(x0, x1);
    const float r0 = x0 - low_bf16(hi), r1 = x1 - high_bf16(hi);
    const uint32_t mid = pack_bf16(r0, r1);
    to.p[f][0][t] = hi;
    to.p[f][1][t] = mid;
    to.p[f][2][t] = pack_bf16(r0 - low_bf16(mid), r1 - high_bf16(mid));
    smallest = min(min(smallest, 2 * __float_as_uint(x0) - 1), 2 * __float_as_uint(x1) - 1);
  };
  auto piece = [&](const Pieces& of, int f, int n) {
    return make_uint4(of.p[f][n][0], of.p[f][n][1], of.p[f][n][2], of.p[f][n][3]);
  };

  // Multiplies one step while the next one, loaded, is split and the one behind it is loaded.
  auto step = [&](const Pieces& now, Pieces& next) {
    constexpr int LHS_PIECE[6] = {2, 0, 1, 1, 0, 0}, RHS_PIECE[6] = {0, 2, 1, 0, 1, 0};
    constexpr int MULTIPLIES = 6 * FA * FB, PAIRS = 4 * F;
    const uint32_t lhs_at = lhs.at, rhs_at = rhs.at;
    int t = 0;
#pragma unroll
    for (int j = 0; j < FB; ++j) {
#pragma unroll
      for (int n = 0; n < 6; ++n) {
#pragma unroll
        for (int i = 0; i < FA; ++i) {
          v16f32& to = n == 5 ? acc[i][j] : rest[i][j];
          to = mfma<kBF16>(piece(now, FA + j, RHS_PIECE[n]), piece(now, i, LHS_PIECE[n]), to);
#pragma unroll
          for (int p = t * PAIRS / MULTIPLIES; p < (t + 1) * PAIRS / MULTIPLIES; ++p) {
            split_pair(p >> 2, p & 3, next);
            if ((p & 3) == 3) load(p >> 2, lhs_at, rhs_at);
          }
          __builtin_amdgcn_sched_barrier(0);
          ++t;
        }
      }
    }
    next_step();
  };

  // Sums over the wavefronts.
  auto put = [&](int slot, const v16f32& v) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *(v4f32*)(partial + (slot * 4 + e) * 64 + lane) = v4f32{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
  };
  auto add = [&](int slot, v16f32& v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const v4f32 p = *(const v4f32*)(partial + (slot * 4 + e) * 64 + lane);
#pragma unroll
      for (int x = 0; x < 4; ++x) v[4 * e + x] += p[x];
    }
  };
  constexpr int OWN = FB == 4 ? FA : 1;  // fragments that the wavefront has the sums of in the end
  auto sum = [&]() {
#pragma unroll
    for (int j = FB - 1; j >= 0; --j)
#pragma unroll
      for (int i = FA - 1; i >= 0; --i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += rest[i][j][e];
        if (FB == 4 ? j >= 2 : i >= 1) put(FB == 4 ? (wave * FA + i) * 2 + j - 2 : wave * 2 + j, acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    __syncthreads();
    if constexpr (FB == 4) {
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) add(((wave ^ 2) * FA + i) * 2 + j, acc[i][j]);
      constexpr int SECOND = WAVES * FA * 2;
#pragma unroll
      for (int i = 0; i < FA; ++i) put(SECOND + wave * FA + i, acc[i][1]);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < FA; ++i) add(SECOND + (wave ^ 1) * FA + i, acc[i][0]);
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) add((wave ^ 4) * 2 + j, acc[0][j]);
      put(WAVES * 2 + wave, acc[0][1]);
      __syncthreads();
      add(WAVES * 2 + (wave ^ 2), acc[0][0]);
      put(WAVES * 3 + wave, acc[0][0]);
      __syncthreads();
      add(WAVES * 3 + (wave ^ 1), acc[0][0]);
    }
  };
  uint32_t* const flags = (uint32_t*)(partial + partial_fragments(FA, FB, WAVES) * 256);

  clear();
  load_first();
  if (count > 0) {
    Pieces p, n;
    auto split_first = [&](Pieces& to) {
#pragma unroll
      for (int f = 0; f < F; ++f) {
#pragma unroll
        for (int t = 0; t < 4; ++t) split_pair(f, t, to);
        load(f, lhs.at, rhs.at);
      }
      next_step();
    };
    // An odd number of steps: the first one ahead of the loop, or a step of zeros behind it where registers are short (leaving
    // the loop in the middle makes the register allocator move the accumulators through memory).
    constexpr bool ODD_FIRST = WAVES == 4 || G == 4;
    const int32_t odd = ODD_FIRST ? count & 1 : 0;
    if (odd) {
      split_first(n);
      step(n, p);
    } else {
      split_first(p);
    }
    for (int32_t s = odd; s < count; s += 2) {
      step(p, n);
      step(n, p);
    }
  }

  // Where the wavefront's sums go, and what an accumulating call finds there, asked for ahead of the sums if registers allow.
  constexpr bool OLD_FIRST = WAVES == 8;
  const int32_t M0 = 1 << a.log2_M0, N0 = 1 << a.log2_N0;
  auto place = [&](int i, int e, v4f32** to) {
    const int64_t row = first_row + 32 * (i ^ row_swap) + r, col = first_col + 32 * swap + 8 * e + 4 * h;
    *to = (v4f32*)a.out + ((row >> a.log2_M0) * a.out_stride0 + ((col >> a.log2_N0) << (a.log2_M0 + a.log2_N0)) +
                           ((row & (M0 - 1)) << a.log2_N0) + (col & (N0 - 1))) / 4;
    return row < total_rows && col < total_cols && (WAVES == 4 || e >> 1 == (wave & 1));
  };
  v4f32 old[OWN][4];
  if (OLD_FIRST && a.accumulate) {
#pragma unroll
    for (int i = 0; i < OWN; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v4f32* from;
        if (place(i, e, &from)) old[i][e] = *from;
      }
  }

  sum();
  {
    float finite = 0;
#pragma unroll
    for (int i = 0; i < OWN; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) finite = __builtin_fmaf(acc[i][0][e], 0.0f, finite);
    const bool redo = smallest < 2 * (27u << 23) - 1 || !(finite == 0.0f);
    flags[wave] = __builtin_amdgcn_ballot_w64(redo) != 0;
  }
  __syncthreads();
  uint32_t redo = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) redo |= flags[w];
  if (__builtin_amdgcn_readfirstlane(redo)) {
    clear();
    load_first();
    for (int32_t s = 0; s < count; ++s) {
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < FA; ++i)
#pragma unroll
          for (int j = 0; j < FB; ++j)
            if (t & 1) rest[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(raw[FA + j][t], raw[i][t], rest[i][j], 0, 0, 0);
            else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(raw[FA + j][t], raw[i][t], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int f = 0; f < F; ++f) load(f, lhs.at, rhs.at);
      next_step();
    }
    sum();
  }

#pragma unroll
  for (int i = 0; i < OWN; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v4f32* to;
      if (!place(i, e, &to)) continue;
      v4f32 v = {acc[i][0][4 * e], acc[i][0][4 * e + 1], acc[i][0][4 * e + 2], acc[i][0][4 * e + 3]};
      if (a.accumulate) v += OLD_FIRST ? old[i][e] : *to;
      *to = v;
    }
  }
}

template <int G>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void mmt4d_mfma_split_f32_64x64_kernel(const MfmaArgs a) {
  split_f32_tile<G, 2, 2, 8>(a);
}

template <int G>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mmt4d_mfma_split_f32_64x128_kernel(const MfmaArgs a) {
  split_f32_tile<G, 2, 4, 4>(a);
}

template <int FA, int FB, int WAVES>
hipError_t launch_tile(MfmaArgs m, void (*kernel)(const MfmaArgs), hipStream_t stream) {
  unsigned grid;
  set_tile_grid(&m, 32 * FA, 32 * FB, &grid);
  constexpr int lds_bytes = 4096 * partial_fragments(FA, FB, WAVES) + 4 * WAVES;
  static_assert(lds_bytes <= 160 * 1024, "partial sums do not fit the LDS");
  const hipError_t attr = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  if (attr != hipSuccess) return attr;
  return launch_kernel<MfmaArgs>(kernel, grid, 64 * WAVES, lds_bytes, stream, m);
}

}  // namespace

hipError_t launch_split_f32(const MfmaArgs& m, int gather, int shape, hipStream_t stream, const char** name) {
  if (shape == 0) {
    *name = "mmt4d_mfma_split_f32_64x64";
    return launch_tile<2, 2, 8>(m, gather == 16 ? mmt4d_mfma_split_f32_64x64_kernel<16> : mmt4d_mfma_split_f32_64x64_kernel<4>, stream);
  }
  *name = "mmt4d_mfma_split_f32_64x128";
  return launch_tile<2, 4, 4>(m, gather == 16 ? mmt4d_mfma_split_f32_64x128_kernel<16> : mmt4d_mfma_split_f32_64x128_kernel<4>, stream);
}

}  // namespace uk
