// MFMA mmt4d for problems with few output tiles (batched decode, small layers,
// few rows against a long K): K is split over the wavefronts of a workgroup.
//
// The block kernels (mmt4d_mfma_kernels.h) walk K one 64-byte chunk per
// workgroup barrier, about 150 ns a chunk whatever the tile, and a problem with
// fewer tiles than compute units has nothing to hide that behind. Here a
// workgroup of 8 wavefronts owns a (16*FA) x (16*FB) tile and every wavefront
// multiplies the WHOLE tile over its own share of K: operands go from
// global memory straight to the MFMA's registers, DEPTH - 1 64-byte steps in
// flight while one is multiplied, with no LDS and no barrier until the partial
// tiles are summed through LDS at the end, in wavefront order (results do not
// depend on scheduling). Where the caches hold the operands a workgroup is bound
// by what a compute unit's load path moves, (16*FA + 16*FB) * 64 bytes per step
// at 70 to 90 bytes a nanosecond, f32 by the matrix pipe.
//
// Operand registers. Fragments are 16 rows x 64 bytes of K
// (v_mfma_i32_16x16x64_i8, v_mfma_f32_16x16x32_{f16,bf16}, four
// v_mfma_f32_16x16x4_f32): lane 16*q + r holds 16 bytes of row r. Which k those
// are is free as long as lhs and rhs agree. A load is 16 contiguous bytes per
// lane and covers one fragment's step, 1 KiB. G = bytes of a row piece:
//   16 (or more): lane 16*q + r loads 16-byte column q of row r: the operand.
//   4, as pieces: lane 16*q + r loads the pieces of k steps 4*d + q of row r, d = 0 .. 3, one at a time: 256 contiguous
//     bytes an instruction with 16-row tiles. (wave_k_loads_pieces says when.)
//   8, 4, 2, staged: 16 contiguous bytes are 16 / G rows of one k step. They pass through
//     1 KiB of LDS that only this wavefront uses (no barrier), as [k][16 rows][G
//     bytes], and come back as the pieces of k steps 4*d + q of row r (8, 4: reads
//     linear in the lane number) resp. 16*d + 4*q + {0..3} (2: the transposing
//     read ds_read_b64_tr_b16). (8-byte pieces one at a time: 3 to 15 % slower; the
//     instruction moves half of what the others do.)
//   int4 rhs (K0 = 32 or 64): a step is 128 values of K; a lane's 16 bytes are 32
//     nibbles, widened to two int8 operands of 16x the values, against two
//     16-byte pieces of the lhs; the sums are shifted right by 4 at the end.
// K may end inside a step: what lies beyond K in the last one is zeroed in both
// operands.
#ifndef IREE_AMD_CSRC_MMT4D_WAVE_K_KERNELS_H_
#define IREE_AMD_CSRC_MMT4D_WAVE_K_KERNELS_H_

#include <type_traits>

#define UK_MFMA_KERNEL_BODIES
#include "mmt4d_mfma_kernels.h"

namespace uk {
namespace {

typedef float v4f32 __attribute__((ext_vector_type(4)));

template <int KIND> struct Acc16 { typedef v4f32 type; };
template <> struct Acc16<kI8> { typedef v4i32 type; };

// Product of two 16-row x 64-byte fragments.
template <int KIND>
__device__ __forceinline__ typename Acc16<KIND>::type mfma16(uint4 row_operand, uint4 col_operand,
                                                             typename Acc16<KIND>::type acc) {
  if constexpr (KIND == kI8) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i32, row_operand),
                                                 __builtin_bit_cast(v4i32, col_operand), acc, 0, 0, 0);
  } else if constexpr (KIND == kF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8f16, row_operand),
                                                  __builtin_bit_cast(v8f16, col_operand), acc, 0, 0, 0);
  } else if constexpr (KIND == kBF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf16, row_operand),
                                                   __builtin_bit_cast(v8bf16, col_operand), acc, 0, 0, 0);
  } else {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(row_operand.x), __uint_as_float(col_operand.x), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(row_operand.y), __uint_as_float(col_operand.y), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(row_operand.z), __uint_as_float(col_operand.z), acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(row_operand.w), __uint_as_float(col_operand.w), acc, 0, 0, 0);
  }
}

// 8 bytes per lane from LDS, transposed within each group of 16 lanes (ds_read_b64_tr_b16): the lanes' 8-byte chunks
// are taken as 4 rows of 32 bytes (chunks 4j .. 4j + 3 make row j), and lane i of the group receives the i-th 16-bit
// element of every row.
__device__ __forceinline__ uint2 lds_read_transposed_b16(const uint8_t* p) {
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  const v4i16 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)(p));
  return __builtin_bit_cast(uint2, v);
}

// Operand memory, said to be global: the base comes from scalar registers by way of an integer (uniform_pointer), and from a
// pointer that may lead anywhere the compiler makes flat loads. Those may return in any order and count as LDS accesses too,
// so that the only wait it can put in front of a batch's MFMAs is for every load in flight, the next batch's among them, and
// nothing is prefetched. Nor may the loads' addresses be made on the vector unit, in 64 bits (see load): those additions and
// f32 MFMAs get in each other's way. f32 288 x 1584 x 8128 in 32x64 tiles: flat loads 103 us, global ones with additions in
// front of them 109, with a scalar base and a 32-bit offset 60. bf16 and int8, bound by the loads, 1 to 5 %.
typedef const __attribute__((address_space(1))) uint8_t* global_bytes_t;
typedef const __attribute__((address_space(1))) v4i32* global_v4i32_t;
typedef const __attribute__((address_space(1))) uint32_t* global_u32_t;

// One operand of a workgroup's tile: F fragments, pieces of G bytes. WIDE: the int8 operand that meets an int4 one,
// two 16-byte pieces per fragment and step.
// PIECES: 4-byte pieces are loaded one at a time.
template <int G, int F, bool WIDE, bool PIECES>
struct Operand {
  static constexpr int RAW = WIDE ? 2 * F : F;  // 16-byte registers that hold what one step loads
  global_bytes_t base;   // uniform: the tile's first row of tiles, k = 0
  uint32_t off[F];       // per lane, from base, at step 0
  uint32_t step_bytes;   // from one step to the next
  uint32_t kstep_bytes;  // from one k step to the next
  int32_t k_lane;        // k step (within a step) of what this lane loads
  uint32_t lds_slot;     // staged: where in a fragment's 1 KiB the lane's 16 bytes go

  // What step `s` holds. CHECKED: a lane whose k step (`k0` = the step's first) is not below `K` loads that of K - 1 instead,
  // for zero_beyond to clear: no branches, and nothing that waits for a load in front of the next one.
  // STREAMED: the caller reads every byte once (non-temporal loads).
  template <bool CHECKED, bool STREAMED>
  __device__ __forceinline__ void load(int32_t s, int32_t k0, int32_t K, uint4 (&raw)[RAW]) {
    // (The empty statements keep base and offset apart up to the load: where the compiler widens the offset to 64 bits ahead
    // of the loop, or adds the bases of a step's pieces to it, every load has 64-bit additions in front of it.)
    global_bytes_t at[PIECES ? 4 : 1];
#pragma unroll
    for (int d = 0; d < (PIECES ? 4 : 1); ++d) {
      at[d] = base + (uint64_t)(uint32_t)s * step_bytes + d * (uint64_t)(step_bytes / 4);
      asm volatile("" : "+s"(at[d]));
    }
    int32_t back[PIECES ? 4 : 1];  // bytes (the k steps that a step has are a power of two)
    if constexpr (CHECKED) {
#pragma unroll
      for (int d = 0; d < (PIECES ? 4 : 1); ++d)
        back[d] = max(k0 + k_lane + 4 * d - (K - 1), 0) * (int32_t)kstep_bytes;
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
      asm volatile("" : "+v"(off[f]));
#pragma unroll
      for (int w = 0; w < RAW / F; ++w) {
        uint4& to = raw[(RAW / F) * f + w];
        if constexpr (PIECES) {
          uint32_t piece[4];
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            global_u32_t from = (global_u32_t)(at[d] + off[f]);
            if constexpr (CHECKED) from = (global_u32_t)((global_bytes_t)from - back[d]);
            piece[d] = *from;
          }
          to = make_uint4(piece[0], piece[1], piece[2], piece[3]);
        } else {
          global_v4i32_t from = (global_v4i32_t)(at[0] + off[f] + 16 * w);
          if constexpr (CHECKED) from = (global_v4i32_t)((global_bytes_t)from - back[0]);
          if constexpr (STREAMED) to = __builtin_bit_cast(uint4, __builtin_nontemporal_load(from));
          else to = __builtin_bit_cast(uint4, *from);
        }
      }
    }
  }
  // Clears what a checked load brought from k steps that are not below K.
  __device__ __forceinline__ void zero_beyond(int32_t k0, int32_t K, uint4 (&raw)[RAW]) const {
#pragma unroll
    for (int i = 0; i < RAW; ++i) {
      if constexpr (PIECES) {
        raw[i].x = k0 + k_lane < K ? raw[i].x : 0u;
        raw[i].y = k0 + k_lane + 4 < K ? raw[i].y : 0u;
        raw[i].z = k0 + k_lane + 8 < K ? raw[i].z : 0u;
        raw[i].w = k0 + k_lane + 12 < K ? raw[i].w : 0u;
      } else {
        const bool below = k0 + k_lane < K;
        raw[i] = make_uint4(below ? raw[i].x : 0u, below ? raw[i].y : 0u, below ? raw[i].z : 0u, below ? raw[i].w : 0u);
      }
    }
  }

  // Staged: the loaded 16 bytes of every fragment into the wavefront's LDS, and fragment f back out of it.
  __device__ __forceinline__ void to_lds(const uint4 (&raw)[RAW], uint8_t* lds) const {
#pragma unroll
    for (int f = 0; f < F; ++f) *(uint4*)(lds + 1024 * f + lds_slot) = raw[f];
  }
  __device__ __forceinline__ uint4 from_lds(const uint8_t* lds, int f, int lane) const {
    const uint8_t* p = lds + 1024 * f;
    if constexpr (G == 8) {
      const uint2 lo = *(const uint2*)(p + 8 * lane), hi = *(const uint2*)(p + 512 + 8 * lane);
      return make_uint4(lo.x, lo.y, hi.x, hi.y);
    } else if constexpr (G == 4) {
      return make_uint4(*(const uint32_t*)(p + 4 * lane), *(const uint32_t*)(p + 256 + 4 * lane),
                        *(const uint32_t*)(p + 512 + 4 * lane), *(const uint32_t*)(p + 768 + 4 * lane));
    } else {
      const uint2 lo = lds_read_transposed_b16(p + 8 * lane), hi = lds_read_transposed_b16(p + 512 + 8 * lane);
      return make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
  }
};

template <int KIND, bool RHS_I4, bool NARROW, int G, int FA, int FB, int WAVES, int DEPTH, bool STREAMED, bool PIECES>
__global__ __launch_bounds__(64 * WAVES)
__attribute__((amdgpu_waves_per_eu(2, FA * FB >= 16 ? 2 : 4)))
void mmt4d_wave_k_kernel(const MfmaArgs a) {
  typedef typename Acc16<KIND>::type acc_t;
  typedef Operand<G, FA, RHS_I4, PIECES> lhs_t;
  typedef Operand<G, FB, false, PIECES> rhs_t;
  static_assert(!PIECES || (G == 4 && !STREAMED), "4-byte pieces, which are read through the caches");
  constexpr bool STAGED = G < 16 && !PIECES;  // operands pass through LDS
  static_assert(!RHS_I4 || (KIND == kI8 && G == 16), "int4 rhs");
  // The wavefronts' staging of narrow row pieces, [WAVES][FA + FB][1 KiB]; then [WAVES][FA * FB][64] partial sums.
  extern __shared__ uint4 ring[];

  fetch_arguments(a);
  int tile_row, tile_col;
  if (!locate_block(a, &tile_row, &tile_col)) return;
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t total_rows = (int64_t)a.M << a.log2_M0, total_cols = (int64_t)a.N << a.log2_N0;
  const int64_t first_row = (int64_t)tile_row * (16 * FA), first_col = (int64_t)tile_col * (16 * FB);

  // Tiles past the end of the matrix are redirected to its last one: computed, never stored. (32 bits: offsets from the
  // workgroup's first tile, which the plan has checked. This runs once, in front of the first load.)
  auto set_up = [&](auto& op, const uint8_t* base, int64_t first, int32_t tiles, int log2_t0, int64_t stride, int32_t rb,
                    int log2_rb, int32_t lane_bytes) {
    const uint32_t kstep = (uint32_t)rb << log2_t0;
    const int32_t first_tile = (int32_t)(first >> log2_t0);
    const int32_t last_tile = tiles - 1 - first_tile;
    op.base = (global_bytes_t)uniform_pointer(base + first_tile * stride);
    op.step_bytes = (uint32_t)(4 * lane_bytes) << log2_t0;
    op.kstep_bytes = kstep;
    int32_t row;  // of the fragment
    uint32_t lane_off;
    if constexpr (PIECES) {
      row = r;
      op.k_lane = q;
      lane_off = (uint32_t)q << (log2_rb + log2_t0);
      op.lds_slot = 0;
    } else if constexpr (G == 16) {
      row = r;
      op.k_lane = (lane_bytes * q) >> log2_rb;
      lane_off = ((uint32_t)op.k_lane << (log2_rb + log2_t0)) + ((lane_bytes * q) & (rb - 1));
      op.lds_slot = 0;
    } else {
      // Lanes go along a tile's step (64 bytes per row, contiguous), then to the fragment's next tile.
      const int32_t in_tile = lane & ((4 << log2_t0) - 1);
      const int32_t log2_lanes_per_kstep = log2_t0 + log2_rb - 4;  // (16 bytes of one k step at least: the host's check)
      const int32_t group = in_tile & ((1 << log2_lanes_per_kstep) - 1);
      op.k_lane = in_tile >> log2_lanes_per_kstep;
      row = ((lane >> (2 + log2_t0)) << log2_t0) + group * (16 / G);
      lane_off = (uint32_t)op.k_lane << (log2_rb + log2_t0);
      op.lds_slot = (uint32_t)(op.k_lane * 16 + row) * G;
    }
#pragma unroll
    for (int f = 0; f < (int)(sizeof op.off / sizeof op.off[0]); ++f) {
      const int32_t tile = min((16 * f + row) >> log2_t0, last_tile);
      op.off[f] = (uint32_t)tile * (uint32_t)stride + ((uint32_t)(row & ((1 << log2_t0) - 1)) << log2_rb) + lane_off;
    }
  };
  lhs_t lhs;
  rhs_t rhs;
  set_up(lhs, a.lhs, first_row, a.M, a.log2_M0, a.lhs_stride_bytes, a.lhs_rb, a.log2_lhs_rb, RHS_I4 ? 32 : 16);
  set_up(rhs, a.rhs, first_col, a.N, a.log2_N0, a.rhs_stride_bytes, a.rhs_rb, a.log2_rhs_rb, 16);
  uint8_t* const staging = (uint8_t*)ring + wave * ((FA + FB) * 1024);  // (narrow pieces only)

  acc_t acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  // The steps are dealt out to the wavefronts in turn: at any time the workgroup reads one contiguous stretch of every row
  // panel. (A contiguous share of K per wavefront puts all loads of a launch at the same few offsets modulo the share: 5 to
  // 10 % slower.)
  static_assert(WAVES == 8, "a shift by three");
  const int32_t log2_ksteps = (RHS_I4 ? 7 : 6) - a.log2_lhs_rb, ksteps_per_step = 1 << log2_ksteps;
  const int32_t steps = (a.K + ksteps_per_step - 1) >> log2_ksteps;
  const int32_t whole = a.K >> log2_ksteps;
  const int32_t count = (whole - wave + WAVES - 1) >> 3;

  struct Step {
    uint4 l[lhs_t::RAW], r[rhs_t::RAW];
  };
  auto fetch = [&](int32_t b, Step& to) {
    rhs.template load<false, STREAMED>(b * WAVES + wave, 0, 0, to.r);
    lhs.template load<false, false>(b * WAVES + wave, 0, 0, to.l);
  };
  // A step that K ends in goes to the last wavefront. Staged, on the tiles of two fragments, it is loaded ahead of all others:
  // loaded behind them it came an almost whole latency late, which few steps do not hide (f16 8 x 22064 x 530, 8x16x1 tiles
  // 7.9 -> 7.1 us, x 793 9.0 -> 8.8, bf16 8x8x4 136 x 760 x 784 3.74 -> 3.48). Its registers cost the other forms up to 5 %.
  constexpr bool REST_FIRST = STAGED && FA * FB == 2;
  const bool has_rest = wave == WAVES - 1 && whole < steps;
  auto fetch_rest = [&](Step& to) {
    rhs.template load<true, false>(whole, whole * ksteps_per_step, a.K, to.r);
    lhs.template load<true, false>(whole, whole * ksteps_per_step, a.K, to.l);
  };
  auto zero_rest = [&](Step& of) {
    rhs.zero_beyond(whole * ksteps_per_step, a.K, of.r);
    lhs.zero_beyond(whole * ksteps_per_step, a.K, of.l);
  };
  auto multiply = [&](const Step& from) {
    if constexpr (STAGED) {
      lhs.to_lds(from.l, staging);
      rhs.to_lds(from.r, staging + FA * 1024);
      __builtin_amdgcn_wave_barrier();
    }
    if constexpr (RHS_I4) {
#pragma unroll
      for (int j = 0; j < FB; ++j) {
        const uint4 w = from.r[j];
        const uint4 lo = widen_i4_times16(make_uint2(w.x, w.y)), hi = widen_i4_times16(make_uint2(w.z, w.w));
#pragma unroll
        for (int i = 0; i < FA; ++i) {
          acc[i][j] = mfma16<KIND>(lo, from.l[2 * i], acc[i][j]);
          acc[i][j] = mfma16<KIND>(hi, from.l[2 * i + 1], acc[i][j]);
        }
      }
    } else {
      uint4 fa[FA];
#pragma unroll
      for (int i = 0; i < FA; ++i) {
        if constexpr (STAGED) fa[i] = lhs.from_lds(staging, i, lane); else fa[i] = from.l[i];
      }
#pragma unroll
      for (int j = 0; j < FB; ++j) {
        uint4 fb;
        if constexpr (STAGED) fb = rhs.from_lds(staging + FA * 1024, j, lane); else fb = from.r[j];
#pragma unroll
        for (int i = 0; i < FA; ++i) acc[i][j] = mfma16<KIND>(fb, fa[i], acc[i][j]);
      }
    }
  };
  if constexpr (DEPTH > 2) {
    // A ring: each step's registers are loaded again as soon as they are multiplied. What is left at the end, any number of
    // steps, is one batch of loads.
    Step ring_of[DEPTH], rest;
    if (has_rest) fetch_rest(rest);
    int32_t b = 0;
    if (count >= DEPTH) {
#pragma unroll
      for (int u = 0; u < DEPTH; ++u) fetch(u, ring_of[u]);
      b = DEPTH;
      for (; b + DEPTH <= count; b += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
          multiply(ring_of[u]);
          __builtin_amdgcn_sched_barrier(0);
          fetch(b + u, ring_of[u]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int u = 0; u < DEPTH; ++u) {
        multiply(ring_of[u]);
        if (b + u < count) fetch(b + u, ring_of[u]);
      }
    } else {
#pragma unroll
      for (int u = 0; u < DEPTH - 1; ++u)
        if (u < count) fetch(u, ring_of[u]);
    }
#pragma unroll
    for (int u = 0; u < DEPTH - 1; ++u)
      if (b + u < count) multiply(ring_of[u]);
    if (has_rest) {
      zero_rest(rest);
      multiply(rest);
    }
  } else {
    Step p, n, rest;
    if (REST_FIRST && has_rest) fetch_rest(rest);
    const bool rest_last = !REST_FIRST && has_rest;
    int32_t b = 0;
    if (count > 0) {
      fetch(0, p);
      for (; b + 2 < count; b += 2) {
        fetch(b + 1, n);
        __builtin_amdgcn_sched_barrier(0);
        multiply(p);
        __builtin_amdgcn_sched_barrier(0);
        fetch(b + 2, p);
        __builtin_amdgcn_sched_barrier(0);
        multiply(n);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (b + 1 < count) {
        fetch(b + 1, n);
        multiply(p);
        if (rest_last) fetch_rest(p);
        multiply(n);
        if (rest_last) {
          zero_rest(p);
          multiply(p);
        }
      } else {
        if (rest_last) fetch_rest(n);
        multiply(p);
        if (rest_last) {
          zero_rest(n);
          multiply(n);
        }
      }
    } else if (rest_last) {
      fetch_rest(p);
      zero_rest(p);
      multiply(p);
    }
    if (REST_FIRST && has_rest) {
      zero_rest(rest);
      multiply(rest);
    }
  }

  if constexpr (STAGED) __syncthreads();  // the staging memory takes the partial sums
  acc_t* partial = (acc_t*)ring;
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) partial[(wave * (FA * FB) + i * FB + j) * 64 + lane] = acc[i][j];
  __syncthreads();

  // The sums, and the output: lane 16*q + r of fragment (i, j) holds lhs row r and rhs rows 4*q .. 4*q + 3 of the
  // fragments, four consecutive j0 of one output row.
  const int32_t M0 = 1 << a.log2_M0, N0 = 1 << a.log2_N0;
  auto total_of = [&](int f) -> acc_t {
    acc_t v = partial[f * 64 + lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += partial[(w * (FA * FB) + f) * 64 + lane];
    if constexpr (RHS_I4) v = acc_t{v.x >> 4, v.y >> 4, v.z >> 4, v.w >> 4};
    return v;
  };
  auto store_quad = [&](int64_t row, int64_t col, acc_t v) {
    if (row >= total_rows || col >= total_cols) return;
    const int64_t index = (row >> a.log2_M0) * a.out_stride0 + ((col >> a.log2_N0) << (a.log2_M0 + a.log2_N0)) +
                          ((row & (M0 - 1)) << a.log2_N0) + (col & (N0 - 1));
    if constexpr (NARROW) {
      constexpr int EBITS = KIND == kF16 ? 5 : 8;
      uint2* dst = (uint2*)(a.out + 2 * index);
      if (a.accumulate) {
        const uint2 old = *dst;
        v += acc_t{widen16_first<EBITS>(old.x), widen16_second<EBITS>(old.x), widen16_first<EBITS>(old.y), widen16_second<EBITS>(old.y)};
      }
      *dst = make_uint2(narrow16_pair<EBITS>(v.x, v.y), narrow16_pair<EBITS>(v.z, v.w));
    } else {
      acc_t* dst = (acc_t*)(a.out + 4 * index);
      if (a.accumulate) v += *dst;
      *dst = v;
    }
  };
  for (int f = wave; f < FA * FB; f += WAVES) {
    const int i = f / FB, j = f % FB;
    store_quad(first_row + 16 * i + r, first_col + 16 * j + 4 * q, total_of(f));
  }
}

template <int KIND, bool RHS_I4, bool NARROW, int G, int FA, int FB, int WAVES, int DEPTH, bool PIECES>
hipError_t launch_wave_k_loads(MfmaArgs m, bool streamed, hipStream_t stream) {
  unsigned grid;
  set_tile_grid(&m, 16 * FA, 16 * FB, &grid);
  constexpr int staging_kib = G < 16 && !PIECES ? WAVES * (FA + FB) : 0, partial_kib = WAVES * FA * FB;
  constexpr int lds_bytes = 1024 * (staging_kib > partial_kib ? staging_kib : partial_kib);
  static_assert(lds_bytes <= 160 * 1024, "partial sums do not fit the LDS");
  auto kernel = mmt4d_wave_k_kernel<KIND, RHS_I4, NARROW, G, FA, FB, WAVES, DEPTH, false, PIECES>;
  if constexpr (G == 16) {
    if (streamed) kernel = mmt4d_wave_k_kernel<KIND, RHS_I4, NARROW, G, FA, FB, WAVES, DEPTH, true, PIECES>;
  }
  if (lds_bytes > 65536) {
    const hipError_t attr = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (attr != hipSuccess) return attr;
  }
  return launch_kernel<MfmaArgs>(kernel, grid, 64 * WAVES, lds_bytes, stream, m);
}

template <int KIND, bool RHS_I4, bool NARROW, int G, int FA, int FB, int WAVES, int DEPTH>
hipError_t launch_wave_k_tile(const MfmaArgs& m, bool streamed, hipStream_t stream) {
  if constexpr (G != 4) {
    return launch_wave_k_loads<KIND, RHS_I4, NARROW, G, FA, FB, WAVES, DEPTH, false>(m, streamed, stream);
  } else if constexpr (KIND == kF32) {
    return launch_wave_k_loads<KIND, RHS_I4, NARROW, G, FA, FB, WAVES, DEPTH, true>(m, streamed, stream);
  } else {
    return wave_k_loads_pieces(m, KIND, G, FA, FB)
               ? launch_wave_k_loads<KIND, RHS_I4, NARROW, G, FA, FB, WAVES, DEPTH, true>(m, streamed, stream)
               : launch_wave_k_loads<KIND, RHS_I4, NARROW, G, FA, FB, WAVES, DEPTH, false>(m, streamed, stream);
  }
}

// One 64-byte step of K in flight ahead of the one that is multiplied, for each of eight wavefronts. With one fragment either
// way that step is multiplied before the next one is there, and a long K has two in flight: f16 16x16x1 16 x 560 x 7148 8.7
// -> 7.6 us, f32 32 x 352 x 8740 15.5 -> 13.5, bf16 16 x 1360 x 6576 7.2 -> 7.0. With fewer steps the ring's longer code
// costs more than it hides. Two ahead against one, 144 problems, on operands that every launch reads again, that the
// last-level cache holds and from HBM: 36 to 48 chunks of 64 bytes 6 % slower, 2 % slower and level, 48 to 100 4 % slower,
// level and 2 % faster, more 2 % slower, 4 and 6 % faster; f32 from 28 to 48 chunks 1 % slower, 2 and 3 % faster, to 100 4 %
// slower, 2 and 5 % faster, beyond 1 % slower, 7 and 7 % faster; 4-byte pieces from 28 to 48 chunks level, 1 and 1 % faster.
// (48 x 560 x 1640 f16 in 16x16x1 tiles, 52 chunks, from HBM 5.25 us with one, 4.92 with two.) int8 in 16-byte pieces 1 % slower; three and more, or two for larger tiles, give nothing.
template <int KIND, int G>
bool two_steps_ahead(const MfmaArgs& m) { return m.chunks >= (KIND == kF32 || G == 4 ? 32 : 48); }

template <int KIND, bool RHS_I4, bool NARROW, int G>
hipError_t launch_wave_k_piece(const MfmaArgs& m, int shape, bool streamed, hipStream_t stream) {
  switch (shape) {
    case 0:
      if constexpr (KIND != kI8 || G < 16) {
        if (two_steps_ahead<KIND, G>(m)) return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 1, 1, 8, 3>(m, streamed, stream);
      }
      return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 1, 1, 8, 2>(m, streamed, stream);
    case 1: return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 1, 2, 8, 2>(m, streamed, stream);
    case 2: return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 2, 2, 8, 2>(m, streamed, stream);
    case 3: return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 2, 4, 8, 2>(m, streamed, stream);
    case 4: return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 4, 2, 8, 2>(m, streamed, stream);
    case 5: return launch_wave_k_tile<KIND, RHS_I4, NARROW, G, 4, 4, 8, 2>(m, streamed, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace
}  // namespace uk

#endif  // IREE_AMD_CSRC_MMT4D_WAVE_K_KERNELS_H_
