// MFMA mmt4d for products of about one large tile per compute unit: every
// wavefront multiplies the workgroup's WHOLE tile over every fourth 64 bytes of
// K, its operands straight from global memory in its own registers.
//
// The block kernels (mmt4d_mfma_kernels.h) bring both operands through LDS,
// where each row is read by two wavefronts: 48 KiB of LDS traffic per 64 bytes
// of K of a 128x128 tile, and a barrier. Where a wavefront has a tile of its own
// nothing is shared until the four partial tiles are summed, and the operands
// are loaded once a workgroup all the same. What a wavefront needs for that is
// the register file of a SIMD: 256 accumulators of a 128x128 tile and two steps
// of 64 bytes of K (128 registers). It is mmt4d_wave_k_kernel's split of K
// (mmt4d_wave_k_kernels.h), with tiles that the eight wavefronts there have no
// registers for. A step is bound by the matrix pipe at the clock that the data
// leaves it: 0.8 us for four chunks of 64 bytes of bf16 N(0, 1) in 128x128
// tiles, 0.6 of zeros.
//
//   128x128, 16-bit operands: bf16 784 x 4112 x 4096 34.0 -> 31.9 us, 1744 x
//     2112 x 3392 31.9 -> 29.8, 2976 x 1232 x 4024 35.1 -> 32.7, accumulating 1312
//     x 2432 x 2248 24.6 -> 22.3; operands and output from HBM 592 x 6016 x 2512
//     33.2 -> 29.5 (block kernel, two groups of wavefronts -> this one).
//   64x128, int4 rhs, which is half the bytes: 224 x 4944 x 2592 11.9 -> 9.0 us,
//     496 x 2192 x 2912 12.1 -> 9.5, from HBM 14.3 -> 12.0 (32x64 tiles of the
//     eight wavefronts -> this one). 206 registers, so that a second workgroup
//     fits a unit.
//   (Three steps in registers instead of two 1 to 9 % slower, with few chunks 20;
//   eight wavefronts on the 64x128 tile 5 to 20 %. 64x128 and 128x64 tiles of
//   16-bit operands, 64x64 ones of eight wavefronts and 128x64 and 128x128 of int4
//   gain nothing on what the other kernels do.)
//
// Operand registers: a fragment is 32 rows, a step's half feeds one
// v_mfma_f32_32x32x16_{f16,bf16} or v_mfma_i32_32x32x32_i8 with it; lane 32*h + r
// holds 16 bytes of row r. Which k those are is free as long as lhs and rhs
// agree: 16-byte column 2*u + h of the row's 64 in half u, with an int4 rhs
// 2*h + u, whose 16 bytes of nibbles are k step h. Four consecutive lanes touch one
// 128-byte line where a k step's row pieces are 16 or 32 bytes and tiles have
// four rows at least, which is what the kernel covers.
//
// No load and no multiply has a condition: loads are buffer loads, and where
// there is nothing to load (a row behind the last tile, a step behind the last
// one) they are out of their buffer's range, read nothing and give zeros. What
// the compiler counts of loads in flight is exact that way, and rows of padding
// cost no traffic and next to no power.
//
// K that ends inside a chunk: chunk 0 is the odd one, as in the block kernels.
#include <type_traits>

#define UK_MFMA_KERNEL_BODIES
#include "mmt4d_mfma_kernels.h"

namespace uk {
namespace {

constexpr int kWaves = 4;
// A buffer's bytes, and an offset that is outside of it: the plan keeps all others below.
constexpr uint32_t kBufferBytes = 0x80000000u;

// One operand of the workgroup's tile, F fragments of 32 rows.
template <int F>
struct TileOperand {
  const uint8_t* base;  // uniform: the tile's first row of tiles, k = 0
  uint32_t off[F];      // per lane, from base, of what it holds of a fragment in a step's first half
  uint32_t step_bytes;  // from one chunk of 64 bytes to the next
  uint32_t at;          // uniform: from base to the chunk of the wavefront that `off` counts from

  // 16 bytes of fragment f, `from` bytes on from base. `records`: bytes of the buffer, 0 to load nothing.
  __device__ __forceinline__ uint4 load(int f, uint32_t from, uint32_t records) const {
    const auto buffer = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)records, 0x00020000);
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(buffer, (int)off[f], (int)from, 0));
  }
};

template <int KIND, bool RHS_I4, bool NARROW, int FA>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(FA == 2 ? 2 : 1, FA == 2 ? 2 : 1)))
void mmt4d_mfma_wave_tile_kernel(const MfmaArgs a) {
  typedef typename AccType<KIND>::type acc_t;
  typedef typename AccType<KIND>::scalar scalar;
  typedef scalar v4 __attribute__((ext_vector_type(4)));
  constexpr int FB = 4;
  extern __shared__ uint4 partial[];  // [wavefront][fragment sent][4][lane]

  fetch_arguments(a);
  int tile_row, tile_col;
  if (!locate_block(a, &tile_row, &tile_col)) return;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t total_rows = (int64_t)a.M << a.log2_M0, total_cols = (int64_t)a.N << a.log2_N0;
  const int64_t first_row = (int64_t)tile_row * (32 * FA), first_col = (int64_t)tile_col * (32 * FB);

  const int log2_ksteps = 6 - a.log2_lhs_rb;            // of a chunk
  const int32_t cut = (a.chunks << log2_ksteps) - a.K;  // k steps that K lacks to whole chunks

  // `swap`: fragment f of the wavefront is fragment f ^ swap of the tile (see the sums).
  auto set_up = [&](auto& op, const uint8_t* base, int64_t first, int32_t tiles, int log2_t0, int64_t stride, int log2_rb,
                    int swap, uint32_t chunk_row_bytes, uint32_t lane_bytes) {
    const int32_t first_tile = (int32_t)(first >> log2_t0), last_tile = tiles - 1 - first_tile;
    op.base = uniform_pointer(base + first_tile * stride);
    op.step_bytes = chunk_row_bytes << log2_t0;
    op.at = wave * op.step_bytes - ((uint32_t)cut << (log2_rb + log2_t0));
    const uint32_t in_chunk = lane_bytes * h;
    const uint32_t lane_off = ((in_chunk >> log2_rb) << (log2_rb + log2_t0)) + (in_chunk & ((1u << log2_rb) - 1));
#pragma unroll
    for (int f = 0; f < (int)(sizeof op.off / sizeof op.off[0]); ++f) {
      const int32_t row = 32 * (f ^ swap) + r, tile = row >> log2_t0;
      const uint32_t off =
          (uint32_t)tile * (uint32_t)stride + ((uint32_t)(row & ((1 << log2_t0) - 1)) << log2_rb) + lane_off;
      op.off[f] = tile <= last_tile ? off : kBufferBytes;
    }
  };
  TileOperand<FA> lhs;
  TileOperand<FB> rhs;
  set_up(lhs, a.lhs, first_row, a.M, a.log2_M0, a.lhs_stride_bytes, a.log2_lhs_rb, 0, 64, RHS_I4 ? 32 : 16);
  set_up(rhs, a.rhs, first_col, a.N, a.log2_N0, a.rhs_stride_bytes, a.log2_rhs_rb, wave, RHS_I4 ? 32 : 64, 16);
  const uint32_t lhs_half = RHS_I4 ? 16 : lhs.step_bytes >> 1, rhs_half = rhs.step_bytes >> 1;

  acc_t acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

  // The wavefronts take chunks in turn. Step s of a wavefront lies in slot s & 1; its first half is loaded while the second
  // half of step s - 2 is multiplied, its second half behind that. (An int4 rhs has both halves in one load.)
  uint4 l[2][2][FA], w[2][RHS_I4 ? 1 : 2][FB];
  int32_t left = (a.chunks - wave + kWaves - 1) / kWaves;  // steps, from the one that is multiplied next
  // The buffer's bytes for a load that belongs to the step `ahead` from there, 0 where there is none. (On the scalar unit:
  // as a selection the compiler makes it on the vector unit, and the load a loop over the lanes' descriptors.)
  auto records = [&](int ahead) {
    int32_t v = ahead - left;
    asm("s_ashr_i32 %0, %0, 31\n\ts_and_b32 %0, %0, 0x80000000" : "+s"(v) : : "scc");
    return (uint32_t)v;
  };
  {
    // (Chunk 0 is the first 64 bytes, chunk 1 begins where chunk 0 less what K lacks ends.)
    const uint32_t lhs_first = wave == 0 ? 0 : lhs.at, rhs_first = wave == 0 ? 0 : rhs.at;
    lhs.at += kWaves * lhs.step_bytes;
    rhs.at += kWaves * rhs.step_bytes;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int s = k >> 1, u = k & 1;
      const uint32_t wanted = records(s);
#pragma unroll
      for (int f = 0; f < FB; ++f) {
        if (!RHS_I4) w[s][u][f] = rhs.load(f, (s ? rhs.at : rhs_first) + u * rhs_half, wanted);
        else if (k == 0) w[0][0][f] = rhs.load(f, rhs_first, wanted);
      }
#pragma unroll
      for (int f = 0; f < FA; ++f) l[s][u][f] = lhs.load(f, (s ? lhs.at : lhs_first) + u * lhs_half, wanted);
    }
  }
  if (wave == 0 && cut != 0) {
    const int32_t whole = (1 << log2_ksteps) - cut;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bool keep = (RHS_I4 ? 32 * h + 16 * u : 32 * u + 16 * h) >> a.log2_lhs_rb < whole;
      auto clear = [&](uint4& x) { x = make_uint4(keep ? x.x : 0, keep ? x.y : 0, keep ? x.z : 0, keep ? x.w : 0); };
#pragma unroll
      for (int f = 0; f < FA; ++f) clear(l[0][u][f]);
      if constexpr (!RHS_I4) {
#pragma unroll
        for (int f = 0; f < FB; ++f) clear(w[0][u][f]);
      }
    }
  }

  auto step = [&](auto slot) {
    constexpr int s = decltype(slot)::value;
    const uint32_t next = records(1), behind = records(2);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      // u = 0 loads the second half of the next step, u = 1 the first half of the one behind it, which has this one's slot.
      const int to = u == 0 ? 1 - s : s, half = 1 - u;
      const uint32_t lhs_at = lhs.at + (u == 0 ? lhs_half : kWaves * lhs.step_bytes);
      const uint32_t rhs_at = rhs.at + (u == 0 ? (RHS_I4 ? 0 : rhs_half) : kWaves * rhs.step_bytes);
      const int rhs_loads = RHS_I4 && u == 1 ? 0 : FB, loads = rhs_loads + FA;
      int t = 0;
#pragma unroll
      for (int j = 0; j < FB; ++j) {
        uint4 b;
        if constexpr (RHS_I4) {
          const uint4 both = w[s][0][j];
          b = widen_i4_times16(u == 0 ? make_uint2(both.x, both.y) : make_uint2(both.z, both.w));
        } else {
          b = w[s][u][j];
        }
#pragma unroll
        for (int i = 0; i < FA; ++i) {
          acc[i][j] = mfma<KIND>(b, l[s][u][i], acc[i][j]);
          // The loads are dealt out among the multiplies.
#pragma unroll
          for (int p = t * loads / (FA * FB); p < (t + 1) * loads / (FA * FB); ++p) {
            if (p < rhs_loads) w[to][RHS_I4 ? 0 : half][p] = rhs.load(p, rhs_at, u == 0 ? next : behind);
            else l[to][half][p - rhs_loads] = lhs.load(p - rhs_loads, lhs_at, u == 0 ? next : behind);
          }
          if (t & 1) __builtin_amdgcn_sched_barrier(0);
          ++t;
        }
      }
    }
    lhs.at += kWaves * lhs.step_bytes;
    rhs.at += kWaves * rhs.step_bytes;
    --left;
  };
  // (An odd number of steps has one of zeros behind it. Leaving the loop in the middle makes the register allocator move
  // the accumulators through memory.)
  while (left > 0) {
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
  }

  // Where the wavefront's column of fragments goes, and what an accumulating call finds there, asked for ahead of the sums.
  const int32_t M0 = 1 << a.log2_M0, N0 = 1 << a.log2_N0;
  typedef typename std::conditional<NARROW, uint2, v4>::type out_t;
  auto place = [&](int i, int e, out_t** to) {
    const int64_t row = first_row + 32 * i + r, col = first_col + 32 * wave + 8 * e + 4 * h;
    *to = (out_t*)a.out + ((row >> a.log2_M0) * a.out_stride0 + ((col >> a.log2_N0) << (a.log2_M0 + a.log2_N0)) +
                           ((row & (M0 - 1)) << a.log2_N0) + (col & (N0 - 1))) / 4;
    return row < total_rows && col < total_cols;
  };
  out_t old[FA][4];
  if (a.accumulate) {
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        out_t* from;
        if (place(i, e, &from)) old[i][e] = *from;
      }
  }

  // The sums, halving the columns of fragments that a wavefront is left with: two columns to the wavefront two on, one to its
  // neighbour. Column j of wavefront w is column j ^ w of the tile, so that each sends its last ones and keeps its first,
  // registers that the compiler knows, and ends with column w. ((0 + 2) + (1 + 3) whoever adds.)
  auto put = [&](int n, const acc_t& v) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      partial[(n * 4 + e) * 64 + lane] =
          make_uint4(value_bits(v[4 * e]), value_bits(v[4 * e + 1]), value_bits(v[4 * e + 2]), value_bits(v[4 * e + 3]));
  };
  auto add = [&](int n, acc_t& v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint4 p = partial[(n * 4 + e) * 64 + lane];
      const uint32_t q[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
      for (int x = 0; x < 4; ++x) v[4 * e + x] += __builtin_bit_cast(scalar, q[x]);
    }
  };
  auto halve = [&](auto to) {
    constexpr int cols = decltype(to)::value;
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < cols; ++j) put((wave * FA + i) * cols + j, acc[i][cols + j]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < cols; ++j) add(((wave ^ cols) * FA + i) * cols + j, acc[i][j]);
  };
  halve(std::integral_constant<int, 2>{});
  __syncthreads();  // (the partial sums are read)
  halve(std::integral_constant<int, 1>{});

#pragma unroll
  for (int i = 0; i < FA; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      out_t* to;
      if (!place(i, e, &to)) continue;
      v4 v = {acc[i][0][4 * e], acc[i][0][4 * e + 1], acc[i][0][4 * e + 2], acc[i][0][4 * e + 3]};
      if constexpr (RHS_I4) v = v4{v.x >> 4, v.y >> 4, v.z >> 4, v.w >> 4};
      if constexpr (NARROW) {
        constexpr int EBITS = KIND == kF16 ? 5 : 8;
        if (a.accumulate) {
          const uint2 o = old[i][e];
          v += v4{widen16_first<EBITS>(o.x), widen16_second<EBITS>(o.x), widen16_first<EBITS>(o.y), widen16_second<EBITS>(o.y)};
        }
        *to = make_uint2(narrow16_pair<EBITS>(v.x, v.y), narrow16_pair<EBITS>(v.z, v.w));
      } else {
        if (a.accumulate) v += old[i][e];
        *to = v;
      }
    }
  }
}

template <int KIND, bool RHS_I4, bool NARROW, int FA>
hipError_t launch_tile(MfmaArgs m, hipStream_t stream) {
  unsigned grid;
  set_tile_grid(&m, 32 * FA, 128, &grid);
  constexpr int lds_bytes = kWaves * FA * 2 * 4096;
  auto kernel = mmt4d_mfma_wave_tile_kernel<KIND, RHS_I4, NARROW, FA>;
  if (lds_bytes > 65536) {
    const hipError_t attr = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (attr != hipSuccess) return attr;
  }
  return launch_kernel<MfmaArgs>(kernel, grid, 64 * kWaves, lds_bytes, stream, m);
}

}  // namespace

hipError_t launch_wave_tile(const MfmaArgs& m, int kind, bool rhs_i4, bool narrow, hipStream_t stream) {
  if (rhs_i4) return launch_tile<kI8, true, false, 2>(m, stream);
  if (kind == kF16) return narrow ? launch_tile<kF16, false, true, 4>(m, stream) : launch_tile<kF16, false, false, 4>(m, stream);
  return narrow ? launch_tile<kBF16, false, true, 4>(m, stream) : launch_tile<kBF16, false, false, 4>(m, stream);
}

}  // namespace uk
