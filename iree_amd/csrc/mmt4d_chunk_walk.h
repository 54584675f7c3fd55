// Which chunks of K a workgroup of the direct-to-LDS kernel (mmt4d_mfma_kernels.h) loads, from where, and which stage of its
// ring each lies in. For the host too: tests/host_checks/chunk_walk_check.hip walks it.
#ifndef IREE_AMD_CSRC_MMT4D_CHUNK_WALK_H_
#define IREE_AMD_CSRC_MMT4D_CHUNK_WALK_H_

#include <stdint.h>

#include "uk_device.h"

namespace uk {

// K in whole chunks of 64 bytes per row but for the first: where K is none, chunk 0 is the first 64 bytes of every row all the
// same and chunk 1 begins where chunk 0 without its last `cut_bytes` ends. Every load stays inside the operands (there is a whole
// chunk at least), and what chunk 0 shares with chunk 1 is zeroed in its fragments of both operands once, in front of the
// loop (0 * 0 adds nothing, whatever the data; with an int4 rhs, where 0 * anything does, in the lhs alone). (The last
// chunk was the odd one before: a mask in every step, which the compiler makes unconditional, 24 of a step's 120
// instructions on the 256x128 tile, or a further step behind the loop, and four more scalar selects for where the last
// chunk lies.)
// Two groups: chunk i of group g is chunk 2*i + g of K, or one less where K has an odd number of chunks; the first group's
// first is none then, loaded as chunk 0 and zeroed whole.
template <int GROUPS>
struct GroupChunks {
  int32_t count, last;  // of the group: step i multiplies chunk i
  int32_t from;         // chunk i of the group is chunk GROUPS * i + from of K
  int32_t cut_of_row;   // bytes per row that K lacks to whole chunks
  int32_t cut_bytes;    // the last so many of chunk 0's 64 bytes per row are zeroed

  __host__ __device__ __forceinline__ GroupChunks(int32_t chunks, int32_t K, int log2_row_piece, int group)
      : count(GROUPS == 1 ? chunks : (chunks + 1) >> 1), last(count - 1), from(GROUPS == 1 ? 0 : group - (chunks & 1)),
        cut_of_row((int32_t)((64 - (((int64_t)K << log2_row_piece) & 63)) & 63)),
        cut_bytes(from < 0 ? 64 : (from == 0 ? cut_of_row : 0)) {}

  // Bytes from an operand's first to chunk i's first, `chunk_bytes` and `cut` (cut_of_row) in all of a tile's rows. For the
  // first few chunks (32 bits), and with minima and maxima instead of branches: this runs in front of the first load. Chunks
  // beyond the last one are that one again.
  __host__ __device__ __forceinline__ uint32_t offset(int32_t i, int32_t chunk_bytes, int32_t cut) const {
    const int32_t chunk = GROUPS * (i < last ? i : last) + from, bytes = chunk * chunk_bytes - cut;
    return (uint32_t)(bytes > 0 ? bytes : 0);
  }
};

// Where the next step loads from and to and reads from: running values (a few scalar adds per step) rather than recomputed from
// the chunk's number (64-bit multiplies on the scalar unit, in front of the step's first MFMA). Step i loads chunk
// i + AHEAD and reads the fragments of chunk i + 1; chunk c lies in stage c - 1 modulo their number.
template <int STAGES, int GROUPS, uint32_t STAGE_BYTES>
struct RingPlace {
  static constexpr int AHEAD = STAGES - 1;
  static constexpr uint32_t RING_BYTES = STAGES * STAGE_BYTES;

  const uint8_t *load_a, *load_b;
  uint32_t ring_begin;              // LDS offset that loads count from
  uint32_t load_off, read_off = 0;  // LDS offsets: the former's count from 0 of the LDS, the latter's from the ring's first stage
  int32_t load_chunk = AHEAD;

  __host__ __device__ __forceinline__ RingPlace(const uint8_t* a, const uint8_t* b, uint32_t begin)
      : load_a(a), load_b(b), ring_begin(begin), load_off((STAGES - 2) * STAGE_BYTES + begin) {}

  // The next step's. (Clamped at the last chunk: the loads issued beyond it are redundant, their stages are never read.)
  __host__ __device__ __forceinline__ void advance(int32_t last, int32_t a_chunk_bytes, int32_t b_chunk_bytes) {
    const bool more = load_chunk < last;
    load_a += (uint32_t)(more ? GROUPS * a_chunk_bytes : 0);
    load_b += (uint32_t)(more ? GROUPS * b_chunk_bytes : 0);
    ++load_chunk;
    load_off = load_off + STAGE_BYTES == RING_BYTES + ring_begin ? ring_begin : load_off + STAGE_BYTES;
    read_off = read_off + STAGE_BYTES == RING_BYTES ? 0 : read_off + STAGE_BYTES;
  }
};

// Four steps at a time while all of their loads are of chunks that exist: step s of the four reads stage s of `reads()` and
// loads, from s * GROUPS chunks beyond the place's load_a and load_b, into stage `loads_into(s)` of `loads(s)`.
template <int STAGES, int GROUPS, uint32_t STAGE_BYTES>
struct FourSteps {
  typedef RingPlace<STAGES, GROUPS, STAGE_BYTES> Place;
  static_assert(STAGES == 4 || STAGES == 8, "two fours at most");
  // LDS offsets of the four stages that four steps read, whose last two steps load into the first two of them, and of
  // those before, which the first two load into (four stages: the same).
  uint32_t this_four, other_four;

  __host__ __device__ __forceinline__ explicit FourSteps(const Place& place)
      : this_four(place.ring_begin), other_four(place.ring_begin + (STAGES == 4 ? 0 : 4 * STAGE_BYTES)) {}

  // (Two rounds at least: the preparation costs a K of few 1 %.)
  static __host__ __device__ __forceinline__ bool pays(int32_t last) { return last >= Place::AHEAD + 8; }
  static __host__ __device__ __forceinline__ bool fits(int32_t step, int32_t last) { return step + 3 + Place::AHEAD <= last; }

  __host__ __device__ __forceinline__ uint32_t reads(const Place& place) const { return this_four - place.ring_begin; }
  __host__ __device__ __forceinline__ uint32_t loads(int s) const { return s < 2 ? other_four : this_four; }
  static constexpr int loads_into(int s) { return (s + 2) % 4; }

  __host__ __device__ __forceinline__ void advance(Place* place, int32_t a_chunk_bytes, int32_t b_chunk_bytes) {
    place->load_a += (uint32_t)(4 * GROUPS * a_chunk_bytes);
    place->load_b += (uint32_t)(4 * GROUPS * b_chunk_bytes);
    if constexpr (STAGES == 8) {
      const uint32_t was = this_four;
      this_four = other_four;
      other_four = was;
    }
  }
  // Back to single steps, `step` being the next. (The chunk after the last one, if the rounds came that far, is the last one
  // again.)
  __host__ __device__ __forceinline__ void leave(Place* place, int32_t step, int32_t last, int32_t a_chunk_bytes,
                                                 int32_t b_chunk_bytes) const {
    place->load_chunk = step + Place::AHEAD;
    const bool beyond = step > 0 && place->load_chunk > last;
    place->load_a -= (uint32_t)(beyond ? GROUPS * a_chunk_bytes : 0);
    place->load_b -= (uint32_t)(beyond ? GROUPS * b_chunk_bytes : 0);
    place->read_off = this_four - place->ring_begin;
    place->load_off = other_four + 2 * STAGE_BYTES;
  }
};

}  // namespace uk

#endif  // IREE_AMD_CSRC_MMT4D_CHUNK_WALK_H_
