// Where the direct-to-LDS kernel loads from, stage by stage (iree_amd/csrc/mmt4d_chunk_walk.h), for every number of chunks: in the
// order of the kernel's steps (mmt4d_mfma_direct_kernel: the first chunks, rounds of four steps where it takes them, single
// steps), that no load leaves the operand, that a stage is not loaded into before its chunk has been read, that a step reads the
// chunk it multiplies next, and that each byte of K counts once over the groups.
#include <stdint.h>
#include <stdio.h>

#include <vector>

#include "mmt4d_chunk_walk.h"

static long walks = 0, wrong = 0;

template <int STAGES, int GROUPS>
struct Walk {
  static constexpr uint32_t kStage = 1024, kRing = STAGES * kStage;
  typedef uk::RingPlace<STAGES, GROUPS, kStage> Place;
  static constexpr int AHEAD = Place::AHEAD;

  int row_bytes, group;
  const int chunk_bytes, other_chunk_bytes;  // of both operands
  const uint8_t *a, *b;
  std::vector<int64_t> a_in, b_in;  // what each stage holds: offsets into the operands, in bytes per row
  std::vector<int> read_by;         // the step that reads each stage's chunk, which step s + 1 is done with
  bool ok = true;

  void check(bool right, const char* what, int step) {
    if (right) return;
    ok = false;
    if (wrong < 10) printf("%s: %d stages, %d groups, %d bytes, group %d, step %d\n", what, STAGES, GROUPS, row_bytes, group, step);
  }

  // `rows`: of the tile, i.e. an operand's bytes per byte of a row.
  int64_t per_row(const uint8_t* from, const uint8_t* base, int chunk, int step) {
    const int64_t off = from - base, rows = chunk / 64;
    check(off >= 0 && off % rows == 0 && off / rows + 64 <= row_bytes, "load outside the operand", step);
    return off / rows;
  }
  // Step `step` loads into the stage at LDS offset `off`; while it does, other wavefronts may be reading what step - 1 reads.
  void load(uint32_t off, const uint8_t* from_a, const uint8_t* from_b, int step) {
    const uint32_t in_ring = off - group * kRing;
    check(in_ring < kRing && in_ring % kStage == 0, "stage outside the ring", step);
    const int stage = in_ring / kStage % STAGES;
    check(read_by[stage] < step - 1, "stage loaded into before it has been read", step);
    a_in[stage] = per_row(from_a, a, chunk_bytes, step);
    b_in[stage] = per_row(from_b, b, other_chunk_bytes, step);
    read_by[stage] = step + AHEAD - 1;
  }
  // Step `step` reads chunk step + 1.
  void read(uint32_t off, int step, const uk::GroupChunks<GROUPS>& c) {
    check(off < kRing && off % kStage == 0, "fragments outside the ring", step);
    if (step + 1 > c.last) return;  // nothing multiplies what the last step reads
    const int stage = off / kStage % STAGES;
    int64_t want = 64ll * (GROUPS * (step + 1) + c.from) - c.cut_of_row;
    if (want < 0) want = 0;
    check(a_in[stage] == want && b_in[stage] == want && read_by[stage] == step, "another chunk's fragments", step);
  }

  Walk(int row_bytes, int log2_piece, int group, int rows, int cols, bool by_four, std::vector<int>* counted)
      : row_bytes(row_bytes), group(group), chunk_bytes(64 * rows), other_chunk_bytes(64 * cols),
        a((const uint8_t*)(1ull << 40)), b((const uint8_t*)(3ull << 40)), a_in(STAGES, -1), b_in(STAGES, -1), read_by(STAGES, -100) {
    const uk::GroupChunks<GROUPS> c((row_bytes + 63) / 64, row_bytes >> log2_piece, log2_piece, group);
    const int a_cut = c.cut_of_row * rows, b_cut = c.cut_of_row * cols;
    auto a_near = [&](int i) { return a + c.offset(i, chunk_bytes, a_cut); };
    auto b_near = [&](int i) { return b + c.offset(i, other_chunk_bytes, b_cut); };
    for (int i = 0; i < AHEAD; ++i)  // as steps 0 - AHEAD, 1 - AHEAD, .. would
      load(group * kRing + (i + STAGES - 1) % STAGES * kStage, a_near(i), b_near(i), i - AHEAD);
    Place at(a_near(AHEAD), b_near(AHEAD), group * kRing);
    read((STAGES - 1) * kStage, -1, c);
    int step = 0;
    if constexpr (STAGES == 4 || STAGES == 8) {
      typedef uk::FourSteps<STAGES, GROUPS, kStage> Fours;
      if (by_four && Fours::pays(c.last)) {
        Fours fours(at);
        while (Fours::fits(step, c.last)) {
          for (int s = 0; s < 4; ++s) {
            const uint32_t further = s * GROUPS;
            load(fours.loads(s) + Fours::loads_into(s) * kStage, at.load_a + further * chunk_bytes,
                 at.load_b + further * other_chunk_bytes, step + s);
            read(fours.reads(at) + s * kStage, step + s, c);
          }
          step += 4;
          fours.advance(&at, chunk_bytes, other_chunk_bytes);
        }
        check(step >= 8, "fewer than two rounds", step);
        fours.leave(&at, step, c.last, chunk_bytes, other_chunk_bytes);
      }
    }
    for (; step < c.count; ++step) {
      load(at.load_off, at.load_a, at.load_b, step);
      read(at.read_off, step, c);
      at.advance(c.last, chunk_bytes, other_chunk_bytes);
    }
    for (int i = 0; i < c.count; ++i) {
      const int64_t first = i == 0 ? (a_near(0) - a) / rows : 64ll * (GROUPS * i + c.from) - c.cut_of_row;
      for (int byte = 0; byte < 64 - (i == 0 ? c.cut_bytes : 0); ++byte)
        if (first + byte < row_bytes) ++(*counted)[first + byte];
    }
    ++walks;
    wrong += !ok;
  }
};

template <int STAGES, int GROUPS>
void all() {
  for (int log2_piece : {0, 1, 2, 3, 4, 5, 6})
    for (int row_bytes = 64; row_bytes <= 64 * 90; row_bytes += 1 << log2_piece) {
      // (two groups, where there is a chunk for each)
      if (GROUPS == 2 && row_bytes < 128) continue;
      if (log2_piece < 2 && row_bytes > 64 * 42) break;
      for (bool by_four : {false, true}) {
        std::vector<int> counted(row_bytes, 0);
        for (int group = 0; group < GROUPS; ++group)
          Walk<STAGES, GROUPS>(row_bytes, log2_piece, group, 16, 8, by_four, &counted);
        for (int n : counted)
          if (n != 1) {
            if (wrong++ < 10) printf("%d stages, %d groups, %d bytes: a byte counts %d times\n", STAGES, GROUPS, row_bytes, n);
            break;
          }
      }
    }
}

int main() {
  all<4, 1>();
  all<8, 1>();
  all<10, 1>();
  all<4, 2>();
  all<8, 2>();
  printf("%ld walks, %ld wrong\n", walks, wrong);
  return wrong != 0;
}
