// divide and tile_of_number (iree_amd/csrc/uk_device.h) against plain divisions: divisors up to the largest with the numbers
// around their multiples; every tile of small grids, and the tiles around the ends of bands and of the grid of large ones.
#include <stdint.h>
#include <stdio.h>

#include "uk_device.h"

static long checked = 0, wrong = 0;

static void check(uint32_t linear, uint32_t rows, uint32_t cols) {
  const uint64_t band = linear / (4ull * cols), in_band = linear - band * 4 * cols;
  const uint64_t band_rows = rows - band * 4 < 4 ? rows - band * 4 : 4;
  int row = -1, col = -1;
  uk::tile_of_number(linear, rows, cols, uk::band_reciprocal(cols), &row, &col);
  ++checked;
  if ((uint64_t)row != band * 4 + in_band % band_rows || (uint64_t)col != in_band / band_rows) {
    if (wrong++ < 10) printf("tile %u of %u x %u: %d, %d\n", linear, rows, cols, row, col);
  }
}

static void check_divide(uint32_t n, uint32_t d) {
  ++checked;
  const uint32_t q = uk::divide(n, d, uk::reciprocal_of(d));
  if (q != n / d && wrong++ < 10) printf("%u / %u: %u\n", n, d, q);
}

int main() {
  for (uint64_t d = 1; d < 1ull << 32; d = d < 5000 ? d + 1 : d + d / 37)
    for (uint64_t q : {0ull, 1ull, 2ull, 3ull, 100ull, 65535ull, 0xFFFFFFFFull / d / 2, 0xFFFFFFFFull / d - 1, 0xFFFFFFFFull / d})
      for (int64_t e = -2; e <= 2; ++e) {
        const int64_t n = (int64_t)(q * d) + e;
        if (n >= 0 && n < 1ll << 32) check_divide((uint32_t)n, (uint32_t)d);
      }
  for (uint32_t d : {1u, 2u, 3u, 7u, 64u, 0x7FFFFFFFu, 0x80000000u, 0xFFFFFFFFu}) check_divide(0xFFFFFFFFu, d);
  for (uint32_t rows = 1; rows <= 40; ++rows)
    for (uint32_t cols = 1; cols <= 130; ++cols)
      for (uint32_t i = 0; i < rows * cols; ++i) check(i, rows, cols);
  const uint32_t sizes[] = {1, 2, 3, 5, 6, 7, 8, 255, 1023, 4097, 65535, 65536, 99991, (1u << 20) - 1, 1u << 24, (1u << 28) + 3,
                            (1u << 29) - 1};
  for (uint32_t rows : sizes)
    for (uint32_t cols : sizes) {
      const uint64_t tiles = (uint64_t)rows * cols;
      if (tiles >= 1ull << 31) continue;
      const uint64_t band = 4ull * cols;
      for (uint64_t b = 0; b < 1000 && b * band < tiles; ++b)
        for (int d = -6; d <= 6; ++d) {
          const int64_t ends[] = {(int64_t)(b * band) + d, (int64_t)(tiles / band * band - b * band) + d, (int64_t)tiles - 1 - (int64_t)b + d};
          for (int64_t i : ends)
            if (i >= 0 && (uint64_t)i < tiles) check((uint32_t)i, rows, cols);
        }
    }
  printf("%ld tiles, %ld wrong\n", checked, wrong);
  return wrong != 0;
}
