// Column tiles of the plain 2-D FFT: a tile fits a workgroup's threads and
// LDS, and enough of its lanes have a column: half of them, or a quarter up to
// 64 points, where a workgroup is one wave with or without the tile.
#include <cstdio>
#include <cstdlib>

#include "../../bldfm_amd/csrc/bldfm_types.h"

#define CHECK(c, ...) do { if (!(c)) { printf(__VA_ARGS__); printf("\n"); exit(1); } } while (0)

int main() {
  long tiled = 0, all = 0;
  for (int n0 = 1; n0 <= 2300; ++n0)
    for (int n1 = 1; n1 <= 300; ++n1)
      for (long batch = 1; batch <= 1L << 24; batch *= 64) {
        ++all;
        const int c = fft2_tile(n0, n1, batch);
        if (!c) continue;
        ++tiled;
        const int lanes = (n0 + 7) / 8, tiles = (n1 + c - 1) / c;
        CHECK(n0 <= 2048 && (c == 4 || c == 8), "%d x %d: %d columns", n0, n1, c);
        CHECK((lanes * c + 63) / 64 * 64 <= 1024, "%d x %d: %d lanes", n0, n1, lanes * c);
        CHECK((n0 * c + tw_table_len(n0)) * 16 <= 160 * 1024, "%d x %d: LDS", n0, n1);
        CHECK((n0 > 64 ? 2 : 4) * n1 >= tiles * c, "%d x %d: %d of %d lanes have a column", n0, n1, n1, tiles * c);
      }
  CHECK(tiled > 0 && tiled < all, "%ld of %ld", tiled, all);
  printf("%ld of %ld in tiles\n", tiled, all);
  return 0;
}
