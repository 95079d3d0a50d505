// Walks the even cells up to 1024 per edge and checks that a post-smoother
// that forms r.z has a partial-sum row for each of its tiles, for every tile
// shape a context may hold; prints the choice for a few cells. Host code
// only; tests/test_tile_rows.py compiles and reads it.
#include <cstdio>

#include "otm_fine_dev.hpp"

using namespace otm;

static Geom cell(int x, int y, int z) { return Geom{x, y, z, (long long)x * y * z}; }

int main() {
  long long cells = 0, fused = 0, apart = 0, bad = 0;
  for (int z = 8; z <= 1024; z += 2)
    for (int y = 8; y <= 1024; y += 2)
      for (int x = 8; x <= 1024; x += 2) {
        const Geom g = cell(x, y, z);
        cells++;
        for (int v = fine_tile_default(g) < 0 ? -1 : 0; v < kFineTileVariants; v++) {
          if (!fine_brick_ok(g, v)) continue;
          if (!fine_brick_dot_ok(g, v)) {
            apart++;
            continue;
          }
          fused++;
          if (fine_brick_tiles(g, v) > fine_dot_rows(g) || fine_dot_rows(g) > kTileDotSlots) bad++;
        }
      }
  std::printf("walk %lld %lld %lld %lld\n", cells, fused, apart, bad);
  for (int n : {64, 256, 384, 400, 416, 512, 1024}) {
    const Geom g = cell(n, n, n);
    const int v = fine_tile_default(g);
    std::printf("cube %d %lld %lld %d\n", n, fine_brick_tiles(g, v), fine_dot_rows(g), fine_brick_dot_ok(g, v) ? 1 : 0);
  }
  return 0;
}
