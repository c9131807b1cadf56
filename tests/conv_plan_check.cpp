// Walks the convolution kernels' shapes (csrc/lbmib_conv_plan.h) on the host:
//   tiles   every output voxel of a tile belongs to exactly one position of
//           its waves, for every line width, tile shape and lines x planes
//           that the plans give.
// Prints what it finds wrong and returns the number of wrong cases.
#include <stdio.h>
#include <string.h>

#include <vector>

#include "../distributed-lb-ib_amd/csrc/lbmib_conv_plan.h"

using namespace lbmib;

static int tiles() {
  int bad = 0;
  std::vector<int> seen;
  const int sides[] = {1, 2, 3, 5, 8, 16, 17, 31, 64, 100, 195, 217, 256, 300, 489, 511, 512, 600, 2048};
  for (int W = 1; W <= 64; ++W)
    for (const TileShape &c : kTileShapes)
      for (int H : sides)
        for (int D : sides) {
          TileGeo q = {};
          if (!tile_geo(1, D, H, W, 64, 64, c.wm, c.nc, c.kw, c.vg, &q)) continue;
          seen.assign((size_t)q.PZ * q.LP * W, 0);
          bool out = false;
          for (int vg = 0; vg < c.vg; ++vg)
            for (int pos = 0; pos < 16 * c.wm; ++pos) {
              const TilePos t = tile_pos(q, W, vg, pos);
              if (!t.in) continue;
              if (t.pz < 0 || t.pz >= q.PZ || t.ly < 0 || t.ly >= q.LP || t.x < 0 || t.x >= W) out = true;
              else ++seen[((size_t)t.pz * q.LP + t.ly) * W + t.x];
            }
          for (int n : seen) out |= n != 1;
          if (out && ++bad <= 10)
            printf("tiles: W %d, H %d, D %d, shape %d %d %d %d, LP %d, PZ %d\n", W, H, D, c.wm, c.nc, c.kw, c.vg, q.LP,
                   q.PZ);
        }
  return bad;
}

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!strcmp(what, "tiles")) return tiles() != 0;
  return 2;
}
