// Walks the convolution kernels' shapes (csrc/lbmib_conv_plan.h) on the host:
//   tiles   every output voxel of a tile belongs to exactly one position of
//           its waves, for every line width, tile shape and lines x planes
//           that the plans give.
//   grids   every launch that a plan gives has fewer than 2^32 threads.
//   ranges  the march's z ranges are the best of all counts, found without
//           trying each.
//   forms   a pyramid's layers take the march and the tile; layers of many
//           narrow samples, on which those mostly compute nothing, do not.
//   views   the weight gradient of a view of a volume is the volume's.
//   pieces  every 16-byte piece of a weight-gradient unit comes from the voxel
//           and channels that the LDS reads expect there.
// Prints what it finds wrong and returns the number of wrong cases.
#include <stdio.h>
#include <string.h>
#include <time.h>

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

static int grids() {
  int bad = 0;
  for (long B : {1L, 1000L, 8388600L, 8388601L, 8388608L, 8388616L, 16777216L, 500000000L})
    for (int side : {1, 2, 8, 64})
      for (int cin : {16, 32, 64, 256})
        for (int cout : {16, 48, 256}) {
          MarchGeo m = {};
          TileGeo t = {};
          int wm = 0, shape = 0;
          const bool mo = march_geo((int)B, side, side, side, cin, cout, &wm, &m);
          const bool to = tile_plan((int)B, side, side, side, cin, cout, &shape, &t);
          const long jobs = (mo && m.jobs > t.jobs) || !to ? (mo ? m.jobs : 0) : t.jobs;
          if ((jobs + 7) / 8 * 8 * 512 >= 1L << 32 && ++bad <= 10)
            printf("grids: %ld samples of %d^3, %d -> %d channels: %ld jobs\n", B, side, cin, cout, jobs);
        }
  return bad;
}

static int ranges() {
  int bad = 0;
  for (int cin : {16, 32})
    for (long cols : {1L, 3L, 17L, 64L, 255L, 256L, 1000L})
      for (int D = 1; D <= 700; ++D) {
        MarchGeo q = {};
        int wm = 0, zc = 0, zs = 0;
        if (!march_geo((int)cols, D, 4, 64, cin, 32, &wm, &q)) return 1;
        long best = -1;
        for (int n = 1; n <= D; ++n) {
          const int c = (D + n - 1) / n, used = (D + c - 1) / c;
          const long cost = (cols * used + 255) / 256 * ((c + 1) / 2 + 2);
          if (best < 0 || cost < best) best = cost, zc = c, zs = used;
        }
        if ((q.zc != zc || q.zs != zs) && ++bad <= 10)
          printf("ranges: %d planes, %ld columns: %d x %d, best %d x %d\n", D, cols, q.zs, q.zc, zs, zc);
      }
  // many planes: no more work for the host than for a few
  const auto spent = [](int D) {
    MarchGeo q = {};
    int wm = 0;
    const clock_t t0 = clock();
    volatile int used = 0;
    for (int k = 0; k < 200; ++k) {
      march_geo(1, D + k % 2, 1, 16, 16, 16, &wm, &q);
      used = used + q.zc;
    }
    return (double)(clock() - t0) / CLOCKS_PER_SEC / 200;
  };
  if (spent(1 << 16) > 2e-5 + 50 * spent(1 << 8)) {
    printf("ranges: %g s for 65,536 planes\n", spent(1 << 16));
    ++bad;
  }
  return bad;
}

static int forms() {
  int bad = 0, wm = 0, shape = 0;
  MarchGeo m = {};
  TileGeo t = {};
  const auto expect = [&](ConvForm want, int B, int D, int H, int W, int cin, int cout) {
    if (conv_form(B, D, H, W, cin, cout, &wm, &m, &shape, &t) == want) return;
    printf("forms: %d x %d x %d x %d, %d -> %d channels\n", B, D, H, W, cin, cout);
    ++bad;
  };
  for (int B : {1, 2, 4}) {
    expect(ConvForm::march, B, 64, 64, 64, 16, 32);
    expect(ConvForm::march, B, 64, 64, 64, 32, 32);
    expect(ConvForm::tile, B, 64, 64, 64, 64, 32);
    for (int side : {2, 4, 8, 16, 32})
      for (int c : {64, 128, 256}) expect(ConvForm::tile, B, side, side, side, c, c);
  }
  for (int c : {64, 128, 256})
    for (int side : {1, 2}) expect(ConvForm::general, 4096, side, side, side, c, c);
  expect(ConvForm::general, 4096, 3, 3, 3, 64, 64);
  expect(ConvForm::general, 64, 64, 1, 1, 64, 256);
  for (int c : {16, 32}) {
    expect(ConvForm::general, 1, 4096, 1, 16, c, 32);
    expect(ConvForm::general, 4096, 2, 4, 8, c, 64);
    expect(ConvForm::general, 4096, 8, 8, 8, c, 32);
  }
  return bad;
}

// The weight gradient of one channel over a volume: dw[t] = sum of dy[v] x[v + o(t)].
static std::vector<long> gradient(const std::vector<int> &x, const std::vector<int> &dy, int B, int D, int H, int W) {
  std::vector<long> dw(27, 0);
  for (int b = 0; b < B; ++b)
    for (int z = 0; z < D; ++z)
      for (int y = 0; y < H; ++y)
        for (int i = 0; i < W; ++i)
          for (int t = 0; t < 27; ++t) {
            const int zz = z + t / 9 - 1, yy = y + t / 3 % 3 - 1, xx = i + t % 3 - 1;
            if (zz < 0 || zz >= D || yy < 0 || yy >= H || xx < 0 || xx >= W) continue;
            dw[t] += (long)dy[((size_t)(b * D + z) * H + y) * W + i] * x[((size_t)(b * D + zz) * H + yy) * W + xx];
          }
  return dw;
}

static int views() {
  int bad = 0;
  for (int B : {1, 2, 7, 24, 64, 97, 130})
    for (int D : {1, 2, 5, 70})
      for (int H : {1, 3, 9, 66})
        for (int W : {1, 2}) {
          std::vector<int> x((size_t)B * D * H * W), dy(x.size());
          for (size_t k = 0; k < x.size(); ++k) x[k] = (int)(k * 7 % 23) - 9, dy[k] = (int)(k * 5 % 19) - 8;
          const WgView v = wgrad_view(B, D, H, W);
          const std::vector<long> want = gradient(x, dy, B, D, H, W), seen = gradient(x, dy, v.B, v.D, v.H, v.W);
          std::vector<long> got(27, -1);
          for (int t = 0; t < 27; ++t) {
            const int l = wgrad_tap(v.taps, t);
            got[l < 0 ? t : l] = l < 0 ? 0 : seen[t];
          }
          const bool narrow = W == 1 && v.W == 1 && (long)B * D * H > 1;
          if (((long)v.B * v.D * v.H * v.W != (long)x.size() || got != want || narrow) && ++bad <= 10)
            printf("views: %d x %d x %d x %d as %d x %d x %d x %d\n", B, D, H, W, v.B, v.D, v.H, v.W);
        }
  return bad;
}

// What lies at byte 16 e of a unit's dy: run e / (16 na) of 8 voxels, 2 na
// pieces each, the upper half first in odd runs.  x: lines of LP voxels.
static int pieces() {
  int bad = 0;
  const int widths[] = {1, 3, 8, 13, 33, 64, 65, 300}, heights[] = {1, 2, 5, 16};
  for (int W : widths)
    for (int H : heights)
      for (int C = 16; C <= 144; C += 16) {
        const int cin = C >= 128 ? 128 : (C >= 64 ? 64 : (C >= 32 ? 32 : 16));
        const WgradPlan p = wgrad_plan(2, 3, H, W, cin, C, 1 << 27);
        const WgGeo &q = p.q;
        for (int co0 = 0; co0 < C; co0 += 32)
          for (int e = 0; e < kWgRuns * 8 * 2 * p.na; ++e) {
            const int v = e / (2 * p.na), run = v / 8, second = p.na == 2 ? e / 2 % 2 : 0;
            const int half = p.na == 2 && run % 2 ? 1 - second : second;
            const int line = run / q.nr % q.R, plane = run / q.nr / q.R, x = run % q.nr * 8 + v % 8;
            const uint32_t w = wg_dy_piece(q, p.na, e, C - co0);
            const bool none = plane >= q.P || co0 + half * 16 >= C;
            const long want = (((long)plane * H + line) * W + x) * C + half * 16 + e % 2 * 8;
            if (none != (w == kWgNoPiece) || (!none && wg_piece_at(w, e, H, W, C) != want)) {
              if (++bad <= 10) printf("pieces: dy, W %d, H %d, %d channels from %d, piece %d\n", W, H, C, co0, e);
            }
          }
        for (int e = 0; e < q.xbytes / 16; ++e) {
          const int v = e / (2 * p.nb), second = p.nb == 2 ? e / 2 % 2 : 0, i = v % q.LP, L = v / q.LP;
          const int half = p.nb == 2 && (i / 8 + L) % 2 ? 1 - second : second;
          const int line = L % (q.R + 2), plane = L / (q.R + 2);
          const uint32_t w = wg_x_piece(q, p.nb, e);
          const long want = (((long)plane * H + line) * W + i) * cin + half * 16 + e % 2 * 8;
          if ((plane >= q.P) != (w == kWgNoPiece) || (plane < q.P && wg_piece_at(w, e, H, W, cin) != want)) {
            if (++bad <= 10) printf("pieces: x, W %d, H %d, %d channels, piece %d\n", W, H, cin, e);
          }
        }
      }
  return bad;
}

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!strcmp(what, "tiles")) return tiles() != 0;
  if (!strcmp(what, "views")) return views() != 0;
  if (!strcmp(what, "forms")) return forms() != 0;
  if (!strcmp(what, "ranges")) return ranges() != 0;
  if (!strcmp(what, "grids")) return grids() != 0;
  if (!strcmp(what, "pieces")) return pieces() != 0;
  return 2;
}
