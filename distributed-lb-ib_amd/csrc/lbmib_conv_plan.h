// lbmib_conv_plan.h -- shapes of the surrogate's convolution kernels
// (lbmib_surr.hip): where each form applies, how it splits a layer, and the
// index arithmetic that host and kernels share.  No HIP call and no device
// type, so that a program on the host can walk every shape.
#pragma once
#include <stddef.h>
#include <stdint.h>

#if defined(__HIP__)
#define LBMIB_HD __host__ __device__ inline
#else
#define LBMIB_HD inline
#endif

namespace lbmib {

LBMIB_HD int ilog2(int v) {
  int r = 0;
  while ((1 << r) < v) ++r;
  return r;
}

// A launch has fewer than 2^32 threads along x: blocks of 512, rounded up to
// eight.  Layers of more jobs (8 million samples) are left to the general form.
constexpr long kMaxJobs = (1L << 23) - 8;

// ------------------------------------------- forward: march (k_conv_march)

struct MarchGeo {
  int G, nyb, zc, zs, cot;  // lines per wave; line groups, planes per block, z ranges, channel tiles
  int plane_bytes;          // of one ring slot
  long jobs;
};

// Where the march applies, and its shape.
inline bool march_geo(int B, int D, int H, int W, int Cin, int Cout, int *wm, MarchGeo *q) {
  if ((Cin != 16 && Cin != 32) || W < 8 || W > 64) return false;
  const long HW = (long)H * W;
  if (HW * (Cin > Cout ? Cin : Cout) * 2 >= (1L << 31)) return false;
  // positions per wave: the multiple of 16 that whole lines fill best
  const int g4 = 64 / W, g3 = 48 / W;
  *wm = g3 && g3 * W * 4 > g4 * W * 3 ? 3 : 4;
  q->G = *wm == 3 ? g3 : g4;
  q->nyb = (H + 4 * q->G - 1) / (4 * q->G);
  q->plane_bytes = ((4 * q->G + 2) * W * 2 * Cin + 1023) / 1024 * 1024;
  q->cot = (Cout + 31) / 32;
  // z ranges: one block a CU (256), so the rounds of blocks times the plane
  // pairs each takes (and about two for its weights and first planes) are
  // least.  Only the counts at which the planes per block change are tried: 2
  // sqrt(D) of them, where all D took 0.28 ms of every call at 65,536 planes.
  const long cols = (long)B * q->nyb * q->cot;
  long best = -1;
  for (int zs = 1; zs <= D;) {
    const int zc = (D + zs - 1) / zs, used = (D + zc - 1) / zc;
    const long cost = (cols * used + 255) / 256 * ((zc + 1) / 2 + 2);
    if (best < 0 || cost < best) {
      best = cost;
      q->zc = zc;
      q->zs = used;
    }
    if (zc == 1) break;
    zs = (D + zc - 2) / (zc - 1);  // the least count with fewer planes a block
  }
  q->jobs = cols * q->zs;
  return q->jobs <= kMaxJobs;
}

// Positions that the march computes for each voxel: those of lines past the
// plane's end, past a line's and of an odd last plane.
inline double march_fill(const MarchGeo &q, int wm, int D, int H, int W) {
  return (double)q.nyb * 4 * 16 * wm * q.zs * ((q.zc + 1) / 2 * 2) / ((double)D * H * W);
}

// --------------------------------------------- forward: tile (k_conv_tile)

struct TileGeo {
  int G, LP, PZ, nty, ntz, cot;  // lines per group; tile lines and planes; tiles in y and z; channel tiles
  int cs, lgp;                   // channels staged at a time; log2 of their 16-byte pieces per voxel
  int box, lds;                  // LDS bytes of the box, and of all
  int mW, mLP;                   // 2^20 / W + 1, 2^20 / LP + 1: quotients (tile_pos)
  long jobs;
};

// Shape of the tile form for 16 WM positions, NC channel groups, KW parts and
// VG voxel groups; false where it does not apply.
inline bool tile_geo(int B, int D, int H, int W, int Cin, int Cout, int wm, int nc, int kw, int vg, TileGeo *q) {
  if (Cin < 32 || W > 16 * wm || W > 64) return false;
  const long S = (long)D * H * W;
  if (S * (Cin > Cout ? Cin : Cout) * 2 >= (1L << 31) || (long)Cout * 27 * Cin * 2 >= (1L << 31)) return false;
  q->G = 16 * wm / W;
  const int nl = q->G * vg;
  // lines x planes: the fewest tiles, then the fewest lines in a tile's box
  long best = -1;
  for (int pz = 1; pz <= nl && pz <= D && pz <= 16; ++pz) {
    const int lp = nl / pz < H ? nl / pz : H;
    const long tiles = (long)((H + lp - 1) / lp) * ((D + pz - 1) / pz);
    const long cost = tiles * 100000 + (long)(lp + 2) * (pz + 2);
    if (best < 0 || cost < best) {
      best = cost;
      q->LP = lp;
      q->PZ = pz;
    }
  }
  q->nty = (H + q->LP - 1) / q->LP;
  q->ntz = (D + q->PZ - 1) / q->PZ;
  q->cot = (Cout + 16 * nc - 1) / (16 * nc);
  q->mW = (1 << 20) / W + 1;
  q->mLP = (1 << 20) / q->LP + 1;
  const long vox = (long)(q->LP + 2) * (q->PZ + 2) * W;
  q->cs = Cin;
  const long most = 160 * 1024 - 8 * 3072;
  while (q->cs > 32 && vox * (q->cs * 2 + 16) > most) q->cs /= 2;
  const long box = vox * (q->cs * 2 + 16), red = kw > 1 ? 8L * wm * 1024 : 0;
  if (box > most) return false;
  q->box = (int)box;
  q->lds = (int)(box + 8 * 3072 > red ? box + 8 * 3072 : red);
  q->lgp = ilog2(q->cs / 8);
  q->jobs = (long)B * q->nty * q->ntz * q->cot;
  return q->jobs <= kMaxJobs;
}

// Position pos of voxel group vg: its plane and line in the tile, and its x.
// n / d as n (2^20 / d + 1) >> 20, which is exact for n d < 2^20 and stays in
// 31 bits: n <= 511 (the lines of a tile at W = 1) and d <= 512.  (With 2^16 the
// last of 512 lines fell out of the tile and were not written.)
struct TilePos {
  int pz, ly, x;
  bool in;
};
LBMIB_HD TilePos tile_pos(const TileGeo &q, int W, int vg, int pos) {
  TilePos t;
  const int l = (pos * q.mW) >> 20, lt = vg * q.G + l;
  t.x = pos - l * W;
  t.pz = (lt * q.mLP) >> 20;
  t.ly = lt - t.pz * q.LP;
  t.in = l < q.G && t.pz < q.PZ;
  return t;
}

// The shape of least estimated time, in us: a block's first loads and box,
// which take longer the more of the 256 CUs fetch at once, its items, and the
// sum over KW.  The constants are a fit to the shapes below on 70 layers (Cin 64 to
// 256, and 32 below 4096 voxels; 4 to 64 voxels a side, Cout 16 to 256): 6.6%
// rms, and the shape it picks takes 2% longer than the fastest on average.
// The narrowest shape leaves room for two blocks a CU where its box is small.
struct TileShape {
  int wm, nc, kw, vg;
};
constexpr TileShape kTileShapes[] = {{8, 8, 1, 1}, {8, 4, 1, 2}, {8, 2, 1, 4}, {8, 4, 2, 1}, {8, 2, 4, 1}, {8, 1, 8, 1},
                                     {4, 4, 2, 1}, {4, 2, 2, 2}, {4, 2, 4, 1}, {4, 1, 8, 1}, {2, 1, 8, 1}};

inline bool tile_plan(int B, int D, int H, int W, int Cin, int Cout, int *shape, TileGeo *q) {
  double best = 0;
  bool any = false;
  for (int k = 0; k < (int)(sizeof(kTileShapes) / sizeof(kTileShapes[0])); ++k) {
    const TileShape &c = kTileShapes[k];
    TileGeo g;
    if (!tile_geo(B, D, H, W, Cin, Cout, c.wm, c.nc, c.kw, c.vg, &g)) continue;
    const int per = c.wm == 2 && g.lds <= 80 * 1024 ? 2 : 1;
    const long rounds = (g.jobs + 256 * per - 1) / (256 * per);
    const double busy = g.jobs < 256 * per ? (double)g.jobs / (256 * per) : 1.0;
    const int slices = Cin / g.cs, items = ((9 * g.cs / 32 + c.kw - 1) / c.kw + 1) / 2 * 2 * slices;
    const double mb = (double)(g.LP + 2) * (g.PZ + 2) * W * (2 * Cin + 16) * 1e-6;
    const double t = rounds * (2.0 * slices + 10.3 * mb * (0.28 + busy) +
                               items * (0.073 * c.wm + 0.1) * (per == 2 ? 1.7 : 1.0) + (c.kw > 1 ? 2.1 : 0.0));
    if (!any || t < best) {
      any = true;
      best = t;
      *shape = k;
      *q = g;
    }
  }
  return any;
}

// Positions that the tiles of a shape compute for each voxel.
inline double tile_fill(const TileGeo &q, int shape, int D, int H, int W) {
  const TileShape &c = kTileShapes[shape];
  return (double)q.nty * q.ntz * 16 * c.wm * c.vg / ((double)D * H * W);
}

// Which form a layer takes.  The march and the tile work on one sample at a
// time, on whole lines; the forms below them (k_conv_fwd, k_conv_fwd_kw) on the
// voxels in linear order, with no position to spare.
//
// Few input channels: the march, from where its ~9 us of first loads and
// launch are no more than the small-grid forms take (16^3 at batch 4, 32 ->
// 64: 9.2 against 10.6 us; 32 -> 32: 9.0 against 8.5), unless it computes four
// positions for each voxel (4096 x 1 x 16, 32 -> 32: 40 us, general 15; 1024
// samples of 8^3, 32 -> 32: 86 and 73; 64 of 10^3, 2.6 positions: 13 and 17).
//
// More channels, and few-channel grids too small for the forms below (8^3 at
// batch 4, 32 -> 64: 6.7 us; from 4096 voxels on those are faster, 7.4 against
// 7.6 us at 16^3): the tile, unless it takes more than two rounds of 256 blocks
// and computes 1.5 positions for each voxel (4096 samples of 2^3, 128 -> 128:
// 345 us, general 66; of 3^3, 64 -> 64: 133 and 59), or two and four (64 of 64 x
// 1 x 1, 64 -> 256: 33 and 19).  Below that its time is a block's, which the
// general forms do not reach (64 of 2^3, 256 -> 64: 9 us, general 23).
enum class ConvForm { march, tile, general };
inline ConvForm conv_form(int B, int D, int H, int W, int Cin, int Cout, int *wm, MarchGeo *m, int *shape,
                          TileGeo *t) {
  const long M = (long)B * D * H * W;
  if ((M >= 24576 || (M >= 16384 && M * Cout >= 1L << 20)) && march_geo(B, D, H, W, Cin, Cout, wm, m) &&
      march_fill(*m, *wm, D, H, W) < 4)
    return ConvForm::march;
  if ((Cin >= 64 || (Cin == 32 && M < 4096)) && tile_plan(B, D, H, W, Cin, Cout, shape, t)) {
    const double fill = tile_fill(*t, *shape, D, H, W);
    if (t->jobs < 512 || (t->jobs == 512 ? fill < 4 : fill < 1.5)) return ConvForm::tile;
  }
  return ConvForm::general;
}

// --------------------------------------------- weight gradient (k_conv_wgrad)

constexpr int kWgRuns = 16;
constexpr int kWgBufs = 3;      // units in LDS: one multiplies, two arrive
constexpr int kWgMaxVox = 288;  // LDS voxels of a unit's x: three units and two blocks a CU in 160 KB

struct WgGeo {
  int TX, nr, R, P;  // voxels of a line segment, its runs of 8, lines per plane, planes
  int halo;          // 1: segments of a longer line, loaded with their x neighbours
  int LP;            // LDS voxels per line: index i is x = xs + i - 1
  int nseg, nyb;     // segments per line, line groups per plane
  int npg, nunits;     // plane groups, units
  long planes;
  int xbytes, ybytes;  // of one LDS buffer, multiples of 1024
};

// Piece e (16 bytes, 8 channels) of a unit's x or dy in LDS, packed: its line,
// plane and x in the unit (x: of the loaded lines, which begin one voxel and
// one line before it), which 16 of a voxel's 32 channels, and bit 31 where
// there is nothing to load.  The half alternates with the 8-voxel block and
// the line, or the run, so that two runs' reads fall on distinct banks.
constexpr uint32_t kWgNoPiece = 0x80000000u;
LBMIB_HD uint32_t wg_pack(int l, int p, int ix, int h) { return (uint32_t)(l | p << 5 | ix << 10 | h << 17); }
LBMIB_HD int wg_line(uint32_t v) { return (int)(v & 31); }
LBMIB_HD int wg_plane(uint32_t v) { return (int)(v >> 5 & 31); }
LBMIB_HD int wg_x(uint32_t v) { return (int)(v >> 10 & 127); }
LBMIB_HD int wg_half(uint32_t v) { return (int)(v >> 17 & 1); }
LBMIB_HD uint32_t wg_x_piece(const WgGeo &q, int nb, int e) {
  const int pc = e & (2 * nb - 1), v = e / (2 * nb);
  const int i = v % q.LP, L = v / q.LP, l = L % (q.R + 2), p = L / (q.R + 2);
  if (p >= q.P) return kWgNoPiece;
  return wg_pack(l, p, i, nb == 2 ? (pc >> 1) ^ (((i >> 3) + L) & 1) : 0);
}
LBMIB_HD uint32_t wg_dy_piece(const WgGeo &q, int na, int e, int channels) {
  const int pc = e & (2 * na - 1), v = e / (2 * na), run = v >> 3;
  const int ix = (run % q.nr) * 8 + (v & 7), l = (run / q.nr) % q.R, p = run / (q.nr * q.R);
  const int h = na == 2 ? (pc >> 1) ^ (run & 1) : 0;
  return p < q.P && h * 16 < channels ? wg_pack(l, p, ix, h) : kWgNoPiece;
}
// Its element offset from the unit's first voxel in a tensor of C channels.
// (The half comes from its own bit: the offset's holds it only where voxels are
// whole 64-byte pieces, and dy has any multiple of 16 channels.)
LBMIB_HD long wg_piece_at(uint32_t v, int e, int H, int W, int C) {
  return (((long)wg_plane(v) * H + wg_line(v)) * W + wg_x(v)) * C + wg_half(v) * 16 + (e & 1) * 8;
}

// Lines of one voxel fill one in eight positions of a run.  Such a volume is
// the same memory as one whose lines run along y or z: (D, H, 1) as (D, 1, H),
// (D, 1, 1) as (1, 1, D), and B samples of one voxel as any volume of B voxels,
// of which only the centre tap counts.  The taps of the view become the
// layer's in wgrad_tap (4096 samples of one voxel, 256 -> 256: 634 us as they
// are, 45 so; 64 of 64 x 1 x 1, 128 -> 128: 130 and 26).
struct WgView {
  int B, D, H, W;
  int taps;  // 0 as they are, 1 y for x, 2 z for x, 3 the centre alone
};
inline WgView wgrad_view(int B, int D, int H, int W) {
  WgView v = {B, D, H, W, 0};
  if (W > 1) return v;
  if (H > 1) {
    v.H = 1, v.W = H, v.taps = 1;
  } else if (D > 1) {
    v.D = 1, v.W = D, v.taps = 2;
  } else if (B > 1) {
    v.B = 1, v.W = B, v.taps = 3;
    for (int w = 64; w >= 8; --w)  // lines of equal length, if there are such
      if (B % w == 0) {
        v.H = B / w, v.W = w;
        break;
      }
  }
  return v;
}
// The layer's tap (9 dz + 3 dy + dx, each 0..2) of the view's; -1: the sum is
// not one of the layer's, whose tap t is zero then.
LBMIB_HD int wgrad_tap(int taps, int t) {
  const int z = t / 9, y = t / 3 % 3, x = t % 3;
  if (taps == 1) return 9 * z + 3 * x + y;
  if (taps == 2) return 9 * x + 3 * y + z;
  return taps == 3 && t != 13 ? -1 : t;
}

// Units and split of the voxel reduction, from the shape only (so every entry
// point that shares it gives the same bits), capped so that the partials fit
// in `cap_bytes`.
struct WgradPlan {
  WgGeo q;
  int ci_tiles, tiles, splits, na, nb, ups;  // ups: units per split
  long n4;  // fragment quads of one split's partials
  size_t lds, part_bytes;
};

inline WgradPlan wgrad_plan(int B, int D, int H, int W, int Cin, int Cout, size_t cap_bytes) {
  WgradPlan p;
  WgGeo &q = p.q;
  // whole lines up to 64 voxels (an LDS line of at most 68), else 32-voxel
  // segments: 64-voxel ones with their two neighbours need a fifth round of
  // loads for 8 pieces
  q.halo = W > 64;
  q.TX = W > 64 ? 32 : (W + 7) / 8 * 8;
  q.nr = q.TX / 8;
  q.R = H < kWgRuns / q.nr ? H : kWgRuns / q.nr;
  q.nseg = (W + q.TX - 1) / q.TX;
  q.nyb = (H + q.R - 1) / q.R;
  q.planes = (long)B * D;
  q.P = 1;
  if (q.R == H && q.nseg == 1) {  // whole planes: as many as the runs hold
    const long fit = kWgRuns / (q.nr * q.R);
    q.P = (int)(fit < q.planes ? fit : q.planes);
    while (q.P > 1 && q.P * (q.R + 2) * (q.TX + 4) > kWgMaxVox) --q.P;
  }
  q.LP = q.TX + 4;
  q.npg = (int)((q.planes + q.P - 1) / q.P);
  q.nunits = q.npg * q.nyb * q.nseg;
  p.na = Cout >= 32 ? 2 : 1;
  p.nb = Cin >= 32 ? 2 : 1;
  q.xbytes = (q.P * (q.R + 2) * q.LP * 32 * p.nb + 1023) / 1024 * 1024;
  q.ybytes = kWgRuns * 8 * 32 * p.na;
  p.lds = ((size_t)kWgBufs * (q.xbytes + q.ybytes) + 12 * 32 * p.nb + 1023) / 1024 * 1024 + 1024;
  const size_t red = (size_t)4 * 3 * p.na * p.nb * 64 * 16;
  if (p.lds < red) p.lds = red;
  p.ci_tiles = (Cin + 31) / 32;
  p.tiles = p.ci_tiles * ((Cout + 31) / 32);
  p.n4 = (long)p.tiles * 27 * p.na * p.nb * 64;
  const size_t per_split = (size_t)p.n4 * 16 + (size_t)Cout * 4;
  // about 512 blocks, one round at 2 per CU
  long want = 512 / (3 * p.tiles);
  if (want < 1) want = 1;
  if (want > q.nunits) want = q.nunits;
  const long cap = (long)(cap_bytes / per_split);
  if (want > cap) want = cap;
  if (want < 1) want = 1;
  p.ups = (int)((q.nunits + want - 1) / want);
  p.splits = (q.nunits + p.ups - 1) / p.ups;
  p.part_bytes = per_split * p.splits;
  return p;
}

}  // namespace lbmib
