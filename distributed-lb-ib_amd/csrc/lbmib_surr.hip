// lbmib_surr.hip -- kernels of the learned surrogate (include/lbmib_surrogate.h):
// 3x3x3 convolutions on channels-last BF16 tensors with BF16 MFMA and FP32
// accumulation, their data and weight gradients, 2x pooling / upsampling, the
// loss, the optimiser and the packing of field planes.
//
// Convolutions are implicit GEMMs over voxels v, output channels n and the
// reduction index k = 27 taps x Cin input channels (tap-major, channel
// fastest, the weight layout [Cout][27][Cin]):
//   y[v][n] = sum_k W[n][k] X(v, k),   X(v, t*Cin + ci) = x[v + o(t)][ci]
// with o(t) the neighbour offset of tap t and zero outside the volume.  One
// v_mfma_f32_16x16x32_bf16 multiplies a 16 x 32 weight fragment (A: row n =
// lane & 15, k = 8 (lane >> 4) .. + 8) by a 32 x 16 input fragment (B:
// column v = lane & 15, the same 8 k), so that every lane fetches 8
// consecutive channels of one voxel (16 bytes) and of one weight row; the
// 16 x 16 result holds, per lane, 4 consecutive output channels of one voxel
// (rows 4 (lane >> 4) + r), stored as one 8-byte write.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "../../include/lbmib.h"
#include "../../include/lbmib_surrogate.h"
#include "lbmib_conv_plan.h"

using namespace lbmib;

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

#define HIPCHK(x)                                   \
  do {                                              \
    if ((x) != hipSuccess) return LBMIB_ERR_HIP;    \
  } while (0)

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
// round to nearest even (finite inputs; NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ bf16x8 ld8(const uint16_t *p) {
  return __builtin_bit_cast(bf16x8, *(const u32x4 *)p);
}
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u}); }

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------- forward
//
// Block: 4 waves stacked along the voxels; a wave owns WM x 16 voxels and
// WN x 16 output channels (WM x WN accumulator fragments).  The reduction
// runs over chunks of 32 k; the fragments of chunk c + 1 are loaded while
// chunk c multiplies.  Operands come straight from global memory (L1/L2):
// every voxel's 8-channel pieces are 16-byte aligned loads.
//
// SPLIT: the reduction is split over gridDim.z (chunks_per_split chunks
// each) and the block writes its FP32 partial sums to part[z][v][n] instead
// of the epilogue; k_conv_reduce then sums the partials in order of z.
template <int WM, int WN, bool SPLIT>
__global__ void __launch_bounds__(256) k_conv_fwd(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                                  const float *__restrict__ bias, const uint16_t *__restrict__ mask,
                                                  uint16_t *__restrict__ y, int D, int H, int W, long M, int Cin,
                                                  int lgCin, int Cout, int K, int relu, float *__restrict__ part,
                                                  int chunks_per_split) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, kq = lane >> 4;
  const long mw = ((long)blockIdx.x * 4 + wave) * (WM * 16);
  const int n0 = blockIdx.y * (WN * 16);
  const long HW = (long)H * W;
  int vz[WM], vy[WM], vx[WM];
  bool vin[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const long m = mw + i * 16 + col;
    vin[i] = m < M;
    long r = vin[i] ? m : 0;
    vx[i] = (int)(r % W);
    r /= W;
    vy[i] = (int)(r % H);
    r /= H;
    vz[i] = (int)(r % D);
  }
  f32x4 acc[WN][WM];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int i = 0; i < WM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  int c_begin = 0, c_end = (K + 31) >> 5;
  if (SPLIT) {
    c_begin = blockIdx.z * chunks_per_split;
    c_end = min(c_end, c_begin + chunks_per_split);
  }
  // The weight tile of a chunk (WN x 16 output channels x 32 k) is the same
  // for the block's four waves: it is loaded once per block, 16 bytes per
  // thread, into LDS (double-buffered, rows padded to 40 elements so that the
  // fragment reads of a wave spread over the banks); each wave reads its A
  // fragments from there.  The input fragments differ per wave and come
  // straight from L1/L2.
  constexpr int kPitch = 40;
  constexpr int kPieces = WN * 16 * 4;  // 16-byte pieces of a weight tile
  __shared__ __attribute__((aligned(16))) uint16_t sw[2][WN * 16 * kPitch];
  const int tid = threadIdx.x;
  const int prow = tid >> 2, pk = (tid & 3) << 3;  // this thread's piece: row, k offset
  u32x4 wpiece = {0u, 0u, 0u, 0u};
  auto load_w = [&](int c) {
    if (tid < kPieces) {
      const int k = (c << 5) + pk, n = n0 + prow;
      wpiece = (k < K && n < Cout) ? *(const u32x4 *)(w + (long)n * K + k) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  auto store_w = [&](int buf) {
    if (tid < kPieces) *(u32x4 *)(&sw[buf][prow * kPitch + pk]) = wpiece;
  };
  bf16x8 b[WM];
  auto load_x = [&](int c) {
    const int k = (c << 5) + (kq << 3);
    const bool kin = k < K;
    const int tap = k >> lgCin, ci = k & (Cin - 1);
    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int zz = vz[i] + dz, yy = vy[i] + dy, xx = vx[i] + dx;
      const bool ok = kin && vin[i] && (unsigned)zz < (unsigned)D && (unsigned)yy < (unsigned)H &&
                      (unsigned)xx < (unsigned)W;
      const long m = mw + i * 16 + col;
      b[i] = ok ? ld8(x + (m + dz * HW + (long)dy * W + dx) * Cin + ci) : zero8();
    }
  };
  if (c_begin < c_end) {
    load_w(c_begin);
    load_x(c_begin);
    store_w(0);
  }
  __syncthreads();
  for (int c = c_begin; c < c_end; ++c) {
    const int buf = (c - c_begin) & 1;
    bf16x8 cb[WM];
#pragma unroll
    for (int i = 0; i < WM; ++i) cb[i] = b[i];
    if (c + 1 < c_end) {
      load_w(c + 1);
      load_x(c + 1);
    }
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const bf16x8 ca = __builtin_bit_cast(bf16x8, *(const u32x4 *)(&sw[buf][(j * 16 + col) * kPitch + (kq << 3)]));
#pragma unroll
      for (int i = 0; i < WM; ++i) acc[j][i] = mfma16(ca, cb[i], acc[j][i]);
    }
    if (c + 1 < c_end) store_w(buf ^ 1);
    __syncthreads();
  }
  // epilogue: lane holds channels n0 + 16 j + 4 kq + r of voxel mw + 16 i + col
  if (SPLIT) {
    float *dst = part + (long)blockIdx.z * M * Cout;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int n = n0 + j * 16 + 4 * kq;
      if (n >= Cout) continue;
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        if (!vin[i]) continue;
        *(f32x4 *)(dst + (mw + i * 16 + col) * Cout + n) = acc[j][i];
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int n = n0 + j * 16 + 4 * kq;
    if (n >= Cout) continue;
    float bs[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias)
#pragma unroll
      for (int r = 0; r < 4; ++r) bs[r] = bias[n + r];
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      if (!vin[i]) continue;
      const long m = mw + i * 16 + col;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = acc[j][i][r] + bs[r];
        if (relu) v[r] = fmaxf(v[r], 0.f);
      }
      if (mask) {
        const u32x2 mk = *(const u32x2 *)(mask + m * Cout + n);
        const uint16_t mb[4] = {(uint16_t)(mk[0] & 0xffff), (uint16_t)(mk[0] >> 16), (uint16_t)(mk[1] & 0xffff),
                                (uint16_t)(mk[1] >> 16)};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!(bf2f(mb[r]) > 0.f)) v[r] = 0.f;
      }
      u32x2 o;
      o[0] = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
      o[1] = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
      *(u32x2 *)(y + m * Cout + n) = o;
    }
  }
}

// Forward convolution of few input channels (CI = 16 or 32) on lines of at
// most 64 voxels.  A block owns 16 WN output channels of 4 G lines (G of them
// a wave: G W <= 16 WM positions) and marches along z two planes at a time,
// four of its eight waves on each: the weights of all 27 taps stay in LDS in
// fragment order, and a ring of four z-planes holds the lines around the
// block's (the next two planes are loaded into registers while these
// multiply).  Each input voxel is thus staged once per (4 G + 2) / 4 G lines
// and the weights once per block, where a box of 8 channels at a time took 132 KB
// for every 256 voxels.
//
// A line's fragment of 16 voxels is read from LDS once for its three dx: the
// products with the weights of each dx go to accumulators of their own, acc[dx][u]
// = sum W[dx] x[u], and out[v] = sum over dx of acc[dx][v + dx] is formed by
// lane shifts at the end.  A whole line is in one wave, so nothing crosses
// waves, and beyond a line's ends there is nothing to add.  Per (dz, dy) a
// wave reads WM + 3 WN fragments for 3 WM WN MFMAs.
//
// Reduction slots 8 kq + e (kq = lane >> 4): CI = 32: channel 8 kq + e of one
// (dz, dy); CI = 16: channel 8 (kq & 1) + e of (dz, dy) number 2 c + (kq >> 1)
// in chunk c (the tenth is zero in both operands).
//
// The LDS holds one block, so two waves a SIMD: one's LDS reads and epilogue
// run beside the other's products (with four waves and one plane at a time
// they did not: 67 us where this takes 53).  Measured, with the former box
// form's
// times: 64^3 32 -> 32 at batch 4 53 us, 1089 TFLOP/s (92 us), at batch 1 18
// us (31); 48^3 32 -> 32 12.5 us (27); 32^3 32 -> 64 at batch 4 16 us (27).
// Matrix units are busy 43% of the time; the rest is the epilogue and, twice a
// step, the barriers around the exchange of planes.
// v of another lane of the row of 16, zero where there is none: the next
// lane's, the previous one's; lane 0's at lane 15 alone, lane 15's at lane 0
// alone.  Added to a sum, each is one v_add_f32 with a DPP operand.
template <int CTRL>
__device__ __forceinline__ float row_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int kFromNext = 0x101, kFromPrev = 0x111, kFirstToLast = 0x11f, kLastToFirst = 0x10f;

// BF16 bits of two floats, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}

template <int WM, int WN, int CI, bool WHOLE>
__global__ void __launch_bounds__(512, 2)
    k_conv_march(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, const float *__restrict__ bias,
                 const uint16_t *__restrict__ mask, uint16_t *__restrict__ y, MarchGeo q, int D, int H, int W, int Cout,
                 int relu) {
  constexpr int VX = 2 * CI, kChunks = CI == 32 ? 9 : 5, kWFrags = kChunks * 3 * WN;
  constexpr int kRounds = 3;  // 16-byte pieces of a plane per thread at most (CI = 16: two)
  constexpr uint32_t kNone = 0x80000000u;
  extern __shared__ __attribute__((aligned(16))) char sm[];  // weights, then the ring of planes
  const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, col = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wl4 = wave & 3;
  const long per = (q.jobs + 7) / 8;
  long job = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((long)(blockIdx.x >> 3) >= per || job >= q.jobs) return;
  const int ct = (int)(job % q.cot);
  job /= q.cot;
  const int zi = (int)(job % q.zs);
  job /= q.zs;
  const int yb = (int)(job % q.nyb);
  const long b = job / q.nyb;
  const int n0 = ct * (16 * WN), y0 = yb * 4 * q.G, z0 = zi * q.zc, z1 = min(z0 + q.zc, D);
  const int HW = H * W;
  char *ring = sm + kWFrags * 1024;

  // A plane's lines are contiguous, and those outside it lie outside the
  // resource, which reads zeros: a plane outside the volume has size zero.
  auto fetch = [&](int z, u32x4(&px)[kRounds]) {
    const bool in = z >= 0 && z < D;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(x + (b * D + (in ? z : 0)) * HW * CI), (short)0, in ? HW * VX : 0, 0x00020000);
    const int first = (y0 - 1) * W * VX + tid * 16;
#pragma unroll
    for (int k = 0; k < kRounds * CI / 32 + (CI == 16); ++k)
      px[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (uint32_t)(first + k * 8192), 0, 0));
  };
  auto put = [&](int z, const u32x4(&px)[kRounds]) {  // (a slot is whole waves of pieces)
    char *d = ring + (z & 3) * q.plane_bytes + tid * 16;
#pragma unroll
    for (int k = 0; k < kRounds * CI / 32 + (CI == 16); ++k)
      if (tid * 16 + k * 8192 < q.plane_bytes) *(u32x4 *)(d + k * 8192) = px[k];
  };
  u32x4 pa[kRounds], pb[kRounds];
  {
    // all of the first loads in flight together
    u32x4 pc[kRounds], pd[kRounds];
    fetch(z0 - 1, pa);
    fetch(z0, pb);
    fetch(z0 + 1, pc);
    fetch(z0 + 2, pd);
    // weights: fragment (chunk, dx, j), lane (row col, slots 8 kq ..)
    constexpr int kWRounds = (kWFrags + 7) / 8;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(w), (short)0,
                                                                      Cout * 27 * VX, 0x00020000);
    u32x4 pw[kWRounds];
#pragma unroll
    for (int k = 0; k < kWRounds; ++k) {
      const int f = 8 * k + wave, j = f % WN, dx = f / WN % 3, c = f / (3 * WN);
      const int line = CI == 32 ? c : 2 * c + (kq >> 1), n = n0 + 16 * j + col;
      const uint32_t o = line < 9 && n < Cout ? (uint32_t)((n * 27 + line * 3 + dx) * VX + (CI == 32 ? kq : kq & 1) * 16)
                                              : kNone;
      pw[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0));
    }
    put(z0 - 1, pa);
    put(z0, pb);
    put(z0 + 1, pc);
    put(z0 + 2, pd);
#pragma unroll
    for (int k = 0; k < kWRounds; ++k)
      if (8 * k + wave < kWFrags) *(u32x4 *)(sm + (8 * k + wave) * 1024 + lane * 16) = pw[k];
  }
  __syncthreads();

  float bs[WN][4];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + 16 * j + 4 * kq + r;
      bs[j][r] = bias && n < Cout ? bias[n] : 0.f;
    }
  // this lane's positions: byte offset of channels n0 + 4 kq in the plane of y
  uint32_t yo[WM];
  bool nxt[WM], prv[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int pos = 16 * i + col, xx = pos % W, lin = (y0 + wl4 * q.G) * W + pos;
    yo[i] = pos < q.G * W && lin < HW ? (uint32_t)((lin * Cout + n0 + 4 * kq) * 2) : kNone;
    nxt[i] = WHOLE ? (16 * i + 16) % W != 0 : xx < W - 1;
    prv[i] = WHOLE ? 16 * i % W != 0 : xx > 0;
  }
  const int bl = (wl4 * q.G * W + col) * VX + (CI == 32 ? kq : kq & 1) * 16;
  const char *wl = sm + lane * 16;
  for (int zp = z0; zp < z1; zp += 2) {
    const bool more = zp + 2 < z1;
    if (more) {
      fetch(zp + 3, pa);
      fetch(zp + 4, pb);
    }
    const int z = zp + (wave >> 2);
    if (z < z1) {
      const long pl = (b * D + z) * HW * Cout;
      u32x2 mk[WN][WM];
      const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(mask + pl), (short)0,
                                                                         mask ? HW * Cout * 2 : 0, 0x00020000);
      if (mask)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int i = 0; i < WM; ++i)
            mk[j][i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rm, yo[i], j * 32, 0));
      f32x4 acc[3][WN][WM];
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) {
          acc[0][j][i] = acc[2][j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
          acc[1][j][i] = f32x4{bs[j][0], bs[j][1], bs[j][2], bs[j][3]};
        }
#pragma unroll
      for (int c = 0; c < kChunks; ++c) {
        const char *p;
        if constexpr (CI == 32) {
          p = ring + ((z - 1 + c / 3) & 3) * q.plane_bytes + (c % 3) * W * VX + bl;
        } else {
          const int c1 = min(2 * c + 1, 8);
          const int o0 = ((z - 1 + 2 * c / 3) & 3) * q.plane_bytes + (2 * c % 3) * W * VX;
          const int o1 = ((z - 1 + c1 / 3) & 3) * q.plane_bytes + (c1 % 3) * W * VX;
          p = ring + (kq >> 1 ? o1 : o0) + bl;
        }
        bf16x8 bf[WM];
#pragma unroll
        for (int i = 0; i < WM; ++i) {
          bf[i] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(p + i * 16 * VX));
          if (CI == 16 && c == kChunks - 1 && kq >> 1) bf[i] = zero8();  // no tenth line: 0 times an infinity is NaN
        }
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
          for (int j = 0; j < WN; ++j) {
            const bf16x8 af = __builtin_bit_cast(bf16x8, *(const u32x4 *)(wl + ((c * 3 + dx) * WN + j) * 1024));
#pragma unroll
            for (int i = 0; i < WM; ++i) acc[dx][j][i] = mfma16(af, bf[i], acc[dx][j][i]);
          }
      }
      // a chunk's LDS reads between the products of the one before
      constexpr int kReads = WM + 3 * WN, kProds = 3 * WM * WN, kPer = kProds / kReads;
      __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
#pragma unroll
      for (int c = 1; c < kChunks; ++c) {
#pragma unroll
        for (int r = 0; r < kReads; ++r) {
          __builtin_amdgcn_sched_group_barrier(0x008, kPer, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, kProds - kPer * kReads, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, kProds, 0);
      const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y + pl, (short)0, HW * Cout * 2, 0x00020000);
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) {
          float v[4];
          if constexpr (WHOLE) {  // lines are whole fragments: a fragment's neighbours are its line's or add nothing
#pragma unroll
            for (int r = 0; r < 4; ++r)
              v[r] = acc[1][j][i][r] + row_shift<kFromNext>(acc[2][j][i][r]) + row_shift<kFromPrev>(acc[0][j][i][r]);
            if (i + 1 < WM && nxt[i])
#pragma unroll
              for (int r = 0; r < 4; ++r) v[r] += row_shift<kFirstToLast>(acc[2][j][i + 1 < WM ? i + 1 : i][r]);
            if (i > 0 && prv[i])
#pragma unroll
              for (int r = 0; r < 4; ++r) v[r] += row_shift<kLastToFirst>(acc[0][j][i > 0 ? i - 1 : 0][r]);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float up = row_shift<kFromNext>(acc[2][j][i][r]), dn = row_shift<kFromPrev>(acc[0][j][i][r]);
              if (i + 1 < WM) up += row_shift<kFirstToLast>(acc[2][j][i + 1 < WM ? i + 1 : i][r]);
              if (i > 0) dn += row_shift<kLastToFirst>(acc[0][j][i > 0 ? i - 1 : 0][r]);
              v[r] = acc[1][j][i][r] + (nxt[i] ? up : 0.f) + (prv[i] ? dn : 0.f);
            }
          }
          if (relu)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.f);
          if (mask) {
            const uint16_t mb[4] = {(uint16_t)(mk[j][i][0] & 0xffff), (uint16_t)(mk[j][i][0] >> 16),
                                    (uint16_t)(mk[j][i][1] & 0xffff), (uint16_t)(mk[j][i][1] >> 16)};
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (!(bf2f(mb[r]) > 0.f)) v[r] = 0.f;
          }
          const u32x2 o = {pack2(v[0], v[1]), pack2(v[2], v[3])};
          __builtin_amdgcn_raw_buffer_store_b64(o, ry, n0 + 16 * j < Cout ? yo[i] : kNone, j * 32, 0);
        }
    }
    if (more) {
      __syncthreads();  // the readers of the two oldest planes are done
      put(zp + 3, pa);
      put(zp + 4, pb);
      __syncthreads();
    }
  }
}

template <int WM, int WN, int CI>
int launch_march(const MarchGeo &q, const void *x, const void *w, const float *bias, const void *mask, void *y, int D,
                 int H, int W, int Cout, int relu, hipStream_t s) {
  const size_t shm = (CI == 32 ? 9 : 5) * 3 * WN * 1024 + 4 * (size_t)q.plane_bytes + 1024;
  auto go = [&](auto kern) {
    kern<<<(unsigned)((q.jobs + 7) / 8 * 8), 512, shm, s>>>((const uint16_t *)x, (const uint16_t *)w, bias,
                                                            (const uint16_t *)mask, (uint16_t *)y, q, D, H, W, Cout,
                                                            relu);
  };
  if (W % 16 == 0) go(k_conv_march<WM, WN, CI, true>);
  else go(k_conv_march<WM, WN, CI, false>);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

template <int CI>
int launch_march_any(int wm, const MarchGeo &q, const void *x, const void *w, const float *bias, const void *mask,
                     void *y, int D, int H, int W, int Cout, int relu, hipStream_t s) {
  if (Cout >= 32) {
    if (wm == 4) return launch_march<4, 2, CI>(q, x, w, bias, mask, y, D, H, W, Cout, relu, s);
    return launch_march<3, 2, CI>(q, x, w, bias, mask, y, D, H, W, Cout, relu, s);
  }
  if (wm == 4) return launch_march<4, 1, CI>(q, x, w, bias, mask, y, D, H, W, Cout, relu, s);
  return launch_march<3, 1, CI>(q, x, w, bias, mask, y, D, H, W, Cout, relu, s);
}

// Forward convolution of 32 or more input channels on lines of at most 64
// voxels (which layers take it is conv_form's to say).  A block owns a tile of LP lines x PZ planes (VG groups of G whole
// lines, 16 WM positions each) and 16 NC output channels.  It stages the box
// around the tile, (LP + 2) x (PZ + 2) lines with zeros outside the volume,
// for all input channels at once (or a slice at a time where that exceeds the
// LDS), and then multiplies without a barrier: its eight waves are NC channel
// groups x VG voxel groups x KW parts of the reduction.  The reduction goes by
// items, one (dz, dy) and 32 channels with its three dx: a wave reads the WM
// input fragments of an item from LDS once for the three dx (as in the march
// above: an accumulator per dx, joined by lane shifts at the end), and each of
// its three weight fragments, straight from L2 three items ahead, serves WM
// products.  The KW partial sums meet in LDS in a fixed order.
//
// Neighbouring lanes load pieces of one weight row, four to its 64 bytes, and
// pass them through 3 KB of LDS of the wave's own into fragment order: loaded
// in that order, with neighbouring lanes on different rows, every load took
// four times the cache lookups and they were the bound (120 us where this takes
// 105, at 24^3, 256 -> 256, batch 2).  LDS voxels are padded by 16 bytes, so
// that a fragment's 16 lanes read distinct banks.
//
// Measured, against the forms it replaced (boxes of 8 channels at a time,
// reductions split over blocks with partial sums in memory): 16^3, 128 -> 128
// at batch 4 20.2 us, 716 TFLOP/s (51.7 us), 64 -> 128 at batch 1 8.8 (13.8);
// 32^3, 64 -> 64 at batch 4 38 (59), at batch 1 14 (27); 8^3, 256 -> 256 at
// batch 1 8.8 (17.9), at batch 4 14.5 (31.5); 24^3, 256 -> 256 at batch 2 105
// (230).  The small ones are launch, first loads and the sum over KW; in the
// large ones the loads of a block's box, which nothing overlaps (one block a
// CU), and LDS reads beside the products.
// TAIL: some wave's share of the items is odd.  (With the odd item's code behind
// the loop, layers that do not need it took 2% longer: 24^3, 256 -> 256 at batch
// 2 104 us, 102 without.)
template <int WM, int NC, int KW, int VG, bool WHOLE, bool TAIL>
__global__ void __launch_bounds__(512, 2)
    k_conv_tile(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, const float *__restrict__ bias,
                const uint16_t *__restrict__ mask, uint16_t *__restrict__ y, TileGeo q, int D, int H, int W, int Cin,
                int Cout, int relu) {
  static_assert(NC * KW * VG == 8, "eight waves");
  constexpr uint32_t kNone = 0x80000000u;
  extern __shared__ __attribute__((aligned(16))) char sm[];  // the box, then 3 KB of weights per wave
  const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, col = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cg = wave % NC, vg = wave / NC % VG, kg = wave / (NC * VG);
  const long per = (q.jobs + 7) / 8;
  long job = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((long)(blockIdx.x >> 3) >= per || job >= q.jobs) return;
  const int ct = (int)(job % q.cot);
  job /= q.cot;
  const int ty = (int)(job % q.nty);
  job /= q.nty;
  const int tz = (int)(job % q.ntz);
  const long b = job / q.ntz;
  const int y0 = ty * q.LP, z0 = tz * q.PZ, n0 = (ct * NC + cg) * 16;
  const int BL = q.LP + 2, nlines = BL * (q.PZ + 2), pitch = q.cs * 2 + 16;
  const long S = (long)D * H * W;

  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(x + b * S * Cin), (short)0,
                                                                      (int)(S * Cin * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(w), (short)0,
                                                                      Cout * 27 * Cin * 2, 0x00020000);
  // items of a slice: (dz, dy) times 32-channel blocks; this wave's are kg, kg
  // + KW, ...  Nothing past the end is multiplied: zero weights would turn an
  // infinity of the voxels read in its place into NaN.
  const int lgc = q.lgp - 2, nitems = 9 << lgc;
  const int mine = TAIL ? (nitems - kg + KW - 1) / KW : nitems / KW;
  const uint32_t wb = n0 < Cout ? (uint32_t)((n0 + (lane >> 2)) * 27 * Cin * 2 + (lane & 3) * 16) : kNone;
  u32x4 wf[2][3];
  auto load_w = [&](int s, int n, int c0) {
    const int t = kg + KW * n, row = t >> lgc;
    const int o = (row * 3 * Cin + c0 + ((t & ((1 << lgc) - 1)) << 5)) * 2;
    const uint32_t at = t < nitems ? wb : kNone;
#pragma unroll
    for (int dx = 0; dx < 3; ++dx)
      wf[s][dx] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, at, o + dx * Cin * 2, 0));
  };
  // row r's four pieces lie in an order that spreads 8 or 16 rows' reads over all banks
  auto turn = [](int r) { return ((r >> 2) + (r & 2)) & 3; };
  char *wst = sm + q.box + wave * 3072;
  const int wput = (lane >> 2) * 64 + (((lane & 3) ^ turn(lane >> 2)) << 4), wget = col * 64 + ((kq ^ turn(col)) << 4);
  bf16x8 wa[2][3];
  auto swap_w = [&](int s) {  // from the order of the loads into the fragments'
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) *(u32x4 *)(wst + dx * 1024 + wput) = wf[s][dx];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) wa[s][dx] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(wst + dx * 1024 + wget));
    __builtin_amdgcn_wave_barrier();
  };
  // LDS offset of item n's lines and channels relative to the voxel's own
  auto item_off = [&](int n) {
    const int t = min(kg + KW * n, nitems - 1), row = t >> lgc;
    return (row / 3 * BL + row % 3) * W * pitch + ((t & ((1 << lgc) - 1)) << 6);
  };

  // positions
  int at[WM];
  uint32_t yo[WM];
  bool nxt[WM], prv[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const TilePos t = tile_pos(q, W, vg, 16 * i + col);
    const bool out = t.in && z0 + t.pz < D && y0 + t.ly < H;
    at[i] = (t.in ? ((t.pz * BL + t.ly) * W + t.x) * pitch : 0) + kq * 16;
    yo[i] = out ? (uint32_t)(((((z0 + t.pz) * H + y0 + t.ly) * W + t.x) * Cout + n0 + 4 * kq) * 2) : kNone;
    nxt[i] = WHOLE ? (16 * i + 16) % W != 0 : t.x < W - 1;
    prv[i] = WHOLE ? 16 * i % W != 0 : t.x > 0;
  }
  f32x4 acc[3][WM];
#pragma unroll
  for (int dx = 0; dx < 3; ++dx)
#pragma unroll
    for (int i = 0; i < WM; ++i) acc[dx][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int c0 = 0; c0 < Cin; c0 += q.cs) {
    load_w(0, 0, c0);
    load_w(1, 1, c0);
    if (c0) __syncthreads();  // the readers of the previous slice are done
    {
      // lines wave, wave + 8, ... of the box, 64 pieces at a time
      constexpr int kBatch = 8;
      const int np = W << q.lgp, rounds = (np + 63) >> 6;
      int ln = wave, bp = 0, ly = wave, r = 0;
      while (ly >= BL) ly -= BL, ++bp;
      while (ln < nlines) {
        u32x4 px[kBatch];
        int dst[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const int e = (r << 6) + lane, v = e >> q.lgp, pc = e & ((1 << q.lgp) - 1);
          const int yy = y0 - 1 + ly, zz = z0 - 1 + bp;
          const bool have = ln < nlines && e < np;
          const bool in = have && (unsigned)yy < (unsigned)H && (unsigned)zz < (unsigned)D;
          const uint32_t src = in ? (uint32_t)((((zz * H + yy) * W + v) * Cin + c0) * 2 + pc * 16) : kNone;
          px[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, src, 0, 0));
          dst[k] = have ? (ln * W + v) * pitch + pc * 16 : -1;
          if (++r == rounds) {
            r = 0;
            ln += 8;
            ly += 8;
            while (ly >= BL) ly -= BL, ++bp;
          }
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
          if (dst[k] >= 0) *(u32x4 *)(sm + dst[k]) = px[k];
      }
    }
    __syncthreads();
    bf16x8 bf[WM];
    {
      const int o = item_off(0);
#pragma unroll
      for (int i = 0; i < WM; ++i) bf[i] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(sm + at[i] + o));
    }
    swap_w(0);
    load_w(0, 2, c0);
    auto multiply = [&](int n, int s) {  // item n from wa[s] and bf; item n + 1 follows in wa[s ^ 1]
      const int o = item_off(n + 1);
      swap_w(s ^ 1);
      load_w(s ^ 1, n + 3, c0);
#pragma unroll
      for (int i = 0; i < WM; ++i) {
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) acc[dx][i] = mfma16(wa[s][dx], bf[i], acc[dx][i]);
        bf[i] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(sm + at[i] + o));
      }
      __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 3, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 1; i < WM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    };
    for (int rd = 0; rd < mine >> 1; ++rd) {
#pragma unroll
      for (int s = 0; s < 2; ++s) multiply(rd * 2 + s, s);
    }
    if (TAIL && mine & 1) {
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) acc[dx][i] = mfma16(wa[0][dx], bf[i], acc[dx][i]);
    }
  }

  // out[v] = sum over dx of acc[dx][v + dx - 1] within v's line
  f32x4 sum[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (WHOLE) {
        float v = acc[1][i][r] + row_shift<kFromNext>(acc[2][i][r]) + row_shift<kFromPrev>(acc[0][i][r]);
        if (i + 1 < WM && nxt[i]) v += row_shift<kFirstToLast>(acc[2][i + 1 < WM ? i + 1 : i][r]);
        if (i > 0 && prv[i]) v += row_shift<kLastToFirst>(acc[0][i > 0 ? i - 1 : 0][r]);
        sum[i][r] = v;
      } else {
        float up = row_shift<kFromNext>(acc[2][i][r]), dn = row_shift<kFromPrev>(acc[0][i][r]);
        if (i + 1 < WM) up += row_shift<kFirstToLast>(acc[2][i + 1 < WM ? i + 1 : i][r]);
        if (i > 0) dn += row_shift<kLastToFirst>(acc[0][i > 0 ? i - 1 : 0][r]);
        sum[i][r] = acc[1][i][r] + (nxt[i] ? up : 0.f) + (prv[i] ? dn : 0.f);
      }
    }
  f32x4 *red = (f32x4 *)sm;  // [kg][fragment of the (cg, vg) group][lane]
  if constexpr (KW > 1) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WM; ++i) red[((kg * NC * VG + wave % (NC * VG)) * WM + i) * 64 + lane] = sum[i];
    __syncthreads();
  }
  if (n0 >= Cout) return;
  float bs[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) bs[r] = bias ? bias[n0 + 4 * kq + r] : 0.f;
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y + b * S * Cout, (short)0, (int)(S * Cout * 2),
                                                                      0x00020000);
  const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(mask + b * S * Cout),
                                                                      (short)0, mask ? (int)(S * Cout * 2) : 0,
                                                                      0x00020000);
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    if (KW > 1 && i % KW != kg) continue;  // each of the KW waves finishes its share of the fragments
    u32x2 mk = {0u, 0u};
    if (mask) mk = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rm, yo[i], 0, 0));
    f32x4 t = sum[i];
    if constexpr (KW > 1) {
      t = red[((wave % (NC * VG)) * WM + i) * 64 + lane];
#pragma unroll
      for (int k = 1; k < KW; ++k) t += red[((k * NC * VG + wave % (NC * VG)) * WM + i) * 64 + lane];
    }
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = t[r] + bs[r];
      if (relu) v[r] = fmaxf(v[r], 0.f);
    }
    if (mask) {
      const uint16_t mb[4] = {(uint16_t)(mk[0] & 0xffff), (uint16_t)(mk[0] >> 16), (uint16_t)(mk[1] & 0xffff),
                              (uint16_t)(mk[1] >> 16)};
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!(bf2f(mb[r]) > 0.f)) v[r] = 0.f;
    }
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])}, ry, yo[i], 0, 0);
  }
}

template <int WM, int NC, int KW, int VG>
int launch_tile(const TileGeo &q, const void *x, const void *w, const float *bias, const void *mask, void *y, int D,
                int H, int W, int Cin, int Cout, int relu, hipStream_t s) {
  auto go = [&](auto kern) {
    kern<<<(unsigned)((q.jobs + 7) / 8 * 8), 512, q.lds, s>>>((const uint16_t *)x, (const uint16_t *)w, bias,
                                                              (const uint16_t *)mask, (uint16_t *)y, q, D, H, W, Cin,
                                                              Cout, relu);
  };
  const bool tail = 9 * (q.cs / 32) % (2 * KW) != 0;
  if (W % 16 == 0) {
    if (tail) go(k_conv_tile<WM, NC, KW, VG, true, true>);
    else go(k_conv_tile<WM, NC, KW, VG, true, false>);
  } else {
    if (tail) go(k_conv_tile<WM, NC, KW, VG, false, true>);
    else go(k_conv_tile<WM, NC, KW, VG, false, false>);
  }
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

int launch_tile_any(int shape, const TileGeo &q, const void *x, const void *w, const float *bias, const void *mask,
                    void *y, int D, int H, int W, int Cin, int Cout, int relu, hipStream_t s) {
  switch (shape) {
    case 0: return launch_tile<8, 8, 1, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 1: return launch_tile<8, 4, 1, 2>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 2: return launch_tile<8, 2, 1, 4>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 3: return launch_tile<8, 4, 2, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 4: return launch_tile<8, 2, 4, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 5: return launch_tile<8, 1, 8, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 6: return launch_tile<4, 4, 2, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 7: return launch_tile<4, 2, 2, 2>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 8: return launch_tile<4, 2, 4, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case 9: return launch_tile<4, 1, 8, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    default: return launch_tile<2, 1, 8, 1>(q, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
  }
}

// Small-grid forward convolution: the KW waves of a block all own the same
// WM x 16 voxels x WN x 16 output channels and split the reduction between
// them -- wave w multiplies chunks w, w + KW, w + 2 KW, ... of 32 k.  Both
// operands come straight from global memory (L1/L2) into a ring of P
// register stages, so that P chunks' loads are in flight while one
// multiplies, and the loop has no barrier.  The loads are raw buffer loads
// whose resources end at the tensors' ends: a lane with nothing to load
// (a neighbour outside the volume, k past 27 Cin) points its offset past
// the end and the hardware returns zeros, so the loads carry no branch and
// the waits stay per stage.  At the end the KW partial sums
// meet in LDS and are added in wave order (a fixed order: the result does
// not depend on timing), then bias, activation and mask as in k_conv_fwd.
// One launch per layer, where a split over blocks needs a second pass over
// FP32 partials in memory.
template <int WM, int WN, int KW, int P>
__global__ void __launch_bounds__(KW * 64) k_conv_fwd_kw(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                                         const float *__restrict__ bias,
                                                         const uint16_t *__restrict__ mask, uint16_t *__restrict__ y,
                                                         int D, int H, int W, long M, int Cin, int lgCin, int Cout,
                                                         int K, int relu) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kq = lane >> 4;
  const long mb = (long)blockIdx.x * (WM * 16);
  const int n0 = blockIdx.y * (WN * 16);
  const long HW = (long)H * W;
  int vz[WM], vy[WM], vx[WM];
  bool vin[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const long m = mb + i * 16 + col;
    vin[i] = m < M;
    long r = vin[i] ? m : 0;
    vx[i] = (int)(r % W);
    r /= W;
    vy[i] = (int)(r % H);
    r /= H;
    vz[i] = (int)(r % D);
  }
  f32x4 acc[WN][WM];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int i = 0; i < WM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nch = (K + 31) >> 5;
  const int nw = nch > wave ? (nch - wave + KW - 1) / KW : 0;  // this wave's chunks
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(w), (short)0,
                                                                      Cout * K * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(x), (short)0,
                                                                      (int)(M * Cin * 2), 0x00020000);
  constexpr uint32_t kNone = 0x80000000u;  // past the end of both resources: loads zeros
  bf16x8 a[P][WN], b[P][WM];
  // stage s <- the wave's t-th chunk; slot 8 kq + e of a fragment is k = 32 c + 8 kq + e
  auto load = [&](int s, int t) {
    const int k = ((wave + t * KW) << 5) + (kq << 3);
    const bool kin = k < K;
    // k past 27 Cin needs no test on this side: the input slot is zero
    // there (the weights are finite), and past the end of w the load is zero
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const uint32_t off = (uint32_t)(((n0 + j * 16 + col) * K + k) * 2);
      a[s][j] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0));
    }
    const int tap = k >> lgCin, ci = k & (Cin - 1);
    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int zz = vz[i] + dz, yy = vy[i] + dy, xx = vx[i] + dx;
      const bool ok = kin && vin[i] && (unsigned)zz < (unsigned)D && (unsigned)yy < (unsigned)H &&
                      (unsigned)xx < (unsigned)W;
      const int m = (int)mb + i * 16 + col;
      const uint32_t off = ok ? (uint32_t)(((m + dz * (int)HW + dy * W + dx) * Cin + ci) * 2) : kNone;
      b[s][i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
    }
  };
#pragma unroll
  for (int s = 0; s < P; ++s) load(s, s);
  for (int t0 = 0; t0 < nw; t0 += P) {
#pragma unroll
    for (int s = 0; s < P; ++s) {
      if (t0 + s < nw) {
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int i = 0; i < WM; ++i) acc[j][i] = mfma16(a[s][j], b[s][i], acc[j][i]);
      }
      load(s, t0 + s + P);
    }
  }
  // the waves' partial sums, fragment f = j WM + i, lane l
  __shared__ f32x4 red[KW][WN * WM][64];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int i = 0; i < WM; ++i) red[wave][j * WM + i][lane] = acc[j][i];
  __syncthreads();
  for (int e = threadIdx.x; e < WN * WM * 64; e += KW * 64) {
    const int f = e >> 6, l = e & 63;
    const int j = f / WM, i = f % WM;
    f32x4 sum = red[0][f][l];
#pragma unroll
    for (int v = 1; v < KW; ++v) sum += red[v][f][l];
    // lane l of fragment (j, i): channels n0 + 16 j + 4 (l >> 4) + r of voxel mb + 16 i + (l & 15)
    const int n = n0 + j * 16 + 4 * (l >> 4);
    const long m = mb + i * 16 + (l & 15);
    if (n >= Cout || m >= M) continue;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = sum[r] + (bias ? bias[n + r] : 0.f);
      if (relu) v[r] = fmaxf(v[r], 0.f);
    }
    if (mask) {
      const u32x2 mk = *(const u32x2 *)(mask + m * Cout + n);
      const uint16_t mbits[4] = {(uint16_t)(mk[0] & 0xffff), (uint16_t)(mk[0] >> 16), (uint16_t)(mk[1] & 0xffff),
                                 (uint16_t)(mk[1] >> 16)};
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!(bf2f(mbits[r]) > 0.f)) v[r] = 0.f;
    }
    u32x2 o;
    o[0] = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
    o[1] = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
    *(u32x2 *)(y + m * Cout + n) = o;
  }
}

template <int WM, int WN, int KW, int P>
int launch_fwd_kw(const void *x, const void *w, const float *bias, const void *mask, void *y, int D, int H, int W,
                  long M, int Cin, int Cout, int relu, hipStream_t s) {
  const dim3 grid((unsigned)((M + WM * 16 - 1) / (WM * 16)), (unsigned)((Cout + WN * 16 - 1) / (WN * 16)));
  k_conv_fwd_kw<WM, WN, KW, P><<<grid, KW * 64, 0, s>>>((const uint16_t *)x, (const uint16_t *)w, bias,
                                                        (const uint16_t *)mask, (uint16_t *)y, D, H, W, M, Cin,
                                                        ilog2(Cin), Cout, 27 * Cin, relu);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

// y[v][n] = act(sum over z < ns of part[z][v][n] + bias[n]) [* (mask > 0)]:
// one thread per (voxel, 4 channels)
__global__ void k_conv_reduce(const float *__restrict__ part, int ns, const float *__restrict__ bias,
                              const uint16_t *__restrict__ mask, uint16_t *__restrict__ y, long M, int Cout, int relu) {
  const long nq = M * (Cout / 4);
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < nq; e += (long)gridDim.x * blockDim.x) {
    const long off = e * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < ns; ++z) s += *(const f32x4 *)(part + (long)z * M * Cout + off);
    const int n = (int)(off % Cout);
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = s[r] + (bias ? bias[n + r] : 0.f);
      if (relu) v[r] = fmaxf(v[r], 0.f);
    }
    if (mask) {
      const u32x2 mk = *(const u32x2 *)(mask + off);
      const uint16_t mb[4] = {(uint16_t)(mk[0] & 0xffff), (uint16_t)(mk[0] >> 16), (uint16_t)(mk[1] & 0xffff),
                              (uint16_t)(mk[1] >> 16)};
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!(bf2f(mb[r]) > 0.f)) v[r] = 0.f;
    }
    u32x2 o;
    o[0] = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
    o[1] = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
    *(u32x2 *)(y + off) = o;
  }
}

int workspace(void **out);

// ksplit > 1: split reduction through the library workspace
template <int WM, int WN>
int launch_fwd(const void *x, const void *w, const float *bias, const void *mask, void *y, int D, int H, int W, long M,
               int Cin, int Cout, int relu, int ksplit, hipStream_t s) {
  const int K = 27 * Cin;
  const long bm = 4L * WM * 16;
  const int nch = (K + 31) / 32;
  dim3 grid((unsigned)((M + bm - 1) / bm), (unsigned)((Cout + WN * 16 - 1) / (WN * 16)));
  if (ksplit <= 1) {
    k_conv_fwd<WM, WN, false><<<grid, 256, 0, s>>>((const uint16_t *)x, (const uint16_t *)w, bias,
                                                    (const uint16_t *)mask, (uint16_t *)y, D, H, W, M, Cin,
                                                    ilog2(Cin), Cout, K, relu, nullptr, nch);
    HIPCHK(hipGetLastError());
    return LBMIB_OK;
  }
  void *ws = nullptr;
  const int rc = workspace(&ws);
  if (rc) return rc;
  const int cps = (nch + ksplit - 1) / ksplit;
  grid.z = (nch + cps - 1) / cps;
  k_conv_fwd<WM, WN, true><<<grid, 256, 0, s>>>((const uint16_t *)x, (const uint16_t *)w, nullptr, nullptr, nullptr,
                                                 D, H, W, M, Cin, ilog2(Cin), Cout, K, relu, (float *)ws, cps);
  HIPCHK(hipGetLastError());
  const long nq = M * (Cout / 4);
  long nb = (nq + 255) / 256;
  if (nb > 4096) nb = 4096;
  k_conv_reduce<<<(unsigned)nb, 256, 0, s>>>((const float *)ws, (int)grid.z, bias, (const uint16_t *)mask,
                                              (uint16_t *)y, M, Cout, relu);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

bool shape_ok(int B, int D, int H, int W, int Cin, int Cout) {
  if (B < 1 || D < 1 || H < 1 || W < 1) return false;
  if (Cin < 16 || Cin > 256 || (Cin & (Cin - 1))) return false;
  if (Cout < 16 || Cout > 512 || Cout % 16) return false;
  const long M = (long)B * D * H * W;
  return M * (long)(Cin > Cout ? Cin : Cout) < (1L << 40);
}

int conv_fwd(const void *x, const void *w, const float *bias, const void *mask, void *y, int B, int D, int H, int W,
             int Cin, int Cout, int relu, hipStream_t s) {
  if (!x || !w || !y || !shape_ok(B, D, H, W, Cin, Cout)) return LBMIB_ERR_ARG;
  const long M = (long)B * D * H * W;
  MarchGeo mg;
  TileGeo tg;
  int wm = 4, shape = 0;
  switch (conv_form(B, D, H, W, Cin, Cout, &wm, &mg, &shape, &tg)) {
    case ConvForm::march:
      return Cin == 32 ? launch_march_any<32>(wm, mg, x, w, bias, mask, y, D, H, W, Cout, relu, s)
                       : launch_march_any<16>(wm, mg, x, w, bias, mask, y, D, H, W, Cout, relu, s);
    case ConvForm::tile:
      return launch_tile_any(shape, tg, x, w, bias, mask, y, D, H, W, Cin, Cout, relu, s);
    case ConvForm::general: break;
  }
  // lines longer than 64 voxels, few channels on small grids, and many samples
  // or planes too narrow for the forms above.  Wave
  // tiles: 4 x 16 voxels when the grid is large, fewer when the voxel count
  // alone cannot fill the device; 64 channels per block (32 / 16 for the
  // narrow layers)
  const int wn = Cout % 64 == 0 ? 4 : (Cout % 32 == 0 ? 2 : 1);
  const long blocks64 = (M + 255) / 256 * (Cout / (16 * wn));
  if (blocks64 >= 512) {
    if (wn == 4) return launch_fwd<4, 4>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, 1, s);
    if (wn == 2) return launch_fwd<4, 2>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, 1, s);
    return launch_fwd<4, 1>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, 1, s);
  }
  // small grids whose weights stay modest: the two waves of a block split
  // the reduction of one 32-voxel tile, one launch and no partial sums in
  // memory; the weights are read once per tile, at most 128 MB in all
  const double kw_bytes = (double)((M + 31) / 32) * Cout * 27 * Cin * 2;
  if ((M >= 4096 || Cin == 16) && kw_bytes <= 128e6 && M * Cin * 2 < (1L << 31)) {
    if (wn == 4) return launch_fwd_kw<2, 4, 2, 2>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, s);
    if (wn == 2) return launch_fwd_kw<2, 2, 2, 2>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, s);
    return launch_fwd_kw<2, 1, 2, 2>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, s);
  }
  // small grids: split the reduction so that about 1024 blocks run, each
  // with at least 4 chunks of 32, within the workspace
  const long blocks = (M + 63) / 64 * (Cout / (16 * wn));
  const int nch = (27 * Cin + 31) / 32;
  long ks = (1024 + blocks - 1) / blocks;
  if (ks > nch / 4) ks = nch / 4;
  const long cap = (long)(LBMIB_SG_WORKSPACE_BYTES / ((size_t)M * Cout * sizeof(float)));
  if (ks > cap) ks = cap;
  if (ks < 1) ks = 1;
  if (wn == 4) return launch_fwd<1, 4>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, (int)ks, s);
  if (wn == 2) return launch_fwd<1, 2>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, (int)ks, s);
  return launch_fwd<1, 1>(x, w, bias, mask, y, D, H, W, M, Cin, Cout, relu, (int)ks, s);
}

// wt[ci][26 - t][co] = w[co][t][ci]
// One 64 x 64 tile of one tap: rows of w come and rows of wt go in 16-byte
// pieces through LDS (one element per lane wrote wt in 2-byte pieces, 27 Cout
// apart: 15.3 us for 256 x 256 channels, and 83 us in a launch for each of a
// network's 14 layers; 7.5 us now, in one launch for the list).
constexpr int kFlipTile = 64;
constexpr int kFlipMax = 32;  // layers per launch
struct FlipItem {
  const uint16_t *w;
  uint16_t *wt;
  int Cin, Cout, first, vec;  // first block; both pointers on 16 bytes
};
struct FlipList {
  FlipItem it[kFlipMax];
  int n;
};

static inline int flip_blocks(int Cin, int Cout) {
  return 27 * ((Cin + kFlipTile - 1) / kFlipTile) * ((Cout + kFlipTile - 1) / kFlipTile);
}

__global__ void __launch_bounds__(256) k_flip(FlipList l) {
  __shared__ uint16_t tile[kFlipTile][kFlipTile + 2];
  int k = 0;
  while (k + 1 < l.n && (int)blockIdx.x >= l.it[k + 1].first) ++k;
  const FlipItem it = l.it[k];
  const int Cin = it.Cin, Cout = it.Cout;
  const int nci = (Cin + kFlipTile - 1) / kFlipTile;
  int b = blockIdx.x - it.first;
  const int t = b % 27;
  b /= 27;
  const int ci0 = b % nci * kFlipTile, co0 = b / nci * kFlipTile;
  for (int e = threadIdx.x; e < kFlipTile * kFlipTile / 8; e += 256) {
    const int co = e / 8, ci = e % 8 * 8;
    if (co0 + co >= Cout || ci0 + ci >= Cin) continue;
    const uint16_t *src = it.w + ((long)(co0 + co) * 27 + t) * Cin + ci0 + ci;
    alignas(16) uint16_t v[8];
    if (it.vec) {
      *(u32x4 *)v = *(const u32x4 *)src;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = src[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[co][ci + j] = v[j];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kFlipTile * kFlipTile / 8; e += 256) {
    const int ci = e / 8, co = e % 8 * 8;
    if (co0 + co >= Cout || ci0 + ci >= Cin) continue;
    uint16_t *dst = it.wt + ((long)(ci0 + ci) * 27 + (26 - t)) * Cout + co0 + co;
    alignas(16) uint16_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = tile[co + j][ci];
    if (it.vec) {
      *(u32x4 *)dst = *(const u32x4 *)v;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) dst[j] = v[j];
    }
  }
}

static int flip_list(int n, const lbmib_sg_flip_item *items, hipStream_t s) {
  for (int k0 = 0; k0 < n; k0 += kFlipMax) {
    FlipList l;
    l.n = n - k0 < kFlipMax ? n - k0 : kFlipMax;
    int blocks = 0;
    for (int k = 0; k < l.n; ++k) {
      const lbmib_sg_flip_item &q = items[k0 + k];
      l.it[k] = FlipItem{(const uint16_t *)q.w, (uint16_t *)q.wt, q.Cin, q.Cout, blocks,
                         (((uintptr_t)q.w | (uintptr_t)q.wt) & 15) == 0};
      blocks += flip_blocks(q.Cin, q.Cout);
    }
    k_flip<<<blocks, 256, 0, s>>>(l);
    HIPCHK(hipGetLastError());
  }
  return LBMIB_OK;
}

// ----------------------------------------------------------- weight grad
//
// dw[co][t][ci] = sum_v dy[v][co] x[v + o(t)][ci]: per tap a GEMM whose
// reduction runs over voxels.  A block owns a 32 x 32 (co, ci) tile (16 for
// 16-channel tensors), the 9 taps of one dz and a contiguous range of units;
// its 4 waves each multiply a quarter of a unit's voxels for all 9 taps (9 x
// NA x NB accumulator fragments), and add up through LDS at the end.
//
// A unit is up to 128 voxels as 16 runs of 8 consecutive x (lane group kq =
// lane >> 4 of wave w takes run 4w + kq as its 8 reduction slots): R whole
// lines of a z-plane, P whole planes where a plane is small, or R lines of a
// 32-voxel x segment where a line is longer than 64.  The unit's dy and the
// lines of x around it at plane z + dz are staged in LDS channel-fastest, as
// they lie in memory, zeros outside the volume; ds_read_b64_tr_b16 hands each
// lane 4 consecutive voxels of its channel, so an operand fragment is two
// 8-byte reads where gathering it takes eight 2-byte ones and the packing.
// Three such reads hold the 12 voxels from one before the run on: taps dx =
// -1 and +1 are registers of them as they are, dx = 0 four v_alignbit.
//
// 36 MFMAs per wave and unit against 22 LDS reads, each group of 6 products
// behind the next group's 3 reads.  The units come by direct loads from memory
// to LDS, two ahead of the one that multiplies, with no register and no store
// on the way (through registers only one unit ahead fitted, with 36 bytes of
// spills).  Alone, the loads take 67 us and the products 70 at batch 4 x 64^3,
// 32 -> 32 channels: each dz fetches its own x and dy, 600 MB from L2.
//
// Measured, against the form with one unit ahead through registers: 98 us
// (593 TFLOP/s) for 139 at batch 4 x 64^3, 32 -> 32; 53 for 74 at 32^3, 64 ->
// 64; 38 for 46 at 16^3, 128 -> 128; 203 for 275 at batch 2 x 24^3, 256 -> 256.
// 16 bytes per lane from r + off to LDS at + 16 lane, without registers in
// between; zeros where off lies past the resource.  Nothing waits: dma_wait.
// (The builtin makes the compiler wait for every such load before the next LDS
// read, whichever buffer it reads.  m0 is among the clobbers so that nothing
// the compiler puts there is expected to survive; it warns that the register
// is reserved.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(u32x4 r, uint32_t off, uint32_t at) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, 0 offen lds"
      :
      : "s"(at), "v"(off), "s"(r)
      : "memory", "m0");
}
#pragma clang diagnostic pop
// all but the last N loads have arrived, and this wave's LDS reads are done
template <int N>
__device__ __forceinline__ void dma_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ u32x4 rsrc_words(const void *p) {
  const uint64_t a = (uint64_t)p;
  return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)((a >> 32) & 0xffff)), 0x7fffffffu, 0x00020000u};
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 4 voxels of one channel: lane i of each 16 passes the address of row
// (i & 15) >> 2 (a voxel), channels 4 (i & 3) .. + 3, and receives rows 0..3
// of channel i & 15.
__device__ __forceinline__ u32x2 lds_tr4(const char *p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p));
}

template <int NA, int NB, bool BIG>
__global__ void __launch_bounds__(256, 2)
    k_conv_wgrad(const uint16_t *__restrict__ x, const uint16_t *__restrict__ dy, float *__restrict__ part,
                 float *__restrict__ bpart, WgGeo q, int D, int H, int W, int Cin, int Cout, int ci_tiles, int tiles,
                 int splits, int units_per_split) {
  constexpr int VX = 32 * NB, VY = 32 * NA;  // bytes per voxel in LDS
  constexpr uint32_t kNone = 0x80000000u;    // past the end of the resources: loads zeros
  constexpr int KX = (kWgMaxVox * VX / 1024 + 3) / 4, KY = kWgRuns * 8 * VY / 4096;  // DMA instructions per wave and unit
  // three buffers of x and dy, 12 voxels of zeros, 1 KB that nothing reads
  extern __shared__ __attribute__((aligned(1024))) char sm[];
  const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup b runs on XCD b % 8: the three dz of a split and tile, which
  // read the same dy and neighbouring planes of x, follow each other there.
  const int jobs = tiles * 3 * splits, per = (jobs + 7) / 8;
  const int job = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || job >= jobs) return;
  const int dzi = job % 3, tile = (job / 3) % tiles, split = job / (3 * tiles);
  const int ci0 = (tile % ci_tiles) * 32, co0 = (tile / ci_tiles) * 32;
  const int buf_bytes = q.xbytes + q.ybytes, zeros_at = kWgBufs * buf_bytes;
  const uint32_t unread_at = (uint32_t)(zeros_at + 12 * VX + 1023) / 1024 * 1024;

  // Instruction k of a wave fills the 1024 bytes number wave + 4 k of a
  // buffer's x (and of its dy): this lane's piece of it, where it lies in
  // memory relative to the unit, and (in one register, wg_x_piece) line, plane,
  // x and half, which decide whether it exists
  uint32_t xo[KX], yo[KY], xl[KX], yl[KY];
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    const int e = (wave + 4 * k) * 64 + lane;
    xl[k] = wg_x_piece(q, NB, e);
    xo[k] = (uint32_t)(wg_piece_at(xl[k], e, H, W, Cin) * 2);
  }
#pragma unroll
  for (int k = 0; k < KY; ++k) {
    const int e = (wave + 4 * k) * 64 + lane;
    yl[k] = wg_dy_piece(q, NA, e, Cout - co0);
    yo[k] = (uint32_t)(wg_piece_at(yl[k], e, H, W, Cout) * 2);
  }
  // this lane's run: LDS addresses of its x (line dy = -1) and dy operands
  const int run = 4 * wave + kq, rx = run % q.nr, rl = (run / q.nr) % q.R, rp = run / (q.nr * q.R);
  const bool has_run = rp < q.P;
  const int rowb = (lane & 15) >> 2, colb = (lane & 3) * 8;
  const int L0 = rp * (q.R + 2) + rl;
  const int xa0 = (L0 * q.LP + 8 * rx + rowb) * VX + colb, xs0 = NB == 2 ? ((rx + L0) & 1) * 32 : 0;
  const int ya0 = q.xbytes + (run * 8 + rowb) * VY + colb, ys0 = NA == 2 ? (run & 1) * 32 : 0;
  const int zero_at = zeros_at + rowb * VX + colb;
  const bool tails = q.halo || (W & 7);  // lines whose last run is not full

  // The unit sequence: plane groups first, so that a plane of x that one dz
  // reads is still in L2 when the next two do; then line groups, segments.  (A
  // single plane whose z + dz lies outside the volume adds nothing and is
  // passed by.)
  const int u_begin = split * units_per_split, u_end = min(u_begin + units_per_split, q.nunits);
  struct Unit {
    int u, pg, sg, yb, z0;  // z0: the first plane's z
  };
  auto step = [&](Unit &t) {
    ++t.u;
    t.z0 += q.P;
    if (++t.pg == q.npg) {
      t.pg = t.z0 = 0;
      if (++t.yb == q.nyb) {
        t.yb = 0;
        ++t.sg;
      }
    }
    while (t.z0 >= D) t.z0 -= D;
  };
  auto skip = [&](Unit &t) {
    if (q.P == 1)
      while (t.u < u_end && (unsigned)(t.z0 + dzi - 1) >= (unsigned)D) step(t);
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)sm;
  auto issue = [&](const Unit &t, int buf) {
    const long pl = (long)t.pg * q.P;
    // the planes that exist at z + dz, by their number in the unit
    uint32_t zin = 1, yin = 1;
    if (q.P > 1) {
      zin = yin = 0;
      for (int p = 0, z = t.z0; p < q.P && pl + p < q.planes; ++p) {
        yin |= 1u << p;
        if ((unsigned)(z + dzi - 1) < (unsigned)D) zin |= 1u << p;
        if (++z == D) z = 0;
      }
    }
    const int y0 = t.yb * q.R, xs = t.sg * q.TX;
    const uint16_t *bx = x + (((pl + dzi - 1) * H + y0 - 1) * W + xs - 1) * Cin + ci0;
    const uint16_t *by = dy + ((pl * H + y0) * W + xs) * Cout + co0;
    const u32x4 rx_ = rsrc_words(bx), ry_ = rsrc_words(by);
    const uint32_t at0 = lds0 + buf * buf_bytes;
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      const int l = wg_line(xl[k]), p = wg_plane(xl[k]), ix = wg_x(xl[k]), at = (wave + 4 * k) * 1024;
      const bool ok = !(xl[k] & kWgNoPiece) & ((unsigned)(y0 - 1 + l) < (unsigned)H) &
                      ((unsigned)(xs - 1 + ix) < (unsigned)W) & (bool)(zin >> p & 1);
      if constexpr (BIG) {
        const uint16_t *src = ok ? bx + wg_piece_at(xl[k], lane, H, W, Cin) : x;
        const u32x4 v = ok ? *(const u32x4 *)src : u32x4{0u, 0u, 0u, 0u};
        if (at < q.xbytes) *(u32x4 *)(sm + buf * buf_bytes + at + lane * 16) = v;
      } else {
        dma16(rx_, ok ? xo[k] : kNone, at < q.xbytes ? at0 + at : lds0 + unread_at);
      }
    }
#pragma unroll
    for (int k = 0; k < KY; ++k) {
      const int l = wg_line(yl[k]), p = wg_plane(yl[k]), ix = wg_x(yl[k]), at = q.xbytes + (wave + 4 * k) * 1024;
      const bool ok = !(yl[k] & kWgNoPiece) & (y0 + l < H) & (xs + ix < W) & (bool)(yin >> p & 1);
      if constexpr (BIG) {
        const uint16_t *src = ok ? by + wg_piece_at(yl[k], lane, H, W, Cout) : dy;
        *(u32x4 *)(sm + buf * buf_bytes + at + lane * 16) = ok ? *(const u32x4 *)src : u32x4{0u, 0u, 0u, 0u};
      } else {
        dma16(ry_, ok ? yo[k] : kNone, at0 + at);
      }
    }
  };

  f32x4 acc[9][NA][NB], accb[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    accb[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[t][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bool want_b = bpart && dzi == 1 && ci0 == 0;  // this block also sums dy over the voxels
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});

  if (tid * 16 < 12 * VX) *(u32x4 *)(sm + zeros_at + tid * 16) = u32x4{0u, 0u, 0u, 0u};
  Unit cur = {u_begin, u_begin % q.npg, u_begin / q.npg / q.nyb, u_begin / q.npg % q.nyb, 0};
  cur.z0 = (int)((long)cur.pg * q.P % D);
  skip(cur);
  Unit ahead = cur;  // the next unit to fetch
  int left = 0, buf = 0;
  for (; left < kWgBufs - 1 && ahead.u < u_end; ++left) {
    issue(ahead, left);
    step(ahead);
    skip(ahead);
  }
  while (left > 0) {
    // this unit's pieces are here (those of the one after may be on their
    // way), and every wave is done with the buffer that is filled next
    if (left > 1) dma_wait<KX + KY>();
    else dma_wait<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    --left;
    if (ahead.u < u_end) {
      issue(ahead, buf == 0 ? kWgBufs - 1 : buf - 1);
      step(ahead);
      skip(ahead);
      ++left;
    }
    // the lanes whose run lies past the unit or the plane multiply zeros by zeros
    const bool in = has_run && cur.yb * q.R + rl < H;
    const int boff = buf * buf_bytes;
    const int xa = in ? boff + xa0 : zero_at, lstep = in ? q.LP * VX : 0, xs1 = in ? xs0 : 0;
    u32x4 tm = {~0u, ~0u, ~0u, ~0u};  // clears x[last voxel] where dx = -1 pairs it with a voxel past the line
    if (tails) {
      const int e0 = W - cur.sg * q.TX - 8 * rx;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (e0 == k) tm[k >> 1] = k & 1 ? 0x0000ffffu : 0xffff0000u;
    }
    step(cur);
    skip(cur);
    bf16x8 fa[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const char *p = sm + boff + ya0 + ((32 * a) ^ ys0);
      const u32x2 lo = lds_tr4(p), hi = lds_tr4(p + 4 * VY);
      fa[a] = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
    // groups of 3 reads and 3 NA products, a group's reads before the products
    // of the one before
    u32x2 v[2][3];
    auto read = [&](int g) {
      // (the half of a voxel's channels alternates with the 8-voxel block and
      // the line, so that two runs' reads fall on distinct banks)
      const int d = g / NB, h = NB == 2 ? 32 * ((g % NB + d) & 1) : 0;
      const char *p = sm + xa + d * lstep;
      const int here = h ^ xs1, next = NB == 2 ? here ^ 32 : 0;
      v[g & 1][0] = lds_tr4(p + here);
      v[g & 1][1] = lds_tr4(p + here + 4 * VX);
      v[g & 1][2] = lds_tr4(p + (in ? next : 0) + 8 * VX);
    };
    read(0);
#pragma unroll
    for (int g = 0; g < 3 * NB; ++g) {
      if (g + 1 < 3 * NB) read(g + 1);
      const int d = g / NB, b = g % NB;
      const u32x2 v0 = v[g & 1][0], v1 = v[g & 1][1], v2 = v[g & 1][2];
      u32x4 m = {v0[0], v0[1], v1[0], v1[1]};
      const u32x4 c = {__builtin_amdgcn_alignbit(v0[1], v0[0], 16), __builtin_amdgcn_alignbit(v1[0], v0[1], 16),
                       __builtin_amdgcn_alignbit(v1[1], v1[0], 16), __builtin_amdgcn_alignbit(v2[0], v1[1], 16)};
      const u32x4 n = {v0[1], v1[0], v1[1], v2[0]};
      if (tails) m &= tm;
      const bf16x8 fm = __builtin_bit_cast(bf16x8, m), fc = __builtin_bit_cast(bf16x8, c),
                   fn = __builtin_bit_cast(bf16x8, n);
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        acc[3 * d][a][b] = mfma16(fa[a], fm, acc[3 * d][a][b]);
        acc[3 * d + 1][a][b] = mfma16(fa[a], fc, acc[3 * d + 1][a][b]);
        acc[3 * d + 2][a][b] = mfma16(fa[a], fn, acc[3 * d + 2][a][b]);
      }
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * NA + 6, 0);
#pragma unroll
    for (int g = 0; g + 2 < 3 * NB; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 3 * NA, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 6 * NA, 0);
    if (want_b)
#pragma unroll
      for (int a = 0; a < NA; ++a) accb[a] = mfma16(fa[a], ones, accb[a]);
    buf = buf == kWgBufs - 1 ? 0 : buf + 1;
  }
  __syncthreads();
  // the four waves' sums, one dy at a time, added in wave order; partials
  // fragment by fragment: lane holds (co = co0 + 16 a + 4 kq + r, ci = ci0 +
  // 16 b + (lane & 15))
  constexpr int NF = 3 * NA * NB;
  f32x4 *red = (f32x4 *)sm;
  f32x4 *dst = (f32x4 *)part + (((long)split * tiles + tile) * 3 + dzi) * (3 * NF * 64);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) red[(wave * NF + (t * NA + a) * NB + b) * 64 + lane] = acc[3 * d + t][a][b];
    __syncthreads();
    for (int e = tid; e < NF * 64; e += 256)
      dst[d * NF * 64 + e] = (red[e] + red[NF * 64 + e]) + (red[2 * NF * 64 + e] + red[3 * NF * 64 + e]);
    __syncthreads();
  }
  if (want_b) {  // every column of the product with ones is the sum
    if ((lane & 15) == 0)
#pragma unroll
      for (int a = 0; a < NA; ++a) red[(wave * NA + a) * 4 + kq] = accb[a];
    __syncthreads();
    const float *rf = (const float *)red;
    if (tid < 16 * NA && co0 + tid < Cout)
      bpart[(long)split * Cout + co0 + tid] = (rf[tid] + rf[16 * NA + tid]) + (rf[32 * NA + tid] + rf[48 * NA + tid]);
  }
}

// dw from the splits' partials (fragment order, see k_conv_wgrad) and db from
// theirs, in a fixed order.  A block covers 16 fragment quads (256 contiguous
// bytes per split); its 16 thread groups take every 16th split, four loads
// in flight at a time, and add up through LDS in group order.  The blocks
// past the weights' take 16 channels of the bias each.  (19 MB: 5.7 us for both
// gradients; one thread walking a quarter of the splits with two loads in
// flight took 23 us for 28 MB, and the bias 34 us in two launches of its own.)
template <int NA, int NB>
__global__ void __launch_bounds__(256) k_wgrad_sum(const float *__restrict__ part, const float *__restrict__ bpart,
                                                   float *__restrict__ dw, float *__restrict__ db, int splits, int Cin,
                                                   int Cout, int ci_tiles, long n4, int taps) {
  __shared__ f32x4 red[16][17];
  const int tid = threadIdx.x, el = tid & 15, g = tid >> 4;
  const long e = (long)blockIdx.x * 16 + el;
  const bool is_w = e < n4;  // uniform: n4 is a multiple of 16
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (is_w) {
    const f32x4 *p = (const f32x4 *)part + e;
    int k = g;
    for (; k + 48 < splits; k += 64) {
      const f32x4 a = p[k * n4], b = p[(k + 16) * n4], c = p[(k + 32) * n4], d = p[(k + 48) * n4];
      s += (a + b) + (c + d);
    }
    for (; k < splits; k += 16) s += p[k * n4];
  } else if (e - n4 < Cout) {
    for (int k = g; k < splits; k += 16) s[0] += bpart[(long)k * Cout + (e - n4)];
  }
  red[g][el] = s;
  __syncthreads();
  if (g) return;
  for (int k = 1; k < 16; ++k) s += red[k][el];
  if (!is_w) {
    if (e - n4 < Cout) db[e - n4] = s[0];
    return;
  }
  const int lane = (int)(e & 63), f = (int)(e >> 6), b = f % NB, a = f / NB % NA, tv = f / (NB * NA) % 27;
  const int tl = wgrad_tap(taps, tv), t = tl < 0 ? tv : tl;
  if (tl < 0) s = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tile = f / (27 * NA * NB);
  const int ci = (tile % ci_tiles) * 32 + 16 * b + (lane & 15);
  const int co = (tile / ci_tiles) * 32 + 16 * a + 4 * (lane >> 4);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (co + r < Cout) dw[((long)(co + r) * 27 + t) * Cin + ci] = s[r];
}

template <int NA, int NB>
int launch_wgrad(const WgradPlan &p, const void *x, const void *dy, float *dw, float *db, const WgView &v, int Cin,
                 int Cout, float *part, hipStream_t s) {
  const int D = v.D, H = v.H, W = v.W;
  float *bpart = db ? part + (size_t)p.n4 * 4 * p.splits : nullptr;
  const int jobs = p.tiles * 3 * p.splits;
  auto go = [&](auto kern) {
    kern<<<(jobs + 7) / 8 * 8, 256, p.lds, s>>>((const uint16_t *)x, (const uint16_t *)dy, part, bpart, p.q, D, H, W, Cin,
                                                Cout, p.ci_tiles, p.tiles, p.splits, p.ups);
  };
  // byte offsets within a unit take 32 bits unless its lines are enormous
  const long span = (long)p.q.P * (p.q.R + 2) * W * (Cin > Cout ? Cin : Cout) * 2;
  if (span < (1L << 31)) go(k_conv_wgrad<NA, NB, false>);
  else go(k_conv_wgrad<NA, NB, true>);
  HIPCHK(hipGetLastError());
  const unsigned nb = (unsigned)(p.n4 / 16 + (db ? (Cout + 15) / 16 : 0));
  k_wgrad_sum<NA, NB><<<nb, 256, 0, s>>>(part, bpart, dw, db, p.splits, Cin, Cout, p.ci_tiles, p.n4,
                                          v.taps);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

int wgrad_with(const void *x, const void *dy, float *dw, float *db, int B, int D, int H, int W, int Cin, int Cout,
               void *ws, size_t ws_bytes, hipStream_t s) {
  const WgView v = wgrad_view(B, D, H, W);
  const WgradPlan p = wgrad_plan(v.B, v.D, v.H, v.W, Cin, Cout, ws_bytes);
  if (p.part_bytes > ws_bytes || p.q.nunits < 1) return LBMIB_ERR_ARG;
  float *part = (float *)ws;
  if (p.na == 2 && p.nb == 2) return launch_wgrad<2, 2>(p, x, dy, dw, db, v, Cin, Cout, part, s);
  if (p.na == 2) return launch_wgrad<2, 1>(p, x, dy, dw, db, v, Cin, Cout, part, s);
  if (p.nb == 2) return launch_wgrad<1, 2>(p, x, dy, dw, db, v, Cin, Cout, part, s);
  return launch_wgrad<1, 1>(p, x, dy, dw, db, v, Cin, Cout, part, s);
}

// The library's workspace: one buffer per device, allocated on first use.
constexpr int kMaxDevices = 64;
void *g_ws[kMaxDevices] = {};
std::mutex g_ws_mu;

// Scratch of lbmib_sg_conv3d_bwd_weight_noalloc: a file-scope device array
// that every GPU the library runs on holds until the process ends.  In host
// code its name is not a device address; each device's own copy is reached
// through the address hipGetSymbolAddress returns with that device current,
// kept per device in g_scratch.
static __device__ __align__(256) float scratch[LBMIB_SG_NOALLOC_SCRATCH_BYTES / sizeof(float)];
void *g_scratch[kMaxDevices] = {};
std::mutex g_scratch_mu;

int scratch_ptr(void **out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return LBMIB_ERR_ARG;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return LBMIB_ERR_HIP;
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return LBMIB_OK;
}

int workspace(void **out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return LBMIB_ERR_ARG;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  if (!g_ws[dev]) {
    void *p = nullptr;
    if (hipMalloc(&p, LBMIB_SG_WORKSPACE_BYTES) != hipSuccess) return LBMIB_ERR_ALLOC;
    g_ws[dev] = p;
  }
  *out = g_ws[dev];
  return LBMIB_OK;
}

// lbmib_sg_sqdiff's block partials (two doubles for each of at most
// kSqBlocks blocks): a buffer of their own, one per device, so that the
// sums a caller takes on one stream never share memory with a network
// running on another stream through the workspace.
constexpr int kSqBlocks = 1024;
void *g_sq[kMaxDevices] = {};

int sq_partials(void **out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return LBMIB_ERR_ARG;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  if (!g_sq[dev]) {
    void *p = nullptr;
    if (hipMalloc(&p, sizeof(double) * 2 * kSqBlocks) != hipSuccess) return LBMIB_ERR_ALLOC;
    g_sq[dev] = p;
  }
  *out = g_sq[dev];
  return LBMIB_OK;
}

// ------------------------------------------------------------ elementwise
//
// One thread per (voxel, 8-channel piece); C is a multiple of 16.

template <class I>
__global__ void k_pool2(const uint16_t *__restrict__ x, uint16_t *__restrict__ y, unsigned D, unsigned H, unsigned W, unsigned C, I n) {
  const I P = C / 8;
  for (I e = (I)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (I)gridDim.x * blockDim.x) {
    const I q = e % P;
    I r = e / P;
    const I ox = r % W;
    r /= W;
    const I oy = r % H;
    r /= H;
    const I oz = r % D;
    const I b = r / D;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const I iz = 2 * oz + (c >> 2), iy = 2 * oy + ((c >> 1) & 1), ix = 2 * ox + (c & 1);
      const I v = ((b * 2 * D + iz) * 2 * H + iy) * 2 * W + ix;
      const u32x4 val = *(const u32x4 *)(x + (size_t)v * C + q * 8);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        acc[2 * k] += bf2f((uint16_t)(val[k] & 0xffff));
        acc[2 * k + 1] += bf2f((uint16_t)(val[k] >> 16));
      }
    }
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o[k] = (uint32_t)f2bf(acc[2 * k] * 0.125f) | ((uint32_t)f2bf(acc[2 * k + 1] * 0.125f) << 16);
    *(u32x4 *)(y + (size_t)e * 8) = o;
  }
}

__device__ __forceinline__ void unpack8(u32x4 v, float f[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = bf2f((uint16_t)(v[k] & 0xffff));
    f[2 * k + 1] = bf2f((uint16_t)(v[k] >> 16));
  }
}
__device__ __forceinline__ u32x4 pack8(const float f[8]) {
  u32x4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = (uint32_t)f2bf(f[2 * k]) | ((uint32_t)f2bf(f[2 * k + 1]) << 16);
  return o;
}

// voxel index of the parent (D, H, W fine dims) of fine voxel v
template <class I>
__device__ __forceinline__ I parent_of(I v, unsigned D, unsigned H, unsigned W) {
  const I x = v % W;
  I r = v / W;
  const I y = r % H;
  r /= H;
  const I z = r % D;
  const I b = r / D;
  return ((b * (D / 2) + z / 2) * (H / 2) + y / 2) * (W / 2) + x / 2;
}

template <class I>
__global__ void k_up2_add(const uint16_t *__restrict__ c, const uint16_t *__restrict__ e, uint16_t *__restrict__ s,
                          unsigned D, unsigned H, unsigned W, unsigned C, I n) {
  const I P = C / 8;
  for (I i = (I)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (I)gridDim.x * blockDim.x) {
    const I q = i % P;
    const I v = i / P;
    const I u = parent_of<I>(v, D, H, W);
    float a[8], b[8];
    unpack8(*(const u32x4 *)(c + (size_t)u * C + q * 8), a);
    if (e) {
      unpack8(*(const u32x4 *)(e + (size_t)i * 8), b);
#pragma unroll
      for (int k = 0; k < 8; ++k) a[k] += b[k];
    }
    *(u32x4 *)(s + (size_t)i * 8) = pack8(a);
  }
}

template <class I>
__global__ void k_pool2_bwd(const uint16_t *__restrict__ a, const uint16_t *__restrict__ g,
                            const uint16_t *__restrict__ mask, uint16_t *__restrict__ out, unsigned D, unsigned H, unsigned W, unsigned C,
                            I n) {
  const I P = C / 8;
  for (I i = (I)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (I)gridDim.x * blockDim.x) {
    const I q = i % P;
    const I v = i / P;
    const I u = parent_of<I>(v, D, H, W);
    float f[8], t[8];
    unpack8(*(const u32x4 *)(g + (size_t)u * C + q * 8), f);
#pragma unroll
    for (int k = 0; k < 8; ++k) f[k] *= 0.125f;
    if (a) {
      unpack8(*(const u32x4 *)(a + (size_t)i * 8), t);
#pragma unroll
      for (int k = 0; k < 8; ++k) f[k] += t[k];
    }
    if (mask) {
      unpack8(*(const u32x4 *)(mask + (size_t)i * 8), t);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (!(t[k] > 0.f)) f[k] = 0.f;
    }
    *(u32x4 *)(out + (size_t)i * 8) = pack8(f);
  }
}

template <class I>
__global__ void k_up2_bwd(const uint16_t *__restrict__ ds, const uint16_t *__restrict__ mask,
                          uint16_t *__restrict__ out, unsigned D, unsigned H, unsigned W, unsigned C, I n) {
  const I P = C / 8;
  for (I i = (I)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (I)gridDim.x * blockDim.x) {
    const I q = i % P;
    I r = i / P;
    const I ox = r % W;
    r /= W;
    const I oy = r % H;
    r /= H;
    const I oz = r % D;
    const I b = r / D;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, t[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const I iz = 2 * oz + (c >> 2), iy = 2 * oy + ((c >> 1) & 1), ix = 2 * ox + (c & 1);
      const I v = ((b * 2 * D + iz) * 2 * H + iy) * 2 * W + ix;
      unpack8(*(const u32x4 *)(ds + (size_t)v * C + q * 8), t);
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[k] += t[k];
    }
    if (mask) {
      unpack8(*(const u32x4 *)(mask + (size_t)i * 8), t);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (!(t[k] > 0.f)) acc[k] = 0.f;
    }
    *(u32x4 *)(out + (size_t)i * 8) = pack8(acc);
  }
}

// loss partials (per block) and the gradient
__global__ void __launch_bounds__(256) k_mse(const uint16_t *__restrict__ out, const float *__restrict__ tgt,
                                             uint16_t *__restrict__ dout, float *__restrict__ part, long M, int C,
                                             int nl, float gscale) {
  __shared__ float red[256];
  float s = 0.f;
  const long n = M * C;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const int c = (int)(e % C);
    const long v = e / C;
    float gval = 0.f;
    if (c < nl) {
      const float d = bf2f(out[e]) - tgt[v * nl + c];
      s += d * d;
      gval = gscale * d;
    }
    dout[e] = f2bf(gval);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) k_final_sum(const float *__restrict__ part, int n, float scale,
                                                   float *__restrict__ out) {
  __shared__ float r[256];
  float s = 0.f;
  for (int k = threadIdx.x; k < n; k += 256) s += part[k];
  r[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) r[threadIdx.x] += r[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = r[0] * scale;
}

// The same for C a multiple of 8 and 16-byte pointers: one lane takes 8
// channels (one element per lane and 64-bit divisions took 47.7 us for 4 x 64^3
// voxels of 16 channels, 22.6 now).
__global__ void __launch_bounds__(256) k_mse8(const uint16_t *__restrict__ out, const float *__restrict__ tgt,
                                              uint16_t *__restrict__ dout, float *__restrict__ part, unsigned n,
                                              unsigned P, int nl, float gscale) {
  __shared__ float red[256];
  float s = 0.f;
  for (unsigned e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
    const unsigned v = e / P;
    const int c0 = (int)(e - v * P) * 8;
    float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c0 < nl) {
      unpack8(*(const u32x4 *)(out + (size_t)e * 8), f);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float d = 0.f;
        if (c0 + k < nl) d = f[k] - tgt[(size_t)v * nl + c0 + k];
        s += d * d;
        f[k] = gscale * d;
      }
    }
    *(u32x4 *)(dout + (size_t)e * 8) = pack8(f);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam on a list of tensors in one launch (a launch per tensor took 3 to 11 us
// for each of a network's 30, 106 us in all; 28 now, 7.4 TB/s): every block takes
// 1024 elements of one tensor, 16 bytes per lane where its pointers allow.
constexpr int kAdamMax = 32;  // tensors per launch
struct AdamItem {
  float *p;
  const float *g;
  float *m, *v;
  uint16_t *w16;
  long n;
  unsigned first;  // first block
  int vec;         // every pointer on 16 bytes (w16: 8)
};
struct AdamList {
  AdamItem it[kAdamMax];
  int n;
};

__device__ __forceinline__ float adam_one(float p, float gr, float &m, float &v, float lr, float b1, float b2,
                                          float eps, float c1, float c2) {
  m = b1 * m + (1.f - b1) * gr;
  v = b2 * v + (1.f - b2) * gr * gr;
  return p - lr * (m / c1) / (sqrtf(v / c2) + eps);
}

__global__ void __launch_bounds__(256) k_adam(AdamList l, float lr, float b1, float b2, float eps, float c1,
                                              float c2) {
  int k = 0;
  while (k + 1 < l.n && blockIdx.x >= l.it[k + 1].first) ++k;
  const AdamItem it = l.it[k];
  const long e0 = (long)(blockIdx.x - it.first) * 1024 + threadIdx.x * 4;
  if (it.vec && e0 + 4 <= it.n) {
    f32x4 p = *(const f32x4 *)(it.p + e0), m = *(const f32x4 *)(it.m + e0), v = *(const f32x4 *)(it.v + e0);
    const f32x4 g = *(const f32x4 *)(it.g + e0);
    uint16_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float mj = m[j], vj = v[j];
      p[j] = adam_one(p[j], g[j], mj, vj, lr, b1, b2, eps, c1, c2);
      m[j] = mj;
      v[j] = vj;
      w[j] = f2bf(p[j]);
    }
    *(f32x4 *)(it.m + e0) = m;
    *(f32x4 *)(it.v + e0) = v;
    *(f32x4 *)(it.p + e0) = p;
    if (it.w16) *(uint2 *)(it.w16 + e0) = make_uint2(w[0] | (uint32_t)w[1] << 16, w[2] | (uint32_t)w[3] << 16);
    return;
  }
  for (long e = e0; e < it.n && e < e0 + 4; ++e) {
    float m = it.m[e], v = it.v[e];
    const float p = adam_one(it.p[e], it.g[e], m, v, lr, b1, b2, eps, c1, c2);
    it.m[e] = m;
    it.v[e] = v;
    it.p[e] = p;
    if (it.w16) it.w16[e] = f2bf(p);
  }
}

static int adam_list(int n, const lbmib_sg_adam_item *items, float lr, float b1, float b2, float eps, int t,
                     hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  for (int k = 0; k < n;) {
    AdamList l;
    l.n = 0;
    long blocks = 0;
    for (; k < n && l.n < kAdamMax; ++k) {
      const lbmib_sg_adam_item &q = items[k];
      const long nb = (q.n + 1023) / 1024;
      if (nb > 0x7fffffffL) return LBMIB_ERR_ARG;
      if (blocks + nb > 0x7fffffffL) break;
      const uintptr_t bits = (uintptr_t)q.p | (uintptr_t)q.g | (uintptr_t)q.m | (uintptr_t)q.v;
      l.it[l.n++] = AdamItem{q.p, q.g, q.m, q.v, (uint16_t *)q.w16, q.n, (unsigned)blocks,
                             (bits & 15) == 0 && ((uintptr_t)q.w16 & 7) == 0};
      blocks += nb;
    }
    k_adam<<<(unsigned)blocks, 256, 0, s>>>(l, lr, b1, b2, eps, c1, c2);
    HIPCHK(hipGetLastError());
  }
  return LBMIB_OK;
}

__global__ void k_cast(const float *__restrict__ src, uint16_t *__restrict__ dst, long n) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    dst[e] = f2bf(src[e]);
}

struct Norm16 {
  float a[16], b[16];
};

__global__ void k_pack(const float *__restrict__ f, int nf, Norm16 nm, int nconst, uint16_t *__restrict__ x, long M,
                       int C) {
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < M; v += (long)gridDim.x * blockDim.x) {
    for (int c0 = 0; c0 < C; c0 += 8) {
      float t[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int c = c0 + k;
        float val = 0.f;
        if (c < nf)
          val = (f[(long)c * M + v] - nm.a[c]) * nm.b[c];
        else if (c < nf + nconst)
          val = nm.a[c];
        t[k] = val;
      }
      *(u32x4 *)(x + v * C + c0) = pack8(t);
    }
  }
}

__global__ void k_target(const float *__restrict__ f0, const float *__restrict__ f1, int nl, Norm16 nm,
                         float *__restrict__ tgt, long M) {
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < M; v += (long)gridDim.x * blockDim.x)
    for (int c = 0; c < nl; ++c) {
      const long i = (long)c * M + v;
      tgt[v * nl + c] = ((f1[i] - f0[i]) - nm.a[c]) * nm.b[c];
    }
}

__global__ void k_unpack(const uint16_t *__restrict__ out, int C, int nl, Norm16 nm, float *__restrict__ d, long M) {
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < M; v += (long)gridDim.x * blockDim.x)
    for (int c = 0; c < nl; ++c) d[(long)c * M + v] = bf2f(out[v * C + c]) * nm.b[c] + nm.a[c];
}

__global__ void __launch_bounds__(256) k_sqdiff(const float *__restrict__ a, const float *__restrict__ b, long n,
                                                double *__restrict__ part) {
  __shared__ double r0[256], r1[256];
  double s0 = 0.0, s1 = 0.0;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const double av = a[e];
    if (b) {
      const double bv = b[e];
      s0 += (av - bv) * (av - bv);
      s1 += bv * bv;
    } else {
      s0 += av * av;
    }
  }
  r0[threadIdx.x] = s0;
  r1[threadIdx.x] = s1;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r0[threadIdx.x] += r0[threadIdx.x + w];
      r1[threadIdx.x] += r1[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r0[0];
    part[2 * blockIdx.x + 1] = r1[0];
  }
}

// one block of 256: strided partial sums, then a fixed tree (deterministic)
__global__ void __launch_bounds__(256) k_sqdiff_final(const double *__restrict__ part, int nb,
                                                      double *__restrict__ out2) {
  __shared__ double r0[256], r1[256];
  double s0 = 0.0, s1 = 0.0;
  for (int k = threadIdx.x; k < nb; k += 256) {
    s0 += part[2 * k];
    s1 += part[2 * k + 1];
  }
  r0[threadIdx.x] = s0;
  r1[threadIdx.x] = s1;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r0[threadIdx.x] += r0[threadIdx.x + w];
      r1[threadIdx.x] += r1[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out2[0] = r0[0];
    out2[1] = r1[0];
  }
}

// Launches a kernel over n 8-channel pieces with a 32-bit index where the
// indices of the finer grid fit too, for the divisions that place a piece
// (up2_add of 4 x 32^3 x 64 channels 9.5 -> 8.1 us, of 64^3 x 32 10.2 -> 9.0).
template <class Fn>
void pool_launch(long n, Fn fn) {
  if (n < (1L << 29)) fn((unsigned)n);
  else fn(n);
}

unsigned grid_for(long n, int per_block = 256, long cap = 8192) {
  long g = (n + per_block - 1) / per_block;
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return (unsigned)g;
}

bool norm_from(const double *a, const double *b, int n, Norm16 &nm) {
  if (n > 16) return false;
  for (int k = 0; k < 16; ++k) {
    nm.a[k] = (k < n && a) ? (float)a[k] : 0.f;
    nm.b[k] = (k < n && b) ? (float)b[k] : 0.f;
  }
  return true;
}

}  // namespace

// ------------------------------------------------------------------ C-ABI

extern "C" int lbmib_sg_conv3d_fwd(const void *x, const void *w, const float *bias, const void *mask, void *y, int B,
                                   int D, int H, int W, int Cin, int Cout, int relu, void *stream) {
  return conv_fwd(x, w, bias, mask, y, B, D, H, W, Cin, Cout, relu, (hipStream_t)stream);
}

extern "C" int lbmib_sg_conv3d_bwd_data(const void *dy, const void *w, void *wt, const void *mask, void *dx, int B,
                                        int D, int H, int W, int Cin, int Cout, void *stream) {
  if (!dy || !w || !wt || !dx) return LBMIB_ERR_ARG;
  // the data gradient convolves dy (Cout channels) with wt into Cin channels
  if (!shape_ok(B, D, H, W, Cout, Cin) || Cin % 16) return LBMIB_ERR_ARG;
  if (Cout & (Cout - 1)) return LBMIB_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  const lbmib_sg_flip_item item = {w, wt, Cin, Cout};
  const int rc = flip_list(1, &item, s);
  if (rc) return rc;
  return conv_fwd(dy, wt, nullptr, mask, dx, B, D, H, W, Cout, Cin, 0, s);
}

extern "C" int lbmib_sg_flip_many(int n, const lbmib_sg_flip_item *items, void *stream) {
  if (n < 1 || !items) return LBMIB_ERR_ARG;
  for (int k = 0; k < n; ++k) {
    const lbmib_sg_flip_item &q = items[k];
    if (!q.w || !q.wt || !shape_ok(1, 1, 1, 1, q.Cout, q.Cin)) return LBMIB_ERR_ARG;
  }
  return flip_list(n, items, (hipStream_t)stream);
}

extern "C" int lbmib_sg_conv3d_bwd_data_flipped(const void *dy, const void *wt, const void *mask, void *dx, int B,
                                                int D, int H, int W, int Cin, int Cout, void *stream) {
  if (!dy || !wt || !dx || !shape_ok(B, D, H, W, Cout, Cin)) return LBMIB_ERR_ARG;
  return conv_fwd(dy, wt, nullptr, mask, dx, B, D, H, W, Cout, Cin, 0, (hipStream_t)stream);
}

extern "C" int lbmib_sg_conv3d_bwd_weight(const void *x, const void *dy, float *dw, float *db, int B, int D, int H,
                                          int W, int Cin, int Cout, void *stream) {
  if (!x || !dy || !dw || !shape_ok(B, D, H, W, Cin, Cout)) return LBMIB_ERR_ARG;
  void *ws = nullptr;
  const int rc = workspace(&ws);
  if (rc) return rc;
  return wgrad_with(x, dy, dw, db, B, D, H, W, Cin, Cout, ws, LBMIB_SG_WORKSPACE_BYTES, (hipStream_t)stream);
}

extern "C" int lbmib_sg_conv3d_bwd_weight_noalloc(const void *x, const void *dy, float *dw, float *db, int B, int D,
                                                  int H, int W, int Cin, int Cout, void *stream) {
  if (!x || !dy || !dw || !shape_ok(B, D, H, W, Cin, Cout)) return LBMIB_ERR_ARG;
  void *ws = nullptr;
  const int rc = scratch_ptr(&ws);
  if (rc) return rc;
  // the same split plan as lbmib_sg_conv3d_bwd_weight (same cap), so the
  // partials and their fixed-order sums are the same bits; every partial is
  // written before it is read, so nothing needs clearing between calls
  return wgrad_with(x, dy, dw, db, B, D, H, W, Cin, Cout, ws, LBMIB_SG_NOALLOC_SCRATCH_BYTES, (hipStream_t)stream);
}

extern "C" int lbmib_sg_pool2(const void *x, void *y, int B, int D, int H, int W, int C, void *stream) {
  if (!x || !y || B < 1 || D < 1 || H < 1 || W < 1 || C < 8 || C % 8) return LBMIB_ERR_ARG;
  const long n = (long)B * D * H * W * (C / 8);
  pool_launch(n, [&](auto nn) {
    k_pool2<<<grid_for(n), 256, 0, (hipStream_t)stream>>>((const uint16_t *)x, (uint16_t *)y, D, H, W, C, nn);
  });
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_up2_add(const void *c, const void *e, void *s, int B, int D, int H, int W, int C,
                                void *stream) {
  if (!c || !s || B < 1 || D < 2 || H < 2 || W < 2 || (D | H | W) & 1 || C < 8 || C % 8) return LBMIB_ERR_ARG;
  const long n = (long)B * D * H * W * (C / 8);
  pool_launch(n, [&](auto nn) {
    k_up2_add<<<grid_for(n), 256, 0, (hipStream_t)stream>>>((const uint16_t *)c, (const uint16_t *)e, (uint16_t *)s, D, H, W, C, nn);
  });
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_pool2_bwd(const void *a, const void *g, const void *mask, void *out, int B, int D, int H, int W,
                                  int C, void *stream) {
  if (!g || !out || B < 1 || D < 2 || H < 2 || W < 2 || (D | H | W) & 1 || C < 8 || C % 8) return LBMIB_ERR_ARG;
  const long n = (long)B * D * H * W * (C / 8);
  pool_launch(n, [&](auto nn) {
    k_pool2_bwd<<<grid_for(n), 256, 0, (hipStream_t)stream>>>((const uint16_t *)a, (const uint16_t *)g, (const uint16_t *)mask, (uint16_t *)out, D, H, W, C, nn);
  });
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_up2_bwd(const void *ds, const void *mask, void *out, int B, int D, int H, int W, int C,
                                void *stream) {
  if (!ds || !out || B < 1 || D < 1 || H < 1 || W < 1 || C < 8 || C % 8) return LBMIB_ERR_ARG;
  const long n = (long)B * D * H * W * (C / 8);
  pool_launch(n, [&](auto nn) {
    k_up2_bwd<<<grid_for(n), 256, 0, (hipStream_t)stream>>>((const uint16_t *)ds, (const uint16_t *)mask, (uint16_t *)out, D, H, W, C, nn);
  });
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_mse(const void *out, const float *tgt, void *dout, float *loss, long M, int C, int nl,
                            void *stream) {
  if (!out || !tgt || !dout || !loss || M < 1 || C < 1 || nl < 1 || nl > C) return LBMIB_ERR_ARG;
  void *ws = nullptr;
  const int rc = workspace(&ws);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const float denom = (float)((double)M * nl);
  const bool wide = C % 8 == 0 && M * (C / 8) < (1L << 31) && (((uintptr_t)out | (uintptr_t)dout) & 15) == 0;
  const unsigned nb = grid_for(wide ? M * (C / 8) : M * C, 256, 1024);
  if (wide)
    k_mse8<<<nb, 256, 0, s>>>((const uint16_t *)out, tgt, (uint16_t *)dout, (float *)ws, (unsigned)(M * (C / 8)),
                              (unsigned)(C / 8), nl, 2.0f / denom);
  else
    k_mse<<<nb, 256, 0, s>>>((const uint16_t *)out, tgt, (uint16_t *)dout, (float *)ws, M, C, nl, 2.0f / denom);
  HIPCHK(hipGetLastError());
  k_final_sum<<<1, 256, 0, s>>>((const float *)ws, (int)nb, 1.0f / denom, loss);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_adam(float *p, const float *g, float *m, float *v, void *w16, long n, float lr, float beta1,
                             float beta2, float eps, int t, void *stream) {
  if (!p || !g || !m || !v || n < 1 || t < 1) return LBMIB_ERR_ARG;
  const lbmib_sg_adam_item item = {p, g, m, v, w16, n};
  return adam_list(1, &item, lr, beta1, beta2, eps, t, (hipStream_t)stream);
}

extern "C" int lbmib_sg_adam_many(int n, const lbmib_sg_adam_item *items, float lr, float beta1, float beta2,
                                  float eps, int t, void *stream) {
  if (n < 1 || !items || t < 1) return LBMIB_ERR_ARG;
  for (int k = 0; k < n; ++k) {
    const lbmib_sg_adam_item &q = items[k];
    if (!q.p || !q.g || !q.m || !q.v || q.n < 1) return LBMIB_ERR_ARG;
  }
  return adam_list(n, items, lr, beta1, beta2, eps, t, (hipStream_t)stream);
}

extern "C" int lbmib_sg_cast_bf16(const float *src, void *dst, long n, void *stream) {
  if (!src || !dst || n < 1) return LBMIB_ERR_ARG;
  k_cast<<<grid_for(n), 256, 0, (hipStream_t)stream>>>(src, (uint16_t *)dst, n);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_pack(const float *f, int nf, const double *mean, const double *istd, int nconst,
                             const double *cval, void *x, long M, int C, void *stream) {
  if (!x || M < 1 || C % 8 || nf < 0 || nconst < 0 || nf + nconst > C || nf + nconst > 16 || (nf && !f))
    return LBMIB_ERR_ARG;
  Norm16 nm;
  for (int k = 0; k < 16; ++k) nm.a[k] = nm.b[k] = 0.f;
  for (int k = 0; k < nf; ++k) {
    nm.a[k] = mean ? (float)mean[k] : 0.f;
    nm.b[k] = istd ? (float)istd[k] : 1.f;
  }
  for (int k = 0; k < nconst; ++k) nm.a[nf + k] = cval ? (float)cval[k] : 0.f;
  k_pack<<<grid_for(M), 256, 0, (hipStream_t)stream>>>(f, nf, nm, nconst, (uint16_t *)x, M, C);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_target(const float *f0, const float *f1, int nl, const double *mean, const double *istd,
                               float *tgt, long M, void *stream) {
  Norm16 nm;
  if (!f0 || !f1 || !tgt || nl < 1 || M < 1 || !norm_from(mean, istd, nl, nm)) return LBMIB_ERR_ARG;
  k_target<<<grid_for(M), 256, 0, (hipStream_t)stream>>>(f0, f1, nl, nm, tgt, M);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_unpack(const void *out, int C, int nl, const double *mean, const double *std, float *d, long M,
                               void *stream) {
  Norm16 nm;
  if (!out || !d || nl < 1 || nl > C || M < 1 || !norm_from(mean, std, nl, nm)) return LBMIB_ERR_ARG;
  k_unpack<<<grid_for(M), 256, 0, (hipStream_t)stream>>>((const uint16_t *)out, C, nl, nm, d, M);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}

extern "C" int lbmib_sg_sqdiff(const float *a, const float *b, long n, double *out2, void *stream) {
  if (!a || !out2 || n < 1) return LBMIB_ERR_ARG;
  void *ws = nullptr;
  const int rc = sq_partials(&ws);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const unsigned nb = grid_for(n, 256, kSqBlocks);
  k_sqdiff<<<nb, 256, 0, s>>>(a, b, n, (double *)ws);
  HIPCHK(hipGetLastError());
  k_sqdiff_final<<<1, 256, 0, s>>>((const double *)ws, (int)nb, out2);
  HIPCHK(hipGetLastError());
  return LBMIB_OK;
}
