// Kernels of the learned initial-guess network (3D U-Net, bf16 on MFMA) for gfx950.
//
// No reference counterpart: the network maps divergence, solid mask and cell
// spacing to a pressure initial guess that the mixed MGPCG then finishes.
//
// Layout: activations are channels-last bf16, voxel index ((z * H + y) * W + x)
// with x fastest, i.e. the fluid's cell index [i][j][k].  Channel counts are
// multiples of 8 (the 5 input channels are padded to 16), so a lane's 8
// consecutive K values of an MFMA operand are 8 channels of one voxel: one
// 16-byte load.
//
// 3x3x3 convolution, zero padding, as an implicit GEMM
//   y[v][co] = bias[co] + sum_{tap, ci} W[co][tap * CIN + ci] * x[v + off(tap)][ci]
// with tap = (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1):
//   M = output channels, N = voxels, K = 27 * CIN,
//   v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][8 (l / 16) .. + 7],
//   B[8 (l / 16) .. + 7][l % 16] and D[4 (l / 16) + i][l % 16], i < 4.
// The data gradient is the same convolution of dy with the flipped, transposed
// weights W'[ci][tap' * COUT + co] = W[co][(26 - tap') * CIN + ci]; the weight
// gradient dW[co][tap][ci] = sum_v dy[v][co] x[v + off(tap)][ci] is an MFMA
// GEMM with K = voxels, both operands transposed on their way out of LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "hfsi_common.hpp"

namespace hfsi {

typedef __bf16 bf16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)), aligned(4))) float f32x4_u;

constexpr int kConvThreads = 256;  // 4 waves

__device__ inline bf16x8 bf16x8_zero() {
  bf16x8 z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = (bf16)0.0f;
  return z;
}

__device__ inline void tap_offset(int tap, int& dz, int& dy, int& dx) {
  dz = tap / 9 - 1;
  dy = (tap / 3) % 3 - 1;
  dx = tap % 3 - 1;
}

// Input of a convolution: CIN channels of x, or, for the two decoder convolutions that follow an
// upsampling and concatenation (conv_cat(CIN) > 0), that many channels of the coarse tensor x at the
// parent voxel and the rest of `skip`: the concatenation (201 MB at 128^3) is never written.
struct ConvIn {
  const bf16* x;
  const bf16* skip;
};
__host__ __device__ constexpr int conv_cat(int cin) { return cin == 48 ? 32 : cin == 96 ? 64 : 0; }

// 8 channels (channel block cb of 16, half `cu`) of voxel (zz, yy, xx); zero outside the grid.
template <int CIN>
__device__ inline bf16x8 conv_input(const ConvIn& in, int cb, int cu, int zz, int yy, int xx, int D, int H, int W) {
  constexpr int CC = conv_cat(CIN);
  if (!(xx >= 0 && xx < W && yy >= 0 && yy < H && zz >= 0 && zz < D)) return bf16x8_zero();
  const bf16* p;
  if (CC == 0) p = in.x + (((long)zz * H + yy) * W + xx) * CIN + cb;
  else if (cb < CC) p = in.x + (((long)(zz >> 1) * (H >> 1) + (yy >> 1)) * (W >> 1) + (xx >> 1)) * CC + cb;
  else p = in.skip + (((long)zz * H + yy) * W + xx) * (CIN - CC) + (cb - CC);
  return *reinterpret_cast<const bf16x8*>(p + 8 * cu);
}

// Bytes that a tile's halo may span for its loads to use 32-bit offsets.
constexpr long kConvSpan = 0xfffff000L;
template <int CIN>
__host__ __device__ inline bool conv_wide(int halo_z, int H, int W) {
  return (long)halo_z * H * W * CIN * 2 >= kConvSpan;
}

// A tile's input with a one-voxel halo (HX x HY x HZ voxels from (x0 - 1, y0 - 1, z0 - 1)), 16 channels
// at a time: 16-byte unit p = voxel p / 2, half p % 2; thread t holds units t, t + 256, ...
// Address arithmetic per load (70 instructions, a branch per boundary, 4 cycles each: 89 against 61 us
// for 16 -> 16 at 128^3) bounds the convolutions, so each thread's offsets from the tile's corner are
// computed once per kernel, the corner is a scalar, and buffer loads return zero for the
// voxels outside the grid (offset ~0), which only tiles at the boundary have to look for.
// WIDE: grids whose halos span more than 32-bit offsets reach, addressed voxel by voxel.
template <int CIN, int HX, int HY, int HZ, bool WIDE>
struct HaloLoader {
  static constexpr int CC = conv_cat(CIN), CS = CIN - CC;
  static constexpr int kUnits = 2 * HX * HY * HZ, XU = (kUnits + kConvThreads - 1) / kConvThreads;
  uint32_t off[XU], coarse[CC > 0 ? XU : 1], at[XU];

  __device__ inline void init(int H, int W) {
#pragma unroll
    for (int q = 0; q < XU; ++q) {
      const int p = threadIdx.x + q * kConvThreads, v = p >> 1;
      const uint32_t hx = v % HX, hy = v / HX % HY, hz = v / (HX * HY);
      const uint32_t half = 16 * (p & 1);
      at[q] = hx | hy << 8 | hz << 16;
      off[q] = p < kUnits ? ((hz * H + hy) * W + hx) * (CS * 2) + half : ~0u;
      // x0 and y0 are even: the parent of corner + h is the corner's parent + (h + 1) / 2; z: see load
      if (CC > 0) coarse[q] = (((hy + 1) >> 1) * (W >> 1) + ((hx + 1) >> 1)) * (CC * 2) + half;
    }
  }

  // channels cb .. cb + 15 into r
  __device__ inline void load(const ConvIn& in, int cb, int x0, int y0, int z0, int D, int H, int W,
                              bf16x8 (&r)[XU]) const {
    if constexpr (WIDE) {
#pragma unroll
      for (int q = 0; q < XU; ++q) {
        r[q] = bf16x8_zero();
        if (off[q] != ~0u)
          r[q] = conv_input<CIN>(in, cb, threadIdx.x & 1, z0 - 1 + (int)(at[q] >> 16), y0 - 1 + (int)(at[q] >> 8 & 255),
                                 x0 - 1 + (int)(at[q] & 255), D, H, W);
      }
    } else {
      const bool up = CC > 0 && cb < CC;
      const bf16* corner =
          up ? in.x + ((((long)(z0 >> 1) - 1) * (H >> 1) + (y0 >> 1) - 1) * (W >> 1) + (x0 >> 1) - 1) * CC + cb
             : (CC > 0 ? in.skip : in.x) + ((((long)z0 - 1) * H + y0 - 1) * W + x0 - 1) * CS + (cb - CC);
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(corner), 0, (int)(uint32_t)kConvSpan, 0x00027000);
      const bool inner = x0 > 0 && y0 > 0 && z0 > 0 && x0 + HX - 2 < W && y0 + HY - 2 < H && z0 + HZ - 2 < D;
      uint32_t o[XU];
#pragma unroll
      for (int q = 0; q < XU; ++q) {
        o[q] = off[q];
        if (up) {
          const uint32_t dz = ((at[q] >> 16) + 1 + (z0 & 1)) >> 1;  // z0 may be odd where tiles are one slice
          const uint32_t parent = coarse[CC > 0 ? q : 0] + dz * ((uint32_t)(H >> 1) * (W >> 1) * (CC * 2));
          o[q] = off[q] == ~0u ? ~0u : parent;
        }
      }
      if (!inner) {
#pragma unroll
        for (int q = 0; q < XU; ++q) {
          const uint32_t xx = x0 - 1 + (at[q] & 255), yy = y0 - 1 + (at[q] >> 8 & 255), zz = z0 - 1 + (at[q] >> 16);
          o[q] = (xx < (uint32_t)W) & (yy < (uint32_t)H) & (zz < (uint32_t)D) ? o[q] : ~0u;
        }
      }
#pragma unroll
      for (int q = 0; q < XU; ++q)
        r[q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)o[q], 0, 0));
    }
  }
};

// The next tile along z, then the next column (tiles of TX x TY x TZ voxels).
template <int TX, int TY, int TZ>
__device__ inline void next_tile(int& x0, int& y0, int& z0, int D, int W) {
  z0 += TZ;
  if (z0 >= D) {
    z0 = 0;
    x0 += TX;
    if (x0 >= W) {
      x0 = 0;
      y0 += TY;
    }
  }
}

// g where y > 0, else 0: the ReLU's backward through its stored output.
__device__ inline bf16x8 relu_gate(bf16x8 g, bf16x8 y) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (!((float)y[e] > 0.0f)) g[e] = (bf16)0.0f;
  return g;
}

// y[v][co] = act(bias[co] + conv(x)[v][co]); bias may be null.  With a gate (the activation that the
// result is the gradient of, laid out like y) the ReLU's backward is applied at the store: the
// gradient would otherwise be read and written once more.
//
// A workgroup (4 waves) owns tiles of 16 x 4 x ZT voxels (x, y, z) and NT blocks of 16 output
// channels; a wave ZT of the tile's 4 ZT rows of 16 voxels.  The tile's input with a one-voxel halo is
// staged 16 channels at a time as two planes of 8 channels (16 bytes per voxel), so that an operand
// read is 256 consecutive bytes per lane group: 8 x 8 x 4 tiles of 32-byte voxels spent 45 % of the LDS
// cycles in bank conflicts.  A = weights (16 channels x 32), B = voxels (32 x 16): lane l ends with 4
// consecutive channels of voxel l % 16, an 8-byte store without staging.  K: 27 taps x 2 planes = 54
// units of 8 channels, tap-major, 4 per MFMA, padded to 56 with zeros; one accumulation chain per
// output in that order for every tile shape (another order, as sharing an operand between the three
// taps along x, changes which sums round to the next bf16, and through the layers and Adam's
// normalised steps a training gradient by up to 3 %).
// The weights come packed in operand order (k_conv_weights) and lie in LDS: all of them, loaded once,
// where they fit (RES), else those of the current 16 channels.  The next input (of the same tile or
// the next) is loaded while one is multiplied.  16 -> 16 at 128^3 80 -> 52 us, 48 -> 16 193 -> 142 us
// without the 2 x 37 us of writing the concatenations, 96 -> 32 at 64^3 90 -> 56 us: the network
// 764 -> 460 us, bit for bit the same.
// Tiles are ordered z fastest along (x, y) columns; a workgroup takes a run of them, the runs of one
// XCD adjacent, so that halos are re-read from that XCD's L2.
constexpr int kConvX = 16, kConvY = 4, kConvUnits = 54, kConvIters = (kConvUnits + 3) / 4;

__host__ __device__ inline int conv_row_tiles(int D, int H, int W, int zt) {
  return ((W + kConvX - 1) / kConvX) * ((H + kConvY - 1) / kConvY) * ((D + zt - 1) / zt);
}

// Packed weights: [cin / 16][14 MFMAs][cout / 16][64 lanes][8], element e of lane l = output channel
// 16 nt + l % 16 of unit u = 4 it + l / 16: tap u / 2, input channel 16 c + 8 (u % 2) + e.
__host__ __device__ constexpr int conv_packed(int cin, int cout) { return cin / 16 * kConvIters * (cout / 16) * 512; }

// All weights in LDS where they leave room for three workgroups per CU (or two with one channel block:
// 48 -> 16 at 128^3 142 against 157 us); reloading them per 16 channels with more workgroups is the
// better one above (32 -> 32 at 64^3 26.0 against 31.7 us, 64 -> 64 at 16^3 8.1 against 11.3).
template <int CIN, int NT>
__host__ __device__ constexpr bool conv_resident() {
  constexpr int kb = CIN / 16 * kConvIters * NT;
  return CIN == 16 || kb <= 28 || (NT == 1 && kb <= 42);
}

template <int CIN, int COUT, int NT, int ZT, bool WIDE>
__global__ void __launch_bounds__(kConvThreads) k_conv3(ConvIn in, const bf16* __restrict__ wt,
                                                         const float* __restrict__ bias, const bf16* __restrict__ gate,
                                                         bf16* __restrict__ y, int D, int H, int W, int relu) {
  static_assert(CIN % 16 == 0 && COUT % (16 * NT) == 0, "channel counts");
  constexpr int HX = kConvX + 2, HY = kConvY + 2, HV = HX * HY * (ZT + 2);
  constexpr int CH = CIN / 16, NC = COUT / 16, FR = kConvIters * NT;  // chunks, channel blocks, operands per chunk
  constexpr bool RES = conv_resident<CIN, NT>();
  using Loader = HaloLoader<CIN, HX, HY, ZT + 2, WIDE>;
  constexpr int XU = Loader::XU, WU = (FR * 64 + kConvThreads - 1) / kConvThreads;
  __shared__ __attribute__((aligned(16))) bf16 tile[2 * HV * 8];
  __shared__ __attribute__((aligned(16))) bf16 wl[(RES ? CH : 1) * FR * 512];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4, nt0 = blockIdx.y * NT;
  const int parts = gridDim.x, b = blockIdx.x;
  const int part = parts % HFSI_NXCD == 0 ? (b % HFSI_NXCD) * (parts / HFSI_NXCD) + b / HFSI_NXCD : b;
  const int gx = (W + kConvX - 1) / kConvX, gz = (D + ZT - 1) / ZT;
  const long tiles = conv_row_tiles(D, H, W, ZT);
  const int tbeg = (int)(tiles * part / parts), tend = (int)(tiles * (part + 1) / parts);
  if (tbeg >= tend) return;  // the whole workgroup, before any barrier
  int x0 = tbeg / gz % gx * kConvX, y0 = tbeg / gz / gx * kConvY, z0 = tbeg % gz * ZT;
  int nx0 = x0, ny0 = y0, nz0 = z0;  // the tile whose input is being loaded
  // 16-byte unit `unit` (operand unit / 64, lane unit % 64) of this workgroup's channel blocks in a
  // chunk's packed weights
  auto packed = [&](int unit) -> uint32_t {
    return (uint32_t)((unit >> 6) / NT * NC + nt0 + (unit >> 6) % NT) * 512 + (unit & 63) * 8;
  };
  constexpr int kChunkWeights = kConvIters * NC * 512;
  uint32_t woff[RES ? 1 : WU];
  if (!RES) {
#pragma unroll
    for (int q = 0; q < WU; ++q) woff[q] = packed(tid + q * kConvThreads);
  }
  Loader loader;
  loader.init(H, W);
  bf16x8 rx[XU], rw[RES ? 1 : WU];
  auto load = [&](int c) {
    loader.load(in, 16 * c, nx0, ny0, nz0, D, H, W, rx);
    if (!RES) {
#pragma unroll
      for (int q = 0; q < WU; ++q)
        if (tid + q * kConvThreads < FR * 64)
          rw[q] = *reinterpret_cast<const bf16x8*>(wt + c * kChunkWeights + woff[q]);
    }
  };
  load(0);
  if (RES)
    for (int c = 0; c < CH; ++c)
      for (int u = tid; u < FR * 64; u += kConvThreads)
        *reinterpret_cast<bf16x8*>(wl + (c * FR * 64 + u) * 8) =
            *reinterpret_cast<const bf16x8*>(wt + c * kChunkWeights + packed(u));
  f32x4 bv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    bv[nt] = bias ? *reinterpret_cast<const f32x4_u*>(bias + (nt0 + nt) * 16 + 4 * g) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // this lane's voxel of the wave's first row at the tap and plane of each MFMA
  const int row0 = wave * ZT;  // row rr of the tile: y = rr % 4, z = rr / 4
  int off[kConvIters];
#pragma unroll
  for (int it = 0; it < kConvIters; ++it) {
    const int u = min(4 * it + g, kConvUnits - 1), tap = u >> 1;
    off[it] = ((u & 1) * HV + (tap / 9 * HY + tap / 3 % 3) * HX + tap % 3 + r) * 8;
  }
  const bool pad = 4 * (kConvIters - 1) + g >= kConvUnits;  // this lane's units of the last MFMA
  const uint32_t lane_out = r * COUT + nt0 * 16 + 4 * g;
  // what `load` fetched, into LDS
  auto put = [&] {
#pragma unroll
    for (int q = 0; q < XU; ++q) {
      const int p = tid + q * kConvThreads;
      if (p < 2 * HV) *reinterpret_cast<bf16x8*>(tile + ((p & 1) * HV + (p >> 1)) * 8) = rx[q];
    }
    if (!RES) {
#pragma unroll
      for (int q = 0; q < WU; ++q)
        if (tid + q * kConvThreads < FR * 64) *reinterpret_cast<bf16x8*>(wl + (tid + q * kConvThreads) * 8) = rw[q];
    }
  };
  put();
  __syncthreads();
  f32x4 acc[ZT][NT];
  for (int t = tbeg; t < tend; ++t) {
#pragma unroll
    for (int m = 0; m < ZT; ++m)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[m][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = 0; c < CH; ++c) {
      const bool more = c + 1 < CH || t + 1 < tend;
      if (c + 1 < CH) {
        load(c + 1);
      } else if (more) {
        next_tile<kConvX, kConvY, ZT>(nx0, ny0, nz0, D, W);
        load(0);
      }
      const bf16* w0 = wl + (RES ? c * FR * 512 : 0) + lane * 8;
#pragma unroll
      for (int it = 0; it < kConvIters; ++it) {
        bf16x8 a[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) a[nt] = *reinterpret_cast<const bf16x8*>(w0 + (it * NT + nt) * 512);
        const bf16* b0 = tile + off[it] + ((row0 >> 2) * HY + (row0 & 3)) * HX * 8;
#pragma unroll
        for (int m = 0; m < ZT; ++m) {  // rows row0 .. row0 + ZT - 1 lie in one z-slice
          bf16x8 v = *reinterpret_cast<const bf16x8*>(b0 + m * HX * 8);
          if (it == kConvIters - 1 && pad) v = bf16x8_zero();
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            acc[m][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[nt], v, acc[m][nt], 0, 0, 0);
        }
      }
      if (c + 1 < CH) {
        __syncthreads();  // consumed
        put();
        __syncthreads();
      }
    }
    __syncthreads();  // the tile is consumed
    // before this tile's stores are issued: its loads are older, and waiting for them then does not wait
    // for the stores
    if (t + 1 < tend) put();
    const bool in_x = x0 + r < W;
#pragma unroll
    for (int m = 0; m < ZT; ++m) {
      const int rr = row0 + m, oy = y0 + (rr & 3), oz = z0 + (rr >> 2);
      if (oy >= H || oz >= D) continue;  // the whole wave
      const long row = (((long)oz * H + oy) * W + x0) * COUT;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float s = acc[m][nt][e] + bv[nt][e];
          if (relu) s = fmaxf(s, 0.0f);
          o[e] = (bf16)s;
        }
        if (gate && in_x) {
          const bf16x4 act = *reinterpret_cast<const bf16x4*>(gate + row + lane_out + nt * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (!((float)act[e] > 0.0f)) o[e] = (bf16)0.0f;
        }
        if (in_x) *reinterpret_cast<bf16x4*>(y + row + lane_out + nt * 16) = o;
      }
    }
    next_tile<kConvX, kConvY, ZT>(x0, y0, z0, D, W);
    __syncthreads();
  }
}

// Weight and bias gradient: dW[co][tap][ci] = sum_v dy[v][co] x[v + off(tap)][ci] for 16 input
// channels (blockIdx.y), with the bias as a 28th tap whose x is 1 everywhere.
//
// An MFMA GEMM with K = voxels.  A workgroup walks a run of 8 x 8 x 4 tiles; a tile's dy and its x
// with a one-voxel halo are staged channels-last, as they lie in memory, and ds_read_tr16_b64 hands
// each lane the four voxels of its channel that an operand needs (lane i of a 16-lane group gives the
// address of voxel i / 4, channels 4 (i % 4) .. + 3 and receives channel i of the four voxels), so
// nothing is transposed by hand and every tap of a tile is one LDS offset.  A K block is 32 voxels
// (rows y of 8 voxels, one per lane group); a wave takes 7 of the 28 taps, its accumulators staying in
// registers over all its tiles, and the next tile's loads are in flight while one is summed.
// Reading x and dy once per tap from L2 and transposing them through LDS with 2-byte writes, the
// 16 x 16 gradient took 69 us at 64^3 and the 48 x 16 one 227 us, and a bias pass 67 us more; now
// 17.8 and 47.9 us with the bias.
constexpr int kWgTaps = 28, kWgWaveTaps = 7;
constexpr int kConvTileX = 8, kConvTileY = 8, kConvTileZ = 4;
constexpr int kWgVox = kConvTileX * kConvTileY * kConvTileZ;  // 256
constexpr int kConvHaloX = kConvTileX + 2, kConvHaloY = kConvTileY + 2, kConvHaloZ = kConvTileZ + 2;
constexpr int kConvHaloVox = kConvHaloX * kConvHaloY * kConvHaloZ;  // 600

__host__ __device__ inline int conv_tiles(int D, int H, int W) {
  return ((W + kConvTileX - 1) / kConvTileX) * ((H + kConvTileY - 1) / kConvTileY) *
         ((D + kConvTileZ - 1) / kConvTileZ);
}

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// Channel (lane % 16) of the 8 voxels p, p + 16, .. p + 112 bf16 (x neighbours of one row).
__device__ inline bf16x8 read_tr8(const bf16* p) {
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p + 64));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Workgroups per 16 input channels: enough for one per CU over all channel blocks (two at sizes where
// the partial sums are small beside the tiles), a multiple of HFSI_NXCD where there are that many tiles.
__host__ __device__ inline int wgrad_parts(int tiles, int cin) {
  const int want = (tiles >= 4096 ? 512 : 256) / (cin / 16);
  if (tiles < HFSI_NXCD) return tiles;
  const int n = tiles < want ? tiles : want;
  return n / HFSI_NXCD * HFSI_NXCD;
}

template <int CIN, int COUT, bool WIDE>
__global__ void __launch_bounds__(kConvThreads) k_conv3_wgrad(ConvIn in, const bf16* __restrict__ dy,
                                                               float* __restrict__ partial, int D, int H, int W) {
  static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channel counts");
  constexpr int MT = COUT / 16;
  using Loader = HaloLoader<CIN, kConvHaloX, kConvHaloY, kConvHaloZ, WIDE>;
  constexpr int XU = Loader::XU;  // 16-byte units per thread
  constexpr int YU = kWgVox * (COUT / 8) / kConvThreads;
  __shared__ __attribute__((aligned(16))) bf16 sx[kConvHaloVox * 16];
  __shared__ __attribute__((aligned(16))) bf16 sdy[MT * kWgVox * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, i = lane & 15;
  const int cb = 16 * blockIdx.y, parts = gridDim.x, b = blockIdx.x;
  const int part = parts % HFSI_NXCD == 0 ? (b % HFSI_NXCD) * (parts / HFSI_NXCD) + b / HFSI_NXCD : b;
  const int gx = (W + kConvTileX - 1) / kConvTileX, gz = (D + kConvTileZ - 1) / kConvTileZ;
  const long tiles = conv_tiles(D, H, W);
  const int tbeg = (int)(tiles * part / parts), tend = (int)(tiles * (part + 1) / parts);
  int x0 = tbeg / gz % gx * kConvTileX, y0 = tbeg / gz / gx * kConvTileY, z0 = tbeg % gz * kConvTileZ;
  Loader loader;
  loader.init(H, W);
  uint32_t yoff[YU];  // this thread's dy units, from the tile's corner
#pragma unroll
  for (int q = 0; q < YU; ++q) {
    const uint32_t p = tid + q * kConvThreads, v = p / (COUT / 8), u = p % (COUT / 8);
    yoff[q] = (((v >> 6) * H + (v >> 3 & 7)) * W + (v & 7)) * (COUT * 2) + 16 * u;
  }
  f32x4 acc[kWgWaveTaps][MT];
#pragma unroll
  for (int j = 0; j < kWgWaveTaps; ++j)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[j][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 rx[XU], ry[YU];
  auto load = [&] {
    loader.load(in, cb, x0, y0, z0, D, H, W, rx);
    const bf16* corner = dy + (((long)z0 * H + y0) * W + x0) * COUT;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(corner), 0, (int)(uint32_t)kConvSpan, 0x00027000);
    const bool inner = x0 + kConvTileX <= W && y0 + kConvTileY <= H && z0 + kConvTileZ <= D;
#pragma unroll
    for (int q = 0; q < YU; ++q) {
      const int v = (tid + q * kConvThreads) / (COUT / 8);
      const bool valid = inner || (x0 + (v & 7) < W && y0 + (v >> 3 & 7) < H && z0 + (v >> 6) < D);
      if constexpr (!WIDE) {
        ry[q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(valid ? yoff[q] : ~0u), 0, 0));
      } else {
        ry[q] = bf16x8_zero();
        if (valid)
          ry[q] = *reinterpret_cast<const bf16x8*>(corner + (((long)(v >> 6) * H + (v >> 3 & 7)) * W + (v & 7)) * COUT +
                                                   8 * ((tid + q * kConvThreads) % (COUT / 8)));
      }
    }
    next_tile<kConvTileX, kConvTileY, kConvTileZ>(x0, y0, z0, D, W);
  };
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (bf16)1.0f;
  if (tbeg < tend) load();
  for (int t = tbeg; t < tend; ++t) {
    __syncthreads();  // the tile before is consumed
#pragma unroll
    for (int q = 0; q < XU; ++q) {
      const int p = tid + q * kConvThreads;
      if (p < 2 * kConvHaloVox) *reinterpret_cast<bf16x8*>(sx + 8 * p) = rx[q];
    }
#pragma unroll
    for (int q = 0; q < YU; ++q) {
      const int p = tid + q * kConvThreads, v = p / (COUT / 8), u = p % (COUT / 8);
      *reinterpret_cast<bf16x8*>(sdy + ((u >> 1) * kWgVox + v) * 16 + 8 * (u & 1)) = ry[q];
    }
    __syncthreads();
    if (t + 1 < tend) load();
#pragma unroll 2
    for (int kb = 0; kb < kWgVox / 32; ++kb) {
      const int z = kb >> 1, y = 4 * (kb & 1) + g, xv = i >> 2, c = 4 * (i & 3);
      const bf16* a0 = sdy + ((z * kConvTileY + y) * kConvTileX + xv) * 16 + c;
      const bf16* b0 = sx + (((z + 1) * kConvHaloY + y + 1) * kConvHaloX + xv + 1) * 16 + c;
      bf16x8 a[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[mt] = read_tr8(a0 + mt * kWgVox * 16);
#pragma unroll
      for (int j = 0; j < kWgWaveTaps; ++j) {
        const int tap = wave * kWgWaveTaps + j;
        int dz, dyo, dx;
        tap_offset(tap, dz, dyo, dx);
        const bf16x8 bt = tap < 27 ? read_tr8(b0 + ((dz * kConvHaloY + dyo) * kConvHaloX + dx) * 16) : ones;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], bt, acc[j][mt], 0, 0, 0);
      }
    }
  }
  float* out = partial + ((size_t)blockIdx.y * parts + part) * kWgTaps * COUT * 16;
#pragma unroll
  for (int j = 0; j < kWgWaveTaps; ++j)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        out[((wave * kWgWaveTaps + j) * COUT + mt * 16 + 4 * g + e) * 16 + i] = acc[j][mt][e];
}

// One convolution layer of the passes over all layers (k_grad_reduce, k_conv_weights).
struct ConvLayer {
  int cin, cout, parts;
  int first;              // first workgroup of the layer
  const float* partial;   // [cin / 16][parts][28][cout][16]
  size_t w_off, b_off;    // into the parameter vector
  bf16 *wf, *wb;          // working weights
};
constexpr int kConvLayers = 10;
struct ConvLayers {
  ConvLayer l[kConvLayers];
};

__device__ inline int conv_layer_of(const ConvLayers& t, int block) {
  int l = 0;
  while (l + 1 < kConvLayers && block >= t.l[l + 1].first) ++l;
  return l;
}

// grads += the partial sums of every layer, added in order in float64: 64 values per workgroup, four
// threads each taking a quarter of the parts.
constexpr int kGradReduceValues = 64;
__global__ void __launch_bounds__(256) k_grad_reduce(ConvLayers tab, float* __restrict__ grads) {
  __shared__ double part[4][kGradReduceValues];
  const ConvLayer& L = tab.l[conv_layer_of(tab, blockIdx.x)];
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int idx = (blockIdx.x - L.first) * kGradReduceValues + lane;  // a multiple of 64 values per layer
  const int block = kWgTaps * L.cout * 16, cblk = idx / block, rem = idx % block;
  const int tap = rem / (L.cout * 16), co = rem / 16 % L.cout, ci = rem % 16;
  const float* src = L.partial + (size_t)cblk * L.parts * block + rem;
  const int n0 = L.parts * q / 4, n1 = L.parts * (q + 1) / 4;
  double s = 0.0;
#pragma unroll 8
  for (int p = n0; p < n1; ++p) s += (double)src[(size_t)p * block];
  part[q][lane] = s;
  __syncthreads();
  if (q != 0) return;
  const float sum = (float)(((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane]);
  if (tap < 27) grads[L.w_off + ((size_t)co * 27 + tap) * L.cin + cblk * 16 + ci] += sum;
  else if (cblk == 0 && ci == 0) grads[L.b_off + co] += sum;
}

// 2x2x2 average pooling (even fine dims): y[D/2][H/2][W/2][C], 8 channels per thread.
__global__ void k_pool2_fwd(const bf16* __restrict__ x, bf16* __restrict__ y, int D, int H, int W, int C) {
  const int d = D / 2, hh = H / 2, w = W / 2, U = C / 8;
  const long n = (long)d * hh * w * U;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int u = (int)(i % U);
    const long v = i / U;
    const int X = (int)(v % w), Y = (int)((v / w) % hh), Z = (int)(v / ((long)w * hh));
    bf16x8 in[8];
#pragma unroll
    for (int o = 0; o < 8; ++o)
      in[o] = *reinterpret_cast<const bf16x8*>(
          x + ((((long)(2 * Z + (o >> 2)) * H) + (2 * Y + ((o >> 1) & 1))) * W + (2 * X + (o & 1))) * C + 8 * u);
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float s = 0.0f;
#pragma unroll
      for (int o = 0; o < 8; ++o) s += (float)in[o][e];
      out[e] = (bf16)(0.125f * s);
    }
    *reinterpret_cast<bf16x8*>(y + v * C + 8 * u) = out;
  }
}

// Gradient of an encoder level's output y[v][0:C]: its skip part dout[v][CC + c] (dout has CC + C
// channels) plus the pooled path dy[parent][c] / 8, through the ReLU of y.
__global__ void k_skip_pool_bwd(const bf16* __restrict__ dout, const bf16* __restrict__ dy, const bf16* __restrict__ y,
                                bf16* __restrict__ g, int D, int H, int W, int CC, int C) {
  const int U = C / 8, hh = H / 2, w = W / 2;
  const long n = (long)D * H * W * U;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int u = (int)(i % U);
    const long v = i / U;
    const int X = (int)(v % W), Y = (int)((v / W) % H), Z = (int)(v / ((long)W * H));
    const bf16x8 skip = *reinterpret_cast<const bf16x8*>(dout + v * (CC + C) + CC + 8 * u);
    const bf16x8 up = *reinterpret_cast<const bf16x8*>(dy + ((((long)(Z / 2) * hh) + Y / 2) * w + X / 2) * C + 8 * u);
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = (bf16)((float)skip[e] + 0.125f * (float)up[e]);
    *reinterpret_cast<bf16x8*>(g + v * C + 8 * u) =
        relu_gate(out, *reinterpret_cast<const bf16x8*>(y + v * C + 8 * u));
  }
}

// dcoarse[p][c] = sum of the 8 children's dout[v][c] (c < CC) through the ReLU of the coarse output y.
__global__ void k_upcat_bwd_coarse(const bf16* __restrict__ dout, const bf16* __restrict__ y,
                                   bf16* __restrict__ dcoarse, int D, int H, int W, int CC, int CS) {
  const int C = CC + CS, U = CC / 8;
  const int d = D / 2, hh = H / 2, w = W / 2;
  const long n = (long)d * hh * w * U;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int u = (int)(i % U);
    const long p = i / U;
    const int X = (int)(p % w), Y = (int)((p / w) % hh), Z = (int)(p / ((long)w * hh));
    bf16x8 in[8];
#pragma unroll
    for (int o = 0; o < 8; ++o)
      in[o] = *reinterpret_cast<const bf16x8*>(
          dout + ((((long)(2 * Z + (o >> 2)) * H) + (2 * Y + ((o >> 1) & 1))) * W + (2 * X + (o & 1))) * C + 8 * u);
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float s = 0.0f;
#pragma unroll
      for (int o = 0; o < 8; ++o) s += (float)in[o][e];
      out[e] = (bf16)s;
    }
    *reinterpret_cast<bf16x8*>(dcoarse + p * CC + 8 * u) =
        relu_gate(out, *reinterpret_cast<const bf16x8*>(y + p * CC + 8 * u));
  }
}

// Output layer: y[v] = b + sum_c w[c] u[v][c]  (CU channels, float output)
template <int CU>
__global__ void k_out_fwd(const bf16* __restrict__ u, const float* __restrict__ w, const float* __restrict__ b,
                          float* __restrict__ y, long nvox) {
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long)gridDim.x * blockDim.x) {
    float s = b[0];
#pragma unroll
    for (int c = 0; c < CU; ++c) s += w[c] * (float)u[v * CU + c];
    y[v] = s;
  }
}

// Output layer backward: du[v][c] = dy[v] w[c] through the ReLU of u; partials of (sum_v dy u[v][c], sum_v dy).
template <int CU>
__global__ void __launch_bounds__(256) k_out_bwd(const bf16* __restrict__ u, const float* __restrict__ w,
                                                 const float* __restrict__ dyv, bf16* __restrict__ du, long nvox,
                                                 double* __restrict__ partials) {
  __shared__ double lds[(CU + 1) * 4];
  double acc[CU + 1];
#pragma unroll
  for (int c = 0; c <= CU; ++c) acc[c] = 0.0;
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long)gridDim.x * blockDim.x) {
    const float g = dyv[v];
#pragma unroll
    for (int c = 0; c < CU; ++c) {
      const float uc = (float)u[v * CU + c];
      acc[c] += (double)(g * uc);
      du[v * CU + c] = (bf16)(uc > 0.0f ? g * w[c] : 0.0f);
    }
    acc[CU] += (double)g;
  }
  block_partials<CU + 1>(acc, partials, lds);
}

// Relative squared error over the masked voxels: partials of
// (sum m (y - t)^2, sum m t^2); the gradient is formed by k_loss_grad.
__global__ void __launch_bounds__(256) k_loss_sums(const float* __restrict__ y, const float* __restrict__ t,
                                                   const uint8_t* __restrict__ mask, long nvox,
                                                   double* __restrict__ partials) {
  __shared__ double lds[2 * 4];
  double acc[2] = {0.0, 0.0};
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long)gridDim.x * blockDim.x) {
    if (mask && !mask[v]) continue;
    const double e = (double)y[v] - (double)t[v];
    acc[0] += e * e;
    acc[1] += (double)t[v] * (double)t[v];
  }
  block_partials<2>(acc, partials, lds);
}

// dy = 2 (y - t) / sum m t^2 on masked voxels, 0 elsewhere (sums in totals[0..1])
__global__ void k_loss_grad(const float* __restrict__ y, const float* __restrict__ t, const uint8_t* __restrict__ mask,
                            long nvox, const double* __restrict__ totals, float* __restrict__ dy) {
  const double den = totals[1] > 0.0 ? totals[1] : 1.0;
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long)gridDim.x * blockDim.x)
    dy[v] = (mask && !mask[v]) ? 0.0f : (float)(2.0 * ((double)y[v] - (double)t[v]) / den);
}

// Adam on the float32 master parameters.
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       long n, float lr, float b1, float b2, float eps, float c1, float c2, float weight_decay) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float gi = g[i] + weight_decay * p[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// bf16 working weights of every conv layer from its float32 master [cout][27 cin], packed as k_conv3
// reads them: forward (wf), and for the data gradient with taps flipped and channels swapped (wb).
constexpr int kWeightsPerBlock = 1024;
__global__ void __launch_bounds__(256) k_conv_weights(ConvLayers tab, const float* __restrict__ params) {
  const ConvLayer& L = tab.l[conv_layer_of(tab, blockIdx.x)];
  const float* wm = params + L.w_off;
  const int nf = conv_packed(L.cin, L.cout), nb = L.wb ? conv_packed(L.cout, L.cin) : 0;
  const int base = (blockIdx.x - L.first) * kWeightsPerBlock;
  for (int i = base + threadIdx.x; i < min(nf + nb, base + kWeightsPerBlock); i += blockDim.x) {
    const bool back = i >= nf;
    const int j = back ? i - nf : i;
    const int nc = (back ? L.cin : L.cout) / 16;  // output channel blocks
    const int e = j & 7, l = j >> 3 & 63, f = j >> 9;
    const int nt = f % nc, it = f / nc % kConvIters, c = f / nc / kConvIters;
    const int u = 4 * it + (l >> 4);
    const int co = 16 * nt + (l & 15), ci = 16 * c + 8 * (u & 1) + e, tap = u >> 1;
    float val = 0.0f;
    if (u < kConvUnits)
      val = back ? wm[(size_t)ci * 27 * L.cin + (26 - tap) * L.cin + co] : wm[(size_t)co * 27 * L.cin + tap * L.cin + ci];
    (back ? L.wb : L.wf)[j] = (bf16)val;
  }
}

// Network input: the 5 float channels of each voxel -> 16 bf16 channels (zero padded).
__global__ void k_unet_input(const float* __restrict__ in5, bf16* __restrict__ x, long nvox) {
  // one thread per voxel: its 5 features, zero-padded to 16 channels, as two 16-byte stores
  for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long)gridDim.x * blockDim.x) {
    bf16x8 lo = bf16x8_zero();
#pragma unroll
    for (int c = 0; c < 5; ++c) lo[c] = (bf16)in5[v * 5 + c];
    *reinterpret_cast<bf16x8*>(x + v * 16) = lo;
    *reinterpret_cast<bf16x8*>(x + v * 16 + 8) = bf16x8_zero();
  }
}

}  // namespace hfsi
