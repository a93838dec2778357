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
//   M = voxels (16 per MFMA row block), N = output channels, K = 27 * CIN,
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
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kConvThreads = 256;  // 4 waves
constexpr int kConvVoxWave = 64;   // voxels per wave (4 MFMA row blocks)

__host__ __device__ constexpr int conv_kp(int cin) { return (27 * cin + 31) / 32 * 32; }

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

// Voxels of a convolution launch: a workgroup owns an 8 x 8 x 4 (x, y, z) tile, its wave w the
// 4 x 4 x 4 brick at (4 (w & 1), 4 (w >> 1), 0) of it; MFMA row block mt of a wave is the brick's
// z-slice mt and row r within it the voxel (r % 4, r / 4).  A wave's 27-tap input footprint is
// 6 x 6 x 6 voxels.  Tiles are ordered z fastest along (x, y) columns, and workgroup b (which
// runs on XCD b % 8) takes tile (b % 8) * (G / 8) + b / 8: each XCD walks a contiguous run of
// columns, so the tiles in flight on one XCD are z-neighbours in adjacent columns and their taps
// re-read inputs from that XCD's L2 instead of HBM (the 48-channel decoder input is 201 MB at
// 128^3, read by 27 taps).  A voxel's K blocks run in the same order under any mapping; the
// hardware's summation inside one MFMA may depend on the row, so results can differ from another
// mapping in the last float32 bits.
constexpr int kConvTileX = 8, kConvTileY = 8, kConvTileZ = 4;

__host__ __device__ inline int conv_tiles(int D, int H, int W) {
  return ((W + kConvTileX - 1) / kConvTileX) * ((H + kConvTileY - 1) / kConvTileY) *
         ((D + kConvTileZ - 1) / kConvTileZ);
}

// Workgroups of a launch: the tile count rounded up to a multiple of HFSI_NXCD.
__host__ __device__ inline int conv_blocks(int D, int H, int W) {
  return (conv_tiles(D, H, W) + HFSI_NXCD - 1) / HFSI_NXCD * HFSI_NXCD;
}

// Origin of this wave's brick (it may lie past the grid's edge); false for the padding
// workgroups past the last tile, for the whole workgroup alike.
__device__ inline bool conv_brick_origin(int D, int H, int W, int& x0, int& y0, int& z0) {
  const int gx = (W + kConvTileX - 1) / kConvTileX, gz = (D + kConvTileZ - 1) / kConvTileZ;
  const int G = (int)gridDim.x, b = blockIdx.x, wave = threadIdx.x >> 6;
  const int t = (b % HFSI_NXCD) * (G / HFSI_NXCD) + b / HFSI_NXCD;
  if (t >= conv_tiles(D, H, W)) return false;
  const int column = t / gz;
  x0 = (column % gx) * kConvTileX + 4 * (wave & 1);
  y0 = (column / gx) * kConvTileY + 4 * (wave >> 1);
  z0 = (t % gz) * kConvTileZ;
  return true;
}

// g where y > 0, else 0: the ReLU's backward through its stored output.
__device__ inline bf16x8 relu_gate(bf16x8 g, bf16x8 y) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (!((float)y[e] > 0.0f)) g[e] = (bf16)0.0f;
  return g;
}

// y[v * ycs + yoff + co] = act(bias[co] + conv(x)[v][co]); bias may be null.  With a gate (the
// activation that the result is the gradient of, laid out like y) the ReLU's backward is applied at
// the store: the gradient would otherwise be read and written once more.
//
// The workgroup stages its tile's input with a one-voxel halo (10 x 10 x 6 voxels) in LDS,
// CC channels at a time (conv_chunk), with 16-byte loads that follow the channels-last
// layout (zero outside the grid: the convolution's padding).  The K dimension is then walked as
// units of 8 channels of one tap, tap-major (unit u = tap * CC / 8 + channel group); a 32-wide
// MFMA K block takes 4 consecutive units, which may straddle two taps, its A operand read from
// LDS and its B operand (the weight row at tap * CIN + channel) from global memory, where the
// weights stay cached.  Every input voxel is read from HBM / L2 about 600 / 256 times per launch
// instead of 27 times.
constexpr int kConvHaloX = kConvTileX + 2, kConvHaloY = kConvTileY + 2, kConvHaloZ = kConvTileZ + 2;
constexpr int kConvHaloVox = kConvHaloX * kConvHaloY * kConvHaloZ;  // 600

// Channels staged per LDS chunk: 16 (a 19.2 KB tile: up to eight workgroups per CU by LDS).
__host__ __device__ constexpr int conv_chunk(int) { return 16; }

template <int CIN, int COUT, bool RELU>
__global__ void __launch_bounds__(kConvThreads) k_conv3_fwd(const bf16* __restrict__ x, const bf16* __restrict__ wt,
                                                             const float* __restrict__ bias,
                                                             const bf16* __restrict__ gate, bf16* __restrict__ y,
                                                             int ycs, int yoff, int D, int H, int W) {
  static_assert(CIN % 8 == 0 && COUT % 16 == 0, "channel counts");
  constexpr int CC = conv_chunk(CIN);
  static_assert(CIN % CC == 0, "channel chunks");
  constexpr int VS = CC;           // LDS voxel stride in bf16 (unpadded: a smaller tile, more workgroups per CU)
  constexpr int UNITS = CC / 8;    // 8-channel units per tap and chunk
  constexpr int KU = 27 * UNITS;   // units per chunk
  constexpr int KP = conv_kp(CIN);
  constexpr int NT = COUT / 16;
  constexpr int MT = kConvVoxWave / 16;  // z-slices of the brick
  constexpr int NIT = (KU + 3) / 4;      // 32-wide K blocks per chunk
  constexpr int PD = NT <= 2 ? 3 : 0;    // weight prefetch distance in K blocks (wide outputs: none)
  __shared__ __attribute__((aligned(16))) bf16 tile[kConvHaloVox * VS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int bx0 = 0, by0 = 0, bz0 = 0;
  if (!conv_brick_origin(D, H, W, bx0, by0, bz0)) return;  // whole workgroup: before any barrier
  const int tx0 = bx0 - 4 * (wave & 1) - 1, ty0 = by0 - 4 * (wave >> 1) - 1, tz0 = bz0 - 1;  // halo origin
  const int r = lane & 15, g = lane >> 4;
  // this lane's A voxel in the halo tile, z-slice 0, tap (0, 0, 0) offset (1, 1, 1)
  const int lx = 1 + 4 * (wave & 1) + (r & 3), ly = 1 + 4 * (wave >> 1) + (r >> 2);
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int cb = 0; cb < CIN; cb += CC) {
    if (cb) __syncthreads();  // the chunk before is consumed
    for (int p = tid; p < kConvHaloVox * UNITS; p += kConvThreads) {
      const int v = p / UNITS, q = p % UNITS;
      const int hx = v % kConvHaloX, hy = (v / kConvHaloX) % kConvHaloY, hz = v / (kConvHaloX * kConvHaloY);
      const int gx = tx0 + hx, gy = ty0 + hy, gz = tz0 + hz;
      bf16x8 val = bf16x8_zero();
      if (gx >= 0 && gx < W && gy >= 0 && gy < H && gz >= 0 && gz < D)
        val = *reinterpret_cast<const bf16x8*>(x + (((long)gz * H + gy) * W + gx) * CIN + cb + 8 * q);
      *reinterpret_cast<bf16x8*>(tile + v * VS + 8 * q) = val;
    }
    __syncthreads();
    // the weight operand of K block it comes from global memory (L2): loaded PD blocks ahead of its
    // use into a ring of registers, so that the MFMAs do not wait on each load in turn
    auto load_b = [&](int it, bf16x8 (&b)[NT]) {
      const int u = 4 * it + g;
      const bool ok = u < KU;
      const int tap = ok ? u / UNITS : 0, cu = ok ? u % UNITS : 0;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        b[nt] = ok ? *reinterpret_cast<const bf16x8*>(wt + (size_t)(nt * 16 + r) * KP + tap * CIN + cb + 8 * cu)
                   : bf16x8_zero();
    };
    bf16x8 bq[PD + 1][NT];
#pragma unroll
    for (int it = 0; it < PD && it < NIT; ++it) load_b(it, bq[it]);
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      if (it + PD < NIT) load_b(it + PD, bq[(it + PD) % (PD + 1)]);
      const int u = 4 * it + g;
      const bool ok = u < KU;
      const int tap = ok ? u / UNITS : 0, cu = ok ? u % UNITS : 0;
      int dz, dy, dx;
      tap_offset(tap, dz, dy, dx);
      const bf16* a0 = tile + ((1 + dz) * kConvHaloY * kConvHaloX + (ly + dy) * kConvHaloX + (lx + dx)) * VS + 8 * cu;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const bf16x8 a = ok ? *reinterpret_cast<const bf16x8*>(a0 + mt * kConvHaloY * kConvHaloX * VS) : bf16x8_zero();
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bq[it % (PD + 1)][nt], acc[mt][nt], 0, 0, 0);
      }
    }
  }
  // Output through LDS, 16 output channels at a time: each wave writes its 64 voxels x 16 channels
  // (bf16, bias and activation applied) into its own 2 KB of the finished tile, then every lane
  // stores two 16-byte runs of 8 channels of one voxel (rather than 16 two-byte stores of one
  // channel each).  Every wave takes part in the barriers; voxels outside the grid are skipped at
  // the store.
  static_assert(kConvHaloVox * VS >= 4 * 64 * 16, "the output staging fits the input tile");
  bf16* stage = tile + wave * 64 * 16;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    __syncthreads();  // the tile (or the previous channel block's staging) is no longer read
    const int co = nt * 16 + r;
    const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float o = acc[mt][nt][i] + bv;
        if (RELU) o = fmaxf(o, 0.0f);
        stage[(mt * 16 + 4 * g + i) * 16 + r] = (bf16)o;  // voxel (i, g) of z-slice mt, channel r
      }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int q = lane;  // voxel of the wave's brick: z-slice q / 16, row q % 16 = 4 g' + i'
      const int ox = bx0 + (q & 3), oy = by0 + ((q >> 2) & 3), oz = bz0 + (q >> 4);
      bf16x8 v8 = *reinterpret_cast<const bf16x8*>(stage + q * 16 + 8 * h);
      if (ox < W && oy < H && oz < D) {
        const long v = ((long)oz * H + oy) * W + ox;
        if (gate) v8 = relu_gate(v8, *reinterpret_cast<const bf16x8*>(gate + v * ycs + yoff + nt * 16 + 8 * h));
        *reinterpret_cast<bf16x8*>(y + v * ycs + yoff + nt * 16 + 8 * h) = v8;
      }
    }
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
constexpr int kWgVox = kConvTileX * kConvTileY * kConvTileZ;  // 256

typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
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

template <int CIN, int COUT>
__global__ void __launch_bounds__(kConvThreads) k_conv3_wgrad(const bf16* __restrict__ x, const bf16* __restrict__ dy,
                                                               float* __restrict__ partial, int D, int H, int W) {
  static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channel counts");
  constexpr int MT = COUT / 16;
  constexpr int XU = (kConvHaloVox * 2 + kConvThreads - 1) / kConvThreads;  // 16-byte units per thread
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
  f32x4 acc[kWgWaveTaps][MT];
#pragma unroll
  for (int j = 0; j < kWgWaveTaps; ++j)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[j][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 rx[XU], ry[YU];
  auto load = [&](int t) {
    const int column = t / gz;
    const int x0 = (column % gx) * kConvTileX, y0 = (column / gx) * kConvTileY, z0 = (t % gz) * kConvTileZ;
#pragma unroll
    for (int q = 0; q < XU; ++q) {
      const int p = tid + q * kConvThreads, v = p >> 1;
      const int xx = x0 - 1 + v % kConvHaloX, yy = y0 - 1 + (v / kConvHaloX) % kConvHaloY,
                zz = z0 - 1 + v / (kConvHaloX * kConvHaloY);
      rx[q] = bf16x8_zero();
      if (v < kConvHaloVox && xx >= 0 && xx < W && yy >= 0 && yy < H && zz >= 0 && zz < D)
        rx[q] = *reinterpret_cast<const bf16x8*>(x + (((long)zz * H + yy) * W + xx) * CIN + cb + 8 * (p & 1));
    }
#pragma unroll
    for (int q = 0; q < YU; ++q) {
      const int p = tid + q * kConvThreads, v = p / (COUT / 8), u = p % (COUT / 8);
      const int xx = x0 + (v & 7), yy = y0 + ((v >> 3) & 7), zz = z0 + (v >> 6);
      ry[q] = bf16x8_zero();
      if (xx < W && yy < H && zz < D)
        ry[q] = *reinterpret_cast<const bf16x8*>(dy + (((long)zz * H + yy) * W + xx) * COUT + 8 * u);
    }
  };
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (bf16)1.0f;
  if (tbeg < tend) load(tbeg);
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
    if (t + 1 < tend) load(t + 1);
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

// out[v][0:CC] = coarse[parent(v)], out[v][CC:CC+CS] = skip[v]   (fine dims D, H, W)
__global__ void k_upcat_fwd(const bf16* __restrict__ coarse, const bf16* __restrict__ skip, bf16* __restrict__ out,
                            int D, int H, int W, int CC, int CS) {
  // one thread per 8-channel unit of an output voxel (CC and CS are multiples of 8): 16-byte copies
  const int UC = CC / 8, U = (CC + CS) / 8, C = CC + CS;
  const long n = (long)D * H * W * U;
  const int hh = H / 2, w = W / 2;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int u = (int)(i % U);
    const long v = i / U;
    bf16x8 val;
    if (u < UC) {
      const int X = (int)(v % W), Y = (int)((v / W) % H), Z = (int)(v / ((long)W * H));
      val = *reinterpret_cast<const bf16x8*>(coarse + ((((long)(Z / 2) * hh) + Y / 2) * w + X / 2) * CC + 8 * u);
    } else {
      val = *reinterpret_cast<const bf16x8*>(skip + v * CS + 8 * (u - UC));
    }
    *reinterpret_cast<bf16x8*>(out + v * C + 8 * u) = val;
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

// bf16 working weights of every conv layer from its float32 master [cout][27 cin]:
// forward [cout][KP(cin)] and flipped-transposed [cin][KP(cout)], zero padded.
constexpr int kWeightsPerBlock = 1024;
__global__ void __launch_bounds__(256) k_conv_weights(ConvLayers tab, const float* __restrict__ params) {
  const ConvLayer& L = tab.l[conv_layer_of(tab, blockIdx.x)];
  const float* wm = params + L.w_off;
  const int cin = L.cin, cout = L.cout;
  const int kpf = conv_kp(cin), kpb = conv_kp(cout);
  const int nf = cout * kpf, nb = L.wb ? cin * kpb : 0;
  const int base = (blockIdx.x - L.first) * kWeightsPerBlock;
  for (int i = base + threadIdx.x; i < min(nf + nb, base + kWeightsPerBlock); i += blockDim.x) {
    if (i < nf) {
      const int co = i / kpf, k = i % kpf;
      L.wf[i] = (bf16)(k < 27 * cin ? wm[(size_t)co * 27 * cin + k] : 0.0f);
    } else {
      const int j = i - nf;
      const int ci = j / kpb, k = j % kpb;
      float val = 0.0f;
      if (k < 27 * cout) {
        const int tapb = k / cout, co = k % cout;
        val = wm[(size_t)co * 27 * cin + (26 - tapb) * cin + ci];
      }
      L.wb[j] = (bf16)val;
    }
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
