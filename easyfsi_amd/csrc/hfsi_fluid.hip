// libhfsi: FV pressure projection on the graded MAC grid for gfx950.
//
// Host orchestration of the reference's flexible PCG with the Jacobi-smoothed
// V-cycle preconditioner (simulation_core/fluid.py:6535-6811, 6085-6262) on
// hand-written HIP kernels.  Scalars of the CG recurrence live on the device;
// the host synchronises only at residual checks (every `check_interval`
// iterations, 16 in the reference) and at the start of a solve.
//
// Precision modes
//   REF64: float64 CG vectors and level-0 V-cycle, float32 coarse-level storage,
//          float64 arithmetic everywhere (the reference's dtypes).
//   FP32 : float32 CG vectors and V-cycle with float32 arithmetic, float64
//          solution x, right-hand side b and dots; every residual check
//          replaces r by the float64 true residual b - A x.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <type_traits>
#include <string>
#include <vector>

#include "../../include/hfsi.h"
#include "fluid_march.hpp"
#include "fluid_mixed.hpp"
#include "fluid_predict.hpp"
#include "fluid_interface.hpp"

namespace hfsi {

static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }

constexpr int kMaxLevels = 16;
constexpr uint32_t kMaxGrid = 2048;      // workgroups of full-grid launches (8 per CU)
// Levels at most this big restrict in tiles: float64 64^3 11.4 -> 8.8 us, 32^3 12.6 -> 7.4 us against the
// marching form, whose columns leave most of the chip idle there; at 128^3 13.9 (marching) against 22.0 us.
constexpr uint32_t kRestrictTileMax = 1u << 19;
constexpr uint32_t kTailCells = 4096;    // levels at most this big run in the single-workgroup tail
// the same for the mixed V-cycle's LDS-resident tail: one workgroup on one CU; a 23^3 level there
// (12 167 cells, 110 KB of LDS) took longer than its own multi-workgroup passes (103 us against
// 49 + 46 us per V-cycle at 256^3)
constexpr uint32_t kMixTailCells = 4096;
constexpr uint32_t kMixTailStaticLds = 8192;  // k_mix_tail's static LDS (dense right-hand side) and slack
constexpr int kTailThreads = 1024;
constexpr uint32_t kTailLdsMax = 152 * 1024;  // dynamic LDS budget of the tail workgroup (160 KB per CU)

// ---------------------------------------------------------------------------
// Device-resident CG scalars
// ---------------------------------------------------------------------------

struct Scalars {
  double rz, dAd, alpha, beta, rr, mz, mx, mr, mb, bnorm2, free_vol, code_dAd;
  int32_t code, pad;
  // mixed V-cycle scaling: level-0 input r * vin (vin = 1 / RMS_V(r)), output z = e * vout (vout = RMS / kappa)
  double vin, vout;
  // learned initial guess: divergence RMS of the network grid, mean of the interpolated guess, the
  // energy-optimal factor's numerator and the factor
  double g_rms, g_mean, g_mean_b, g_num, g_gamma;
};

struct FinNone {
  __device__ void operator()(const double*) const {}
};
// ---- learned initial guess: features and the scaled guess on the device ----------------------
// The network grid is the solve grid coarsened CF:1 per axis (CF = 2, or 1 for grids that do not
// coarsen).  Features of a network cell: the divergence of its free children volume-averaged over
// their volume, the solid volume fraction, log2(width / min width) per axis.
struct FinGuessRms {
  Scalars* s;
  __device__ void operator()(const double* t) const {
    const double r = t[1] > 0.0 ? sqrt(t[0] / t[1]) : 0.0;
    s->g_rms = r > 0.0 ? r : 1.0;
  }
};
struct FinGuessMean {
  Scalars* s;
  __device__ void operator()(const double* t) const {
    s->g_mean = t[1] > 0.0 ? t[0] / t[1] : 0.0;
    s->g_mean_b = t[1] > 0.0 ? t[2] / t[1] : 0.0;
  }
};
struct FinGuessNum {
  Scalars* s;
  __device__ void operator()(const double* t) const { s->g_num = t[0]; }
};
struct FinGuessGamma {
  Scalars* s;
  __device__ void operator()(const double* t) const { s->g_gamma = t[0] > 0.0 ? s->g_num / t[0] : 0.0; }
};

template <int CF>
__global__ void __launch_bounds__(kBlock) k_guess_features(OpGeo<double> g, const float* div, uint32_t cny,
                                                           uint32_t cnz, uint32_t nc, double inv_hmin,
                                                           double* dtmp, float* feat, double* partials) {
  constexpr int NS = 2;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS] = {0.0, 0.0};
  HFSI_CELL_LOOP(nc) {
    uint32_t ci, cj, ck;
    decompose(c, cny, cnz, ci, cj, ck);
    double num = 0.0, vol = 0.0, fvol = 0.0;
#pragma unroll
    for (int oi = 0; oi < CF; ++oi)
#pragma unroll
      for (int oj = 0; oj < CF; ++oj)
#pragma unroll
        for (int ok = 0; ok < CF; ++ok) {
          const uint32_t i = CF * ci + oi, j = CF * cj + oj, k = CF * ck + ok;
          const uint32_t f = i * g.sx + j * g.sy + k;
          const double V = volume64(g, i, j, k);
          const bool fr = !(g.flags[f] & kNotFree);
          vol += V;
          if (fr) {
            fvol += V;
            num += (double)div[f] * V;
          }
        }
    const double d = fvol > 0.0 ? num / fvol : 0.0;
    dtmp[c] = d;
    acc[0] += fvol * d * d;
    acc[1] += fvol;
    double w[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int o = 0; o < CF; ++o) {
      w[0] += g.wd[0][CF * ci + o];
      w[1] += g.wd[1][CF * cj + o];
      w[2] += g.wd[2][CF * ck + o];
    }
    float* fc = feat + 5 * (size_t)c;
    fc[1] = (float)(1.0 - fvol / vol);
#pragma unroll
    for (int a = 0; a < 3; ++a) fc[2 + a] = (float)log2(w[a] * inv_hmin);
  }
  block_partials<NS>(acc, partials, lds);
}

__global__ void __launch_bounds__(kBlock) k_guess_normalise(uint32_t nc, const double* dtmp, float* feat,
                                                            const Scalars* s) {
  const double rms = s->g_rms;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < nc; c += gridDim.x * blockDim.x)
    feat[5 * (size_t)c] = (float)(dtmp[c] / rms);
}

// Network output (network grid) interpolated to the solve grid, trilinear with half-cell centres
// (a fine cell of index o along an axis sits at o / CF - 0.25 network cells for CF = 2, clamped at
// the first cell), times coef * rms; zero on cells that are not free.  Sums V p and V over free cells.
__device__ inline void lin2(uint32_t o, uint32_t n, uint32_t& a, uint32_t& b, double& wa) {
  const uint32_t m = o >> 1;
  if (o & 1u) {  // (m + 0.25): 0.75 m + 0.25 (m + 1)
    a = m;
    b = m + 1 < n ? m + 1 : n - 1;
    wa = 0.75;
  } else if (m == 0) {
    a = b = 0;
    wa = 1.0;
  } else {  // (m - 0.25): 0.25 (m - 1) + 0.75 m
    a = m - 1;
    b = m;
    wa = 0.25;
  }
}

template <int CF>
__global__ void __launch_bounds__(kBlock) k_guess_prolong(OpGeo<double> g, const float* out, uint32_t cny,
                                                          uint32_t cnz, double coef, const Scalars* s, double* p,
                                                          const float* div, const float* src, double rho_over_dt,
                                                          double* partials) {
  constexpr int NS = 3;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS] = {0.0, 0.0, 0.0};
  const double scale = coef * s->g_rms;
  HFSI_CELL_LOOP(g.n) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    double v = 0.0;
    if (!(g.flags[c] & kNotFree)) {
      if (CF == 1) {
        v = (double)out[c] * scale;
      } else {
        uint32_t ia, ib, ja, jb, ka, kb;
        double wi, wj, wk;
        lin2(i, g.nx / 2, ia, ib, wi);
        lin2(j, cny, ja, jb, wj);
        lin2(k, cnz, ka, kb, wk);
        auto at = [&](uint32_t a, uint32_t b, uint32_t d) { return (double)out[(a * cny + b) * cnz + d]; };
        const double x00 = wk * at(ia, ja, ka) + (1.0 - wk) * at(ia, ja, kb);
        const double x01 = wk * at(ia, jb, ka) + (1.0 - wk) * at(ia, jb, kb);
        const double x10 = wk * at(ib, ja, ka) + (1.0 - wk) * at(ib, ja, kb);
        const double x11 = wk * at(ib, jb, ka) + (1.0 - wk) * at(ib, jb, kb);
        const double x0 = wj * x00 + (1.0 - wj) * x01, x1 = wj * x10 + (1.0 - wj) * x11;
        v = (wi * x0 + (1.0 - wi) * x1) * scale;
      }
      const double V = volume64(g, i, j, k);
      acc[0] += V * v;
      acc[1] += V;
      acc[2] += V * (-rho_over_dt * ((double)div[c] - (src ? (double)src[c] : 0.0)));
    }
    p[c] = v;
  }
  block_partials<NS>(acc, partials, lds);
}

// p -= mean on free cells (the closed domain's null space), and the numerator sum V p b with
// b = -(rho/dt) (div - source), its mean removed likewise.
__global__ void __launch_bounds__(kBlock) k_guess_center(OpGeo<double> g, double* p, const float* div,
                                                         const float* src, double rho_over_dt, const Scalars* s,
                                                         int remove_mean, double* partials) {
  constexpr int NS = 1;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS] = {0.0};
  const double mean = remove_mean ? s->g_mean : 0.0, mean_b = remove_mean ? s->g_mean_b : 0.0;
  HFSI_CELL_LOOP(g.n) {
    if (g.flags[c] & kNotFree) continue;
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    const double v = p[c] - mean;
    p[c] = v;
    const double b = -rho_over_dt * ((double)div[c] - (src ? (double)src[c] : 0.0)) - mean_b;
    acc[0] += volume64(g, i, j, k) * v * b;
  }
  block_partials<NS>(acc, partials, lds);
}

// The energy denominator sum V p (A p) over free cells (operator without couplings).
__global__ void __launch_bounds__(kBlock) k_guess_energy(OpGeo<double> g, const double* p, double* partials) {
  constexpr int NS = 1;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS] = {0.0};
  const Ld<double, double> P{p};
  HFSI_CELL_LOOP(g.n) {
    if (g.flags[c] & kNotFree) continue;
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    acc[0] += volume64(g, i, j, k) * p[c] * apply_cell(g, c, i, j, k, P);
  }
  block_partials<NS>(acc, partials, lds);
}

__global__ void __launch_bounds__(kBlock) k_guess_scale(uint32_t n, double* p, const Scalars* s) {
  const double gamma = s->g_gamma;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) p[c] *= gamma;
}

// _mark_sphere_kernel (fluid.py:2828-2844): obstacle = 1 where the cell centre lies within the radius
// (float32, rx*rx + ry*ry + rz*rz <= r*r in that order, no contraction), 0 elsewhere.
__global__ void __launch_bounds__(kBlock) k_mark_sphere(uint32_t nx, uint32_t ny, uint32_t nz, const float* cx,
                                                        const float* cy, const float* cz, float ox, float oy,
                                                        float oz, float radius, int32_t* obstacle) {
#pragma clang fp contract(off)
  const uint32_t n = nx * ny * nz;
  const float r2 = radius * radius;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const uint32_t k = c % nz, j = (c / nz) % ny, i = c / (ny * nz);
    const float rx = cx[i] - ox, ry = cy[j] - oy, rz = cz[k] - oz;
    obstacle[c] = rx * rx + ry * ry + rz * rz <= r2 ? 1 : 0;
  }
}

// ---- velocity rows: prescribed-velocity rows, blended velocity constraints -------------------
// Per-cell arithmetic in float32 without contraction (the order of the reference kernels); the
// reductions are float64 sums of the float32 per-cell values in workgroup order.
constexpr int kRowSlots = 6;   // active cells, sum |dv|, max |dv|, momentum change (3)
constexpr int kConSlots = 12;  // the six above, primary momentum change (3), secondary (3)
constexpr uint64_t kRowMaxMask = 1ull << 2;

struct VelocityRowArgs {
  uint32_t nx, ny, nz;
  float* u;
  const int32_t* obstacle;
  const int32_t* active;  // prescribed rows: vd_active
  const float* value;     // prescribed rows: the row velocity
  const float *sum, *weight, *psum, *pweight, *ssum, *sweight;  // constraints
  const float *wx, *wy, *wz;
  float scale;  // constraints: blend / (1 + solid mobility ratio), float32
  float rho;
  double* partials;
};

__device__ inline float cell_volume(const VelocityRowArgs& a, uint32_t c) {
#pragma clang fp contract(off)
  const uint32_t k = c % a.nz, j = (c / a.nz) % a.ny, i = c / (a.ny * a.nz);
  return a.wx[i] * a.wy[j] * a.wz[k];
}

__device__ inline float norm3(const float (&v)[3]) {
#pragma clang fp contract(off)
  return sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
}

// _apply_velocity_dirichlet_boundary_rows_kernel (fluid.py:2549-2594): free cells of an active
// row take the row velocity.
__global__ void __launch_bounds__(kBlock) k_velocity_rows(VelocityRowArgs a) {
#pragma clang fp contract(off)
  __shared__ double lds[kRowSlots * (kBlock / 64)];
  double acc[kRowSlots];
#pragma unroll
  for (int s = 0; s < kRowSlots; ++s) acc[s] = 0.0;
  const uint32_t n = a.nx * a.ny * a.nz;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    if (a.active[c] == 0 || a.obstacle[c] != 0) continue;
    float dv[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float nw = a.value[3 * c + d];
      dv[d] = nw - a.u[3 * c + d];
      a.u[3 * c + d] = nw;
    }
    const float vol = cell_volume(a, c);
    const float delta = norm3(dv);
    acc[0] += 1.0;
    acc[1] += (double)delta;
    acc[2] = fmax(acc[2], (double)delta);
#pragma unroll
    for (int d = 0; d < 3; ++d) acc[3 + d] += (double)((a.rho * dv[d]) * vol);
  }
  block_partials<kRowSlots>(acc, a.partials, lds, kRowMaxMask);
}

// _apply_velocity_constraints_kernel (fluid.py:2629-2700): free cells with a positive constraint
// weight move towards sum / weight by `scale`; the primary / secondary parts of the change are
// (scale (part_sum - u_old part_weight)) / weight.
__global__ void __launch_bounds__(kBlock) k_velocity_constraints(VelocityRowArgs a) {
#pragma clang fp contract(off)
  __shared__ double lds[kConSlots * (kBlock / 64)];
  double acc[kConSlots];
#pragma unroll
  for (int s = 0; s < kConSlots; ++s) acc[s] = 0.0;
  const uint32_t n = a.nx * a.ny * a.nz;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const float w = a.weight[c];
    if (!(w > 0.0f) || a.obstacle[c] != 0) continue;
    const float pw = a.pweight[c], sw = a.sweight[c];
    const float vol = cell_volume(a, c);
    float dv[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float old = a.u[3 * c + d];
      const float target = a.sum[3 * c + d] / w;
      const float nw = old + a.scale * (target - old);
      dv[d] = nw - old;
      a.u[3 * c + d] = nw;
      const float pdv = (a.scale * (a.psum[3 * c + d] - old * pw)) / w;
      const float sdv = (a.scale * (a.ssum[3 * c + d] - old * sw)) / w;
      acc[3 + d] += (double)((a.rho * dv[d]) * vol);
      acc[6 + d] += (double)((a.rho * pdv) * vol);
      acc[9 + d] += (double)((a.rho * sdv) * vol);
    }
    const float delta = norm3(dv);
    acc[0] += 1.0;
    acc[1] += (double)delta;
    acc[2] = fmax(acc[2], (double)delta);
  }
  block_partials<kConSlots>(acc, a.partials, lds, kRowMaxMask);
}

// The primary / secondary impulse accumulators gain every application's momentum change.
struct FinConstraintImpulse {
  double* primary;
  double* secondary;
  __device__ void operator()(const double* t) const {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      primary[d] += t[6 + d];
      secondary[d] += t[9 + d];
    }
  }
};

// _local_divergence_cleanup_kernel (fluid.py:5766-5836) on a uniform grid.  A free cell's scale is
// s = (-relaxation (div - source)) / denom, denom summing 1/d^2 over its usable faces (the
// neighbour free, no velocity-Dirichlet row on the face, not a wall); the cell's low face gains
// -s/d and its high face +s/d.  A low face of cell c is usable from both sides under the same
// condition, so each thread gathers the two contributions of its own three low faces (its own
// scale first, then the low neighbour's) instead of scattering with atomics.
struct CleanupArgs {
  uint32_t nx, ny, nz;
  float* u;
  const float* div;
  const float* src;
  const int32_t* obstacle;
  const int32_t* vda;
  float inv[3];   // 1 / d
  float inv2[3];  // 1 / (d d)
  float relax;
};

__device__ inline int cleanup_vd(const CleanupArgs& a, uint32_t c) { return a.vda ? a.vda[c] : 0; }

__device__ inline float cleanup_scale(const CleanupArgs& a, uint32_t c, uint32_t i, uint32_t j, uint32_t k) {
#pragma clang fp contract(off)
  const uint32_t sx = a.ny * a.nz, sy = a.nz;
  const float div = a.div[c] - (a.src ? a.src[c] : 0.0f);
  float denom = 0.0f;
  if (i > 0 && a.obstacle[c - sx] == 0 && cleanup_vd(a, c) == 0) denom += a.inv2[0];
  if (i + 1 < a.nx && a.obstacle[c + sx] == 0 && cleanup_vd(a, c + sx) == 0) denom += a.inv2[0];
  if (j > 0 && a.obstacle[c - sy] == 0 && cleanup_vd(a, c) == 0) denom += a.inv2[1];
  if (j + 1 < a.ny && a.obstacle[c + sy] == 0 && cleanup_vd(a, c + sy) == 0) denom += a.inv2[1];
  if (k > 0 && a.obstacle[c - 1] == 0 && cleanup_vd(a, c) == 0) denom += a.inv2[2];
  if (k + 1 < a.nz && a.obstacle[c + 1] == 0 && cleanup_vd(a, c + 1) == 0) denom += a.inv2[2];
  return denom > 0.0f ? (-a.relax * div) / denom : 0.0f;
}

__global__ void __launch_bounds__(kBlock) k_local_divergence_cleanup(CleanupArgs a) {
#pragma clang fp contract(off)
  const uint32_t n = a.nx * a.ny * a.nz, sx = a.ny * a.nz, sy = a.nz;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    if (a.obstacle[c] != 0 || cleanup_vd(a, c) != 0) continue;  // no usable low face
    const uint32_t k = c % a.nz, j = (c / a.nz) % a.ny, i = c / sx;
    const float s = cleanup_scale(a, c, i, j, k);
    if (i > 0 && a.obstacle[c - sx] == 0) {
      const float sm = cleanup_scale(a, c - sx, i - 1, j, k);
      a.u[3 * c + 0] = (a.u[3 * c + 0] + s * -a.inv[0]) + sm * a.inv[0];
    }
    if (j > 0 && a.obstacle[c - sy] == 0) {
      const float sm = cleanup_scale(a, c - sy, i, j - 1, k);
      a.u[3 * c + 1] = (a.u[3 * c + 1] + s * -a.inv[1]) + sm * a.inv[1];
    }
    if (k > 0 && a.obstacle[c - 1] == 0) {
      const float sm = cleanup_scale(a, c - 1, i, j, k - 1);
      a.u[3 * c + 2] = (a.u[3 * c + 2] + s * -a.inv[2]) + sm * a.inv[2];
    }
  }
}

struct FinStore {  // leave totals in place (read by the host)
  __device__ void operator()(const double*) const {}
};
struct FinFreeVol {
  Scalars* s;
  __device__ void operator()(const double* t) const { s->free_vol = t[0]; }
};
// alpha = rz / dAd, code 1 and first dAd latched when dAd <= 0 (fluid.py:4566-4574).
struct FinDad {
  Scalars* s;
  __device__ void operator()(const double* t) const {
    double dAd = t[0];
    s->dAd = dAd;
    s->alpha = 0.0;
    if (dAd <= 0.0) {
      if (s->code == 0) s->code_dAd = dAd;
      s->code = 1;
    } else {
      s->alpha = s->rz / dAd;
    }
  }
};
// After the preconditioner: t = {<r,z>, <z,q>, sum Vz, sum Vr, sum Vq}.  The
// V-mean of z is removed algebraically (fluid.py:4715-4726), the flexible
// numerator z.(r - r_old) = -alpha z.q (r - r_old = -alpha q on free cells and z
// has zero mean), beta per fluid.py:4589-4601, then rz = rz_new.
struct FinDots5 {
  Scalars* s;
  int remove_mean, use_mg;
  __device__ void operator()(const double* t) const {
    double V = s->free_vol;
    double mz = (remove_mean && V > 0.0) ? t[2] / V : 0.0;
    double rz_new = t[0] - mz * t[3];
    double beta_num = use_mg ? -s->alpha * (t[1] - mz * t[4]) : 0.0;
    double beta = 0.0;
    if (s->rz <= 1.0e-300 || rz_new <= 0.0) {
      s->code = 2;
    } else if (use_mg) {
      beta = beta_num / s->rz;
      if (beta < 0.0) beta = 0.0;
    } else {
      beta = rz_new / s->rz;
    }
    s->mz = mz;
    s->beta = beta;
    s->rz = rz_new;
  }
};
// Start / restart: t = {<r,z>, sum Vz, sum Vr}.
struct FinDots3 {
  Scalars* s;
  int remove_mean;
  __device__ void operator()(const double* t) const {
    double V = s->free_vol;
    double mz = (remove_mean && V > 0.0) ? t[1] / V : 0.0;
    s->mz = mz;
    s->rz = t[0] - mz * t[2];
    s->beta = 0.0;
  }
};
struct FinMeansXR {  // t = {sum Vx, sum Vr}
  Scalars* s;
  __device__ void operator()(const double* t) const {
    double V = s->free_vol;
    s->mx = V > 0.0 ? t[0] / V : 0.0;
    s->mr = V > 0.0 ? t[1] / V : 0.0;
  }
};
struct FinMeanR {  // t = {<r,r>, sum Vr}
  Scalars* s;
  int remove_mean;
  __device__ void operator()(const double* t) const {
    double V = s->free_vol;
    s->mr = (remove_mean && V > 0.0) ? t[1] / V : 0.0;
    s->mx = 0.0;
    s->rr = t[0];
  }
};
// t = {<r,r>_V, sum V r} of the true residual: its norm after the mean
// projection (sum V (r - m)^2 = <r,r>_V - (sum V r)^2 / V) into a pinned host
// slot, the per-iteration convergence monitor of the mixed solve.
struct FinTrueMonitor {
  Scalars* s;
  int remove_mean;
  double* slot;
  __device__ void operator()(const double* t) const {
    const double V = s->free_vol;
    double rr = t[0];
    if (remove_mean && V > 0.0) rr -= t[1] * t[1] / V;
    *slot = rr > 0.0 ? rr : 0.0;
  }
};
struct FinRR {
  Scalars* s;
  __device__ void operator()(const double* t) const { s->rr = t[0]; }
};
struct FinBMean {
  Scalars* s;
  int remove_mean;
  __device__ void operator()(const double* t) const {
    double V = s->free_vol;
    s->mb = (remove_mean && V > 0.0) ? t[0] / V : 0.0;
  }
};
struct FinBNorm {
  Scalars* s;
  __device__ void operator()(const double* t) const { s->bnorm2 = t[0]; }
};

// ---------------------------------------------------------------------------
// Pointwise / reduction functors
// ---------------------------------------------------------------------------

struct OpVolume {
  __device__ void operator()(uint32_t, double V, double (&acc)[1]) const { acc[0] += V; }
};

template <typename TA, typename TB>
struct OpDot {
  const TA* a;
  const TB* b;
  __device__ void operator()(uint32_t c, double V, double (&acc)[1]) const {
    acc[0] += (double)a[c] * (double)b[c] * V;
  }
};

// {<r,r>_V, sum V r} of a stored residual (the sums of k_true_residual).
template <typename TR>
struct OpResidualSums {
  const TR* r;
  __device__ void operator()(uint32_t c, double V, double (&acc)[2]) const {
    const double v = (double)r[c];
    acc[0] += v * v * V;
    acc[1] += v * V;
  }
};

template <typename TR, typename TZ, typename TQ>
struct OpDots5 {
  const TR* r;
  const TZ* z;
  const TQ* q;
  __device__ void operator()(uint32_t c, double V, double (&acc)[5]) const {
    double rv = (double)r[c], zv = (double)z[c], qv = (double)q[c];
    acc[0] += rv * zv * V;
    acc[1] += zv * qv * V;
    acc[2] += zv * V;
    acc[3] += rv * V;
    acc[4] += qv * V;
  }
};

template <typename TR, typename TZ>
struct OpDots3 {
  const TR* r;
  const TZ* z;
  __device__ void operator()(uint32_t c, double V, double (&acc)[3]) const {
    double rv = (double)r[c], zv = (double)z[c];
    acc[0] += rv * zv * V;
    acc[1] += zv * V;
    acc[2] += rv * V;
  }
};

template <typename TR>
struct OpSumsXR {
  const double* x;
  const TR* r;
  __device__ void operator()(uint32_t c, double V, double (&acc)[2]) const {
    acc[0] += x[c] * V;
    acc[1] += (double)r[c] * V;
  }
};

template <typename T>
struct OpSum {
  const T* a;
  __device__ void operator()(uint32_t c, double V, double (&acc)[1]) const { acc[0] += (double)a[c] * V; }
};

// x += alpha d, r -= alpha q; obstacle rows zeroed (_cg_apply_alpha_kernel, fluid.py:4576-4587).
template <typename TD, typename TR, typename TQ>
struct OpCgUpdate {
  double* x;
  const TD* d;
  TR* r;
  const TQ* q;
  const Scalars* s;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const {
    if (f & kObst) {
      x[c] = 0.0;
      r[c] = (TR)0;
      return;
    }
    const double a = s->alpha;
    x[c] += a * (double)d[c];
    r[c] = (TR)((double)r[c] - a * (double)q[c]);
  }
};

// d = (z - mean_z) + beta d (_cg_update_direction_and_rz_kernel, fluid.py:4603-4611,
// with _subtract_cg_weighted_mean_kernel folded in).  first: d = z - mean_z.
template <typename TZ, typename TD>
struct OpCgDir {
  const TZ* z;
  TD* d;
  const Scalars* s;
  int remove_mean, first;
  __device__ void operator()(uint32_t c, bool free, uint8_t f) const {
    double zv = (double)z[c];
    if (remove_mean) zv = free ? zv - s->mz : 0.0;
    if (f & kObst) {
      d[c] = (TD)0;
      return;
    }
    d[c] = first ? (TD)zv : (TD)(zv + s->beta * (double)d[c]);
  }
};

// x -= mx, r -= mr on free cells, 0 elsewhere (fluid.py:4715-4726), with <r,r>.
template <typename TR>
struct OpSubMeans {
  double* x;
  TR* r;
  const Scalars* s;
  __device__ void operator()(uint32_t c, double V, double (&acc)[1]) const {
    double rv = (double)r[c] - s->mr;
    if (x) x[c] = x[c] - s->mx;
    TR rs = (TR)rv;
    r[c] = rs;
    acc[0] += (double)rs * (double)rs * V;
  }
};

template <typename TR>
struct OpZeroNonFree {
  double* x;
  TR* r;
  __device__ void operator()(uint32_t c, bool free, uint8_t) const {
    if (!free) {
      if (x) x[c] = 0.0;
      r[c] = (TR)0;
    }
  }
};

// b -= mean_b on non-obstacle rows, with <b,b> (fluid.py:4471-4482 + 6603).
struct OpBFinal {
  double* b;
  const Scalars* s;
  __device__ void operator()(uint32_t c, double V, double (&acc)[1]) const {
    double v = b[c] - s->mb;
    b[c] = v;
    acc[0] += v * v * V;
  }
};

template <typename TS, typename TD>
struct OpCopy {
  const TS* a;
  TD* b;
  __device__ void operator()(uint32_t c, bool, uint8_t) const { b[c] = (TD)a[c]; }
};

template <typename T>
struct OpFill {
  T* a;
  T v;
  __device__ void operator()(uint32_t c, bool, uint8_t) const { a[c] = v; }
};

// ---------------------------------------------------------------------------
// Mixed-precision solve helpers
// ---------------------------------------------------------------------------

// vin / vout of the mixed V-cycle from t = {<r,r>_V}: RMS = sqrt(<r,r>_V / V_free).
constexpr int kMonRing = 8;  // slots of the convergence-monitor ring (lag < kMonRing)

struct FinVScale {
  Scalars* s;
  double kappa;
  __device__ void operator()(const double* t) const { set(t[0]); }
  __device__ void set(double rr) const {
    const double V = s->free_vol > 0.0 ? s->free_vol : 1.0;
    const double rms = sqrt(fmax(rr, 0.0) / V);
    if (rms > 1.0e-300 && isfinite(rms)) {
      s->vin = 1.0 / rms;
      s->vout = rms / kappa;
    } else {
      s->vin = 1.0;
      s->vout = 1.0 / kappa;
    }
  }
};

// Scale from the residual norm already in the scalars (after a true residual).
__global__ void k_mix_scale_from_rr(Scalars* s, double kappa) {
  if (threadIdx.x == 0 && blockIdx.x == 0) FinVScale{s, kappa}.set(s->rr);
}

// x += alpha d, r -= alpha q (obstacle rows zeroed, fluid.py:4576-4587) and
// <r,r>_V over free cells for the mixed V-cycle scale.
__global__ void __launch_bounds__(kBlock) k_cg_update_rr(OpGeo<double> g, double* x, const float* d, float* r,
                                                          const float* q, const Scalars* s, double* partials) {
  __shared__ double lds[kBlock / 64];
  double acc[1] = {0.0};
  const double a = s->alpha;
  HFSI_CELL_LOOP(g.n) {
    const uint8_t f = g.flags[c];
    if (f & kObst) {
      x[c] = 0.0;
      r[c] = 0.0f;
      continue;
    }
    x[c] += a * (double)d[c];
    const float rn = (float)((double)r[c] - a * (double)q[c]);
    r[c] = rn;
    if (!(f & kNotFree)) {
      uint32_t i, j, k;
      decompose(c, g.ny, g.nz, i, j, k);
      acc[0] += (double)rn * (double)rn * volume64(g, i, j, k);
    }
  }
  block_partials<1>(acc, partials, lds);
}

// ---------------------------------------------------------------------------
// The same CG vector updates four cells per thread (a quad of one row, nz a
// multiple of 4): 16-byte loads and stores, four independent cells per
// memory round trip.  fq divides by nz / 4 (quads per row), fy by ny.  Each
// cell is computed exactly as in the one-cell kernels.
// ---------------------------------------------------------------------------

struct QuadPos {
  uint32_t c0, i, j, k0;
};
__device__ inline QuadPos quad_pos(uint32_t q, const FastDiv& fq, const FastDiv& fy) {
  const uint32_t row = fq.div(q);
  const uint32_t i = fy.div(row);
  return QuadPos{4 * q, i, row - i * fy.d, 4 * (q - row * fq.d)};
}

template <typename TE>
struct Quad;
template <>
struct Quad<__half> {
  static __device__ inline void load(const __half* p, float v[4]) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    const __half2 a = *reinterpret_cast<const __half2*>(&u.x), b = *reinterpret_cast<const __half2*>(&u.y);
    v[0] = __low2float(a); v[1] = __high2float(a); v[2] = __low2float(b); v[3] = __high2float(b);
  }
};
template <>
struct Quad<float> {
  static __device__ inline void load(const float* p, float v[4]) {
    const float4 u = *reinterpret_cast<const float4*>(p);
    v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
  }
};

template <int NS, typename TE>
__global__ void __launch_bounds__(kBlock) k_mix_finish4(OpGeo<double> g, FastDiv fq, FastDiv fy, const TE* e,
                                                         const float* r, const float* q, float* z, const Scalars* s,
                                                         double* partials) {
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) acc[t] = 0.0;
  const float vout = (float)s->vout;
  HFSI_CELL_LOOP(g.n >> 2) {
    const QuadPos P = quad_pos(c, fq, fy);
    const uint32_t f4 = *reinterpret_cast<const uint32_t*>(g.flags + P.c0);
    float ev[4];
    Quad<TE>::load(e + P.c0, ev);
    const float4 r4 = *reinterpret_cast<const float4*>(r + P.c0);
    float4 q4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (NS == 5) q4 = *reinterpret_cast<const float4*>(q + P.c0);
    const double wxy = g.wd[0][P.i] * g.wd[1][P.j];
    const double2 wz01 = *reinterpret_cast<const double2*>(g.wd[2] + P.k0);
    const double2 wz23 = *reinterpret_cast<const double2*>(g.wd[2] + P.k0 + 2);
    const float rv[4] = {r4.x, r4.y, r4.z, r4.w}, qv[4] = {q4.x, q4.y, q4.z, q4.w};
    const double wz[4] = {wz01.x, wz01.y, wz23.x, wz23.y};
    float zo[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t f = (f4 >> (8 * m)) & 0xffu;
      if (f & kNotFree) {
        zo[m] = 0.0f;
        continue;
      }
      const float zf = ev[m] * vout;
      zo[m] = zf;
      const double V = wxy * wz[m];
      const double zd = (double)zf, rd = (double)rv[m];
      acc[0] += rd * zd * V;
      if constexpr (NS == 5) {
        const double qd = (double)qv[m];
        acc[1] += zd * qd * V;
        acc[2] += zd * V;
        acc[3] += rd * V;
        acc[4] += qd * V;
      } else {
        acc[1] += zd * V;
        acc[2] += rd * V;
      }
    }
    *reinterpret_cast<float4*>(z + P.c0) = make_float4(zo[0], zo[1], zo[2], zo[3]);
  }
  block_partials<NS>(acc, partials, lds);
}

// d = z (- mean) + beta d on four cells (OpCgDir on float vectors).
__global__ void __launch_bounds__(kBlock) k_cgdir4(uint32_t n, const uint8_t* flags, const float* z, float* d,
                                                    const Scalars* s, int remove_mean, int first) {
  const double mz = s->mz, beta = s->beta;
  HFSI_CELL_LOOP(n >> 2) {
    const uint32_t c0 = 4 * c;
    const uint32_t f4 = *reinterpret_cast<const uint32_t*>(flags + c0);
    const float4 z4 = *reinterpret_cast<const float4*>(z + c0);
    float4 d4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (!first) d4 = *reinterpret_cast<const float4*>(d + c0);
    const float zv4[4] = {z4.x, z4.y, z4.z, z4.w};
    float* dv = reinterpret_cast<float*>(&d4);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t f = (f4 >> (8 * m)) & 0xffu;
      double zv = (double)zv4[m];
      if (remove_mean) zv = !(f & kNotFree) ? zv - mz : 0.0;
      dv[m] = (f & kObst) ? 0.0f : (first ? (float)zv : (float)(zv + beta * (double)dv[m]));
    }
    *reinterpret_cast<float4*>(d + c0) = d4;
  }
}

// z = e * vout on free cells (0 elsewhere) and the PCG sums of FinDots5
// (NS = 5: <r,z>, <z,q>, sum Vz, sum Vr, sum Vq) or FinDots3 (NS = 3: <r,z>,
// sum Vz, sum Vr).
template <int NS, typename TE>
__global__ void __launch_bounds__(kBlock) k_mix_finish(OpGeo<double> g, const TE* e, const float* r, const float* q,
                                                        float* z, const Scalars* s, double* partials) {
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) acc[t] = 0.0;
  const float vout = (float)s->vout;
  HFSI_CELL_LOOP(g.n) {
    const uint8_t f = g.flags[c];
    if (f & kNotFree) {
      z[c] = 0.0f;
      continue;
    }
    const float zf = ldf<TE>(e, c) * vout;
    z[c] = zf;
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    const double V = volume64(g, i, j, k);
    const double zv = (double)zf, rv = (double)r[c];
    acc[0] += rv * zv * V;
    if (NS == 5) {
      const double qv = (double)q[c];
      acc[1] += zv * qv * V;
      acc[2] += zv * V;
      acc[3] += rv * V;
      acc[4] += qv * V;
    } else {
      acc[1] += zv * V;
      acc[2] += rv * V;
    }
  }
  block_partials<NS>(acc, partials, lds);
}

// Coarse masks of the semi-coarsened hierarchy, through the per-axis child
// tables: a coarse cell is solid (obstacle row, not free) only when no child
// is free.  The reference's 2:1 hierarchy marks a coarse cell solid when any
// child is an obstacle row (fluid.py:5334-5388); that thickens the solid on
// every level, and the coarse correction next to it then stalls the V-cycle
// (energy-norm contraction per cycle 0.73 against 0.19 with this rule on a
// sphere, uniform 16^3).
__global__ void k_mix_coarse_flags(uint32_t cnx, uint32_t cny, uint32_t cnz, const int32_t* fi0, const int32_t* fin,
                                   const int32_t* fj0, const int32_t* fjn, const int32_t* fk0, const int32_t* fkn,
                                   uint32_t fny, uint32_t fnz, const uint8_t* fflags, uint8_t* cflags) {
  const uint32_t n = cnx * cny * cnz;
  HFSI_CELL_LOOP(n) {
    uint32_t ci, cj, ck;
    decompose(c, cny, cnz, ci, cj, ck);
    bool any_free = false;
    for (int32_t oi = 0; oi < fin[ci] && !any_free; ++oi)
      for (int32_t oj = 0; oj < fjn[cj] && !any_free; ++oj)
        for (int32_t ok = 0; ok < fkn[ck] && !any_free; ++ok) {
          const uint32_t fc =
              (uint32_t)(fi0[ci] + oi) * fny * fnz + (uint32_t)(fj0[cj] + oj) * fnz + (uint32_t)(fk0[ck] + ok);
          if (!(fflags[fc] & kNotFree)) any_free = true;
        }
    cflags[c] = any_free ? (uint8_t)0 : (uint8_t)(kObst | kNotFree);
  }
}

// ---------------------------------------------------------------------------
// Mask / geometry kernels
// ---------------------------------------------------------------------------

__global__ void k_flags0(uint32_t n, const int32_t* obstacle, uint8_t* flags) {
  HFSI_CELL_LOOP(n) {
    int32_t v = obstacle[c];
    flags[c] = (uint8_t)((v == 1 ? kObst : 0) | (v != 0 ? kNotFree : 0));
  }
}

// Open-face bits from the neighbours' "not free" bit.
__global__ void k_open_bits(uint32_t nx, uint32_t ny, uint32_t nz, uint8_t* flags) {
  const uint32_t n = nx * ny * nz, sx = ny * nz, sy = nz;
  HFSI_CELL_LOOP(n) {
    uint32_t i, j, k;
    decompose(c, ny, nz, i, j, k);
    uint8_t f = flags[c] & (kObst | kNotFree);
    if (i > 0 && !(flags[c - sx] & kNotFree)) f |= kXm;
    if (i + 1 < nx && !(flags[c + sx] & kNotFree)) f |= kXp;
    if (j > 0 && !(flags[c - sy] & kNotFree)) f |= kYm;
    if (j + 1 < ny && !(flags[c + sy] & kNotFree)) f |= kYp;
    if (k > 0 && !(flags[c - 1] & kNotFree)) f |= kZm;
    if (k + 1 < nz && !(flags[c + 1] & kNotFree)) f |= kZp;
    flags[c] = f;
  }
}

// Level-0 velocity-Dirichlet data: active byte, raw weight, low-face weight.
__global__ void k_vd0(uint32_t n, const int32_t* vda, const float* vdw, uint8_t* act, float* wraw, float* fw) {
  HFSI_CELL_LOOP(n) {
    bool a = vda && vda[c] != 0;
    float w = (a && vdw) ? vdw[c] : 0.0f;
    act[c] = a ? 1 : 0;
    wraw[c] = w;
    fw[c] = a ? fminf(fmaxf(w, 0.0f), 1.0f) : 1.0f;
  }
}

// Coarse obstacle = any child obstacle row; coarse vd = any child active with
// the max child weight; coarse interface diagonal = V-mean over children that
// are not obstacle rows (_mg_restrict_residual_kernel, fluid.py:5334-5388).
struct CoarseMaskArgs {
  uint32_t fnx, fny, fnz, cnx, cny, cnz;
  const uint8_t* fflags;
  uint8_t* cflags;
  const uint8_t* fact;
  const float* fwraw;
  uint8_t* cact;
  float* cwraw;
  float* cfw;
  const double* fdiag;
  double* cdiag;
  const float *fwx, *fwy, *fwz;
};

__global__ void k_coarse_masks(CoarseMaskArgs a) {
  const uint32_t n = a.cnx * a.cny * a.cnz;
  const uint32_t fsx = a.fny * a.fnz, fsy = a.fnz;
  HFSI_CELL_LOOP(n) {
    uint32_t ci, cj, ck;
    decompose(c, a.cny, a.cnz, ci, cj, ck);
    int obst = 0, vdn = 0;
    float vdw = 0.0f;
    double dsum = 0.0, vsum = 0.0;
    for (int oi = 0; oi < 2; ++oi)
      for (int oj = 0; oj < 2; ++oj)
        for (int ok = 0; ok < 2; ++ok) {
          uint32_t fi = 2 * ci + oi, fj = 2 * cj + oj, fk = 2 * ck + ok;
          if (fi < a.fnx && fj < a.fny && fk < a.fnz) {
            uint32_t fc = fi * fsx + fj * fsy + fk;
            if (a.fact && a.fact[fc]) {
              ++vdn;
              vdw = fmaxf(vdw, a.fwraw[fc]);
            }
            if (a.fflags[fc] & kObst) {
              ++obst;
            } else {
              double vol = (double)(a.fwx[fi] * a.fwy[fj] * a.fwz[fk]);
              if (a.fdiag) dsum += a.fdiag[fc] * vol;
              vsum += vol;
            }
          }
        }
    a.cflags[c] = obst > 0 ? (uint8_t)(kObst | kNotFree) : (uint8_t)0;
    if (a.cdiag) a.cdiag[c] = obst > 0 ? 0.0 : (double)(float)(dsum / fmax(vsum, 1.0e-30));
    if (a.cact) {
      a.cact[c] = vdn > 0 ? 1 : 0;
      a.cwraw[c] = vdn > 0 ? vdw : 0.0f;
      a.cfw[c] = vdn > 0 ? fminf(fmaxf(vdw, 0.0f), 1.0f) : 1.0f;
    }
  }
}

// ---------------------------------------------------------------------------
// Velocity-side kernels
// ---------------------------------------------------------------------------

// (_compute_divergence_kernel, fluid.py:3450-3486), float32 arithmetic.
__global__ void k_divergence(OpGeo<float> g, const float* u, float* div) {
  HFSI_CELL_LOOP(g.n) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    uint8_t f = g.flags[c];
    float out = 0.0f;
    if (!(f & kObst)) {
      const float* uc = u + 3 * (size_t)c;
      float lx = (f & kXm) ? uc[0] : 0.0f;
      float rx = (f & kXp) ? u[3 * (size_t)(c + g.sx) + 0] : 0.0f;
      float ly = (f & kYm) ? uc[1] : 0.0f;
      float ry = (f & kYp) ? u[3 * (size_t)(c + g.sy) + 1] : 0.0f;
      float lz = ((g.outlet && k == 0) || (f & kZm)) ? uc[2] : 0.0f;
      float rz = (f & kZp) ? u[3 * (size_t)(c + 1) + 2] : 0.0f;
      float dx = (rx - lx) / g.wf[0][i];
      float dy = (ry - ly) / g.wf[1][j];
      float dz = (rz - lz) / g.wf[2][k];
      out = __fadd_rn(__fadd_rn(dx, dy), dz);
    }
    div[c] = out;
  }
}

// rhs0 = f32(rhs_scale) * (div - source) in float32, minus the interface rhs in
// float64; b_raw = -rhs0 on non-obstacle rows (fluid.py:5228-5243), with sum V b_raw.
struct OpRhs {
  const float* div;
  const float* src;
  const double* iface;
  double* b;
  float scale;
  const uint8_t* flags;
  __device__ void operator()(uint32_t c, double V, double (&acc)[1]) const {
    // only called for free cells by k_sums; obstacle rows set by OpRhsObst
    float d = div[c] - (src ? src[c] : 0.0f);
    double rhs0 = (double)__fmul_rn(scale, d);
    if (iface) rhs0 -= iface[c];
    double v = (flags[c] & kObst) ? 0.0 : -rhs0;
    b[c] = v;
    acc[0] += v * V;
  }
};
struct OpRhsNonFree {
  const float* div;
  const float* src;
  const double* iface;
  double* b;
  float scale;
  __device__ void operator()(uint32_t c, bool free, uint8_t f) const {
    if (free) return;
    if (f & kObst) {
      b[c] = 0.0;
      return;
    }
    float d = div[c] - (src ? src[c] : 0.0f);
    double rhs0 = (double)__fmul_rn(scale, d);
    if (iface) rhs0 -= iface[c];
    b[c] = -rhs0;
  }
};

// Legacy-sign level-0 rhs for the standalone solvers (rhs0 itself).
struct OpRhsLegacy {
  const float* div;
  const float* src;
  const double* iface;
  double* out;
  float scale;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const {
    if (f & kObst) {
      out[c] = 0.0;
      return;
    }
    float d = div[c] - (src ? src[c] : 0.0f);
    double rhs0 = (double)__fmul_rn(scale, d);
    if (iface) rhs0 -= iface[c];
    out[c] = rhs0;
  }
};

// (_subtract_pressure_gradient_kernel, fluid.py:5538-5582).
struct GradArgs {
  OpGeo<double> g;
  float* u;
  const double* p;
  const float *dx, *dy, *dz;  // centre distances (float metrics)
  const int32_t* vda;
  const float* vdw;
  const float* vdv;
  float dt_over_rho;
};

__global__ void k_subtract_gradient(GradArgs a) {
  const OpGeo<double>& g = a.g;
  HFSI_CELL_LOOP(g.n) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    uint8_t f = g.flags[c];
    float* uc = a.u + 3 * (size_t)c;
    if (f & kObst) {
      uc[0] = 0.0f;
      uc[1] = 0.0f;
      uc[2] = 0.0f;
      continue;
    }
    double pc = a.p[c];
    double gx = 0.0, gy = 0.0, gz = 0.0;
    if (f & kXm) gx = (pc - a.p[c - g.sx]) / (double)a.dx[i];
    if (f & kYm) gy = (pc - a.p[c - g.sy]) / (double)a.dy[j];
    if (f & kZm)
      gz = (pc - a.p[c - 1]) / (double)a.dz[k];
    else if (g.outlet && k == 0)
      gz = 2.0 * pc / (double)g.wf[2][k];
    double w = 1.0;
    if (a.vda && a.vda[c] != 0) {
      w = fmin(fmax((double)a.vdw[c], 0.0), 1.0);
      if (w <= 0.0 && a.vdv) {
        uc[0] = a.vdv[3 * (size_t)c + 0];
        uc[1] = a.vdv[3 * (size_t)c + 1];
        uc[2] = a.vdv[3 * (size_t)c + 2];
      }
    }
    if (w > 0.0) {
      double s = w * (double)a.dt_over_rho;
      uc[0] = uc[0] - (float)(s * gx);
      uc[1] = uc[1] - (float)(s * gy);
      uc[2] = uc[2] - (float)(s * gz);
    }
  }
}

// (_apply_closed_boundary_no_normal_flow_kernel, fluid.py:5528-5536).
__global__ void k_wall_clamp(uint32_t nx, uint32_t ny, uint32_t nz, float* u, int outlet) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nyz = ny * nz, nxz = nx * nz, nxy = nx * ny;
  if (tid < nyz) u[3 * (size_t)tid + 0] = 0.0f;  // i = 0
  if (tid < nxz) {
    uint32_t i = tid / nz, k = tid % nz;
    u[3 * ((size_t)i * ny * nz + k) + 1] = 0.0f;  // j = 0
  }
  if (!outlet && tid < nxy) {
    uint32_t i = tid / ny, j = tid % ny;
    u[3 * (((size_t)i * ny + j) * nz) + 2] = 0.0f;  // k = 0
  }
}

// Float64 true residual r = b - A x on non-obstacle rows (axpby of
// fluid.py:4518-4531), stored at TR (not stored when r is null), with
// {<r,r>, sum V r} in float64.
template <typename TR>
__global__ void __launch_bounds__(kBlock) k_true_residual(OpGeo<double> g, const double* x, const double* b, TR* r,
                                                           double* partials) {
  __shared__ double lds[2 * (kBlock / 64)];
  double acc[2] = {0.0, 0.0};
  Ld<double, double> P{x};
  HFSI_CELL_LOOP(g.n) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    uint8_t f = g.flags[c];
    double v = 0.0;
    if (!(f & kObst)) v = b[c] - apply_cell(g, c, i, j, k, P);
    if (r) r[c] = (TR)v;
    if (!(f & kNotFree)) {
      double V = volume64(g, i, j, k);
      acc[0] += v * v * V;
      acc[1] += v * V;
    }
  }
  block_partials<2>(acc, partials, lds);
}

// z = r / diag (_apply_jacobi_preconditioner_kernel, fluid.py:4502-4516).
template <typename C, typename TR, typename TZ>
__global__ void __launch_bounds__(kBlock) k_jacobi_precond(OpGeo<C> g, const TR* r, TZ* z) {
  LdZero<C> P;
  HFSI_CELL_LOOP(g.n) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    uint8_t f = g.flags[c];
    C v = (C)0;
    if (!(f & kObst)) {
      C nb, den;
      nb_den(g, c, i, j, k, f, P, nb, den);
      if (g.diag) den += (C)g.diag[c];
      if (den > (C)0) v = (C)r[c] / den;
    }
    z[c] = (TZ)v;
  }
}

// Compact uniform Jacobi (_pressure_jacobi_kernel, fluid.py:3996-4053).
struct LegacyArgs {
  uint32_t nx, ny, nz;
  const double* p;
  double* out;
  const int32_t* obst;
  const float* div;
  const float* src;
  float rhs_scale, ix2, iy2, iz2;
  int outlet;
};

__global__ void k_legacy_jacobi(LegacyArgs a) {
  const uint32_t n = a.nx * a.ny * a.nz, sx = a.ny * a.nz, sy = a.nz;
  HFSI_CELL_LOOP(n) {
    uint32_t i, j, k;
    decompose(c, a.ny, a.nz, i, j, k);
    uint32_t im = i > 0 ? i - 1 : 0, ip = i + 1 < a.nx ? i + 1 : a.nx - 1;
    uint32_t jm = j > 0 ? j - 1 : 0, jp = j + 1 < a.ny ? j + 1 : a.ny - 1;
    uint32_t km = k > 0 ? k - 1 : 0, kp = k + 1 < a.nz ? k + 1 : a.nz - 1;
    const double* p = a.p;
    const int32_t* o = a.obst;
    uint32_t cxm = im * sx + j * sy + k, cxp = ip * sx + j * sy + k;
    uint32_t cym = i * sx + jm * sy + k, cyp = i * sx + jp * sy + k;
    uint32_t czm = i * sx + j * sy + km, czp = i * sx + j * sy + kp;
    double ix2 = a.ix2, iy2 = a.iy2, iz2 = a.iz2;
    double nb = ix2 * (p[cxm] + p[cxp]) + iy2 * (p[cym] + p[cyp]) + iz2 * (p[czm] + p[czp]);
    double den = 2.0 * (double)(a.ix2 + a.iy2 + a.iz2);
    bool adj = o[cxm] == 1 || o[cxp] == 1 || o[cym] == 1 || o[cyp] == 1 || o[czm] == 1 || o[czp] == 1;
    if (adj || (a.outlet && k == 0)) {
      nb = 0.0;
      den = 0.0;
      if (i > 0 && o[c - sx] == 0) { nb += ix2 * p[c - sx]; den += ix2; }
      if (i + 1 < a.nx && o[c + sx] == 0) { nb += ix2 * p[c + sx]; den += ix2; }
      if (j > 0 && o[c - sy] == 0) { nb += iy2 * p[c - sy]; den += iy2; }
      if (j + 1 < a.ny && o[c + sy] == 0) { nb += iy2 * p[c + sy]; den += iy2; }
      if (k > 0 && o[c - 1] == 0) { nb += iz2 * p[c - 1]; den += iz2; }
      if (k + 1 < a.nz && o[c + 1] == 0) { nb += iz2 * p[c + 1]; den += iz2; }
      if (a.outlet && k == 0) den += 2.0 * iz2;
    }
    float rhs = __fmul_rn(a.rhs_scale, a.div[c] - (a.src ? a.src[c] : 0.0f));
    a.out[c] = (o[c] == 1 || den <= 0.0) ? 0.0 : (nb - (double)rhs) / den;
  }
}

// Divergence report: 18 slots x {max, sum of squares, count}.
struct ReportArgs {
  OpGeo<float> g;
  const float* div;
  const float* src;
  const double* idiv;
  const int32_t* vda;
  double* partials;
  unsigned int* counter;
  double* totals;
};

constexpr int kReportSlots = 54;
constexpr uint64_t kReportMaxMask = 0x9249249249249ull;  // bits 0, 3, 6, ..., 51

// Workgroups (two per CU) up to 16 cells per lane; larger grids take more.  The pass is bound by its
// reduction: 54 float64 slots over a wavefront are some 1300 instructions, as much as 20 cells per lane, so
// fewer wavefronts with more cells each are faster.  With a workgroup per 256 cells (up to 2048) and one
// finishing workgroup for all slots a report took 18.8 + 23.6 us at 64^3 and 33.2 + 40.8 us at 150 x 97 x
// 118 cells; with 512 and a finishing workgroup per slot 13.3 + 3.8 and 24.8 + 4.4 us (256: 11.7 and 34.6 us
// for the pass, 1024: 18.7 and 23.9 us).
constexpr uint32_t kReportBlocks = 512;

__global__ void __launch_bounds__(kBlock) k_div_report(ReportArgs a) {
  constexpr int NS = kReportSlots;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const OpGeo<float>& g = a.g;
  auto add = [&](int slot, double v) {
    acc[slot * 3 + 0] = fmax(acc[slot * 3 + 0], v);
    acc[slot * 3 + 1] += v * v;
    acc[slot * 3 + 2] += 1.0;
  };
  HFSI_CELL_LOOP(g.n) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    uint8_t f = g.flags[c];
    if (f & kNotFree) continue;
    double total = (double)a.div[c] + (a.idiv ? a.idiv[c] : 0.0);
    double raw = fabs(total);
    double res = fabs(total - (a.src ? (double)a.src[c] : 0.0));
    bool interior = i > 0 && i + 1 < g.nx && j > 0 && j + 1 < g.ny && k > 0 && k + 1 < g.nz;
    add(0, raw);
    add(1, res);
    if (interior) {
      add(2, raw);
      add(3, res);
    }
    bool uses_vd = false, correctable = false;
    if (a.vda) {
      uses_vd = a.vda[c] != 0 || (i + 1 < g.nx && a.vda[c + g.sx] != 0) || (j + 1 < g.ny && a.vda[c + g.sy] != 0) ||
                (k + 1 < g.nz && a.vda[c + 1] != 0);
      bool own = a.vda[c] == 0;
      correctable = ((f & kXm) && own) || ((f & kXp) && a.vda[c + g.sx] == 0) || ((f & kYm) && own) ||
                    ((f & kYp) && a.vda[c + g.sy] == 0) || ((f & kZm) && own) || ((f & kZp) && a.vda[c + 1] == 0) ||
                    (g.outlet && k == 0 && own);
    } else {
      correctable = (f & (kXm | kXp | kYm | kYp | kZm | kZp)) || (g.outlet && k == 0);
    }
    if (uses_vd) {
      add(4, raw);
      add(5, res);
    } else {
      add(6, raw);
      add(7, res);
    }
    if (correctable) {
      add(8, raw);
      add(9, res);
      if (interior) {
        add(12, raw);
        add(13, res);
      }
    } else {
      add(10, raw);
      add(11, res);
      if (interior) {
        add(14, raw);
        add(15, res);
      }
    }
  }
  // max for slot*3, sums otherwise
  block_partials<NS>(acc, a.partials, lds, kReportMaxMask);
}

// Combine the report's partial rows, a workgroup per slot (the rows come from every XCD: each load is a
// round trip past this XCD's L2, and the slots' trips run side by side).
__global__ void __launch_bounds__(kFinishThreads) k_finish_report(const double* partials, uint32_t nblocks,
                                                                   double* totals) {
  __shared__ double lds[kFinishThreads / 64];
  const uint32_t s = blockIdx.x;
  const bool mx = (kReportMaxMask >> s) & 1;
  double acc[1] = {mx ? -INFINITY : 0.0};
  for (uint32_t b = threadIdx.x; b < nblocks; b += kFinishThreads) {
    const double p = partials[(size_t)b * kReportSlots + s];
    acc[0] = mx ? fmax(acc[0], p) : acc[0] + p;
  }
  if (mx)
    block_reduce<1>(acc, lds, 1ull);
  else
    block_reduce<1>(acc, lds, 0ull);
  if (threadIdx.x == 0) totals[s] = acc[0];
}

// ---------------------------------------------------------------------------
// Single-workgroup V-cycle tail for the small levels
// ---------------------------------------------------------------------------

template <typename C, typename TV>
struct TailLevel {
  OpGeo<C> g;
  TV* p;
  TV* t;
  TV* rhs;
};

// LDS layout of the tail levels (byte offsets into dynamic shared memory).  The flags, coefficients and
// widths of all levels form one image, packed in global memory when the masks are set (k_tail_pack).
struct TailLdsPlan {
  uint32_t bytes;  // 0: the tail does not fit, run it from global memory
  uint32_t off_image, image_bytes;
  uint32_t off_work;  // C per cell of the largest level that is prolongated onto
  uint32_t off_p[kMaxLevels], off_t[kMaxLevels], off_rhs[kMaxLevels], off_flags[kMaxLevels];
  uint32_t off_cl[kMaxLevels][3], off_ch[kMaxLevels][3], off_wf[kMaxLevels][3];
};

template <typename C, typename TV>
struct TailArgs {
  TailLevel<C, TV> lv[kMaxLevels];
  int first, last;  // levels [first, last] run in the tail; last is the coarsest
  TailLdsPlan plan;
};

template <typename C, typename P, typename R, typename TOut>
__device__ inline void tail_sweep(const OpGeo<C>& g, const P& p, const R& rhs, TOut* out, C omega) {
  for (uint32_t c = threadIdx.x; c < g.n; c += blockDim.x) {
    uint32_t i, j, k;
    decompose(c, g.ny, g.nz, i, j, k);
    out[c] = (TOut)jacobi_cell(g, c, i, j, k, p, rhs, omega);
  }
  __syncthreads();
}

// Writes m = 1..W of a level go to P when (W - m) is even, else to T, so the
// final smoothed value always ends in P.
template <typename TV>
__device__ __host__ inline TV* sweep_target(TV* P, TV* T, int W, int m) {
  return ((W - m) % 2 == 0) ? P : T;
}

// V-cycle over levels [first, last] from zero initial guesses, rhs[first]
// given; the result of level `first` ends in lv[first].p.
template <typename C, typename TV>
__device__ inline void tail_body(const TailLevel<C, TV>* lv, int first, int last, int pre, int coarse, int post,
                                 C omega, C scale) {
  TV* cur[kMaxLevels];
  for (int l = first; l < last; ++l) {
    const TailLevel<C, TV>& L = lv[l];
    const int W = pre + post;
    Ld<TV, C> R{L.rhs};
    TV* out = sweep_target(L.p, L.t, W, 1);
    tail_sweep(L.g, LdZero<C>{}, R, out, omega);
    TV* in = out;
    for (int m = 2; m <= pre; ++m) {
      out = sweep_target(L.p, L.t, W, m);
      tail_sweep(L.g, Ld<TV, C>{in}, R, out, omega);
      in = out;
    }
    cur[l] = in;
    const TailLevel<C, TV>& Cl = lv[l + 1];
    for (uint32_t c = threadIdx.x; c < Cl.g.n; c += blockDim.x) {
      uint32_t ci, cj, ck;
      decompose(c, Cl.g.ny, Cl.g.nz, ci, cj, ck);
      C v = (C)0;
      if (!(Cl.g.flags[c] & kObst)) v = restrict_cell<TV>(L.g, ci, cj, ck, Ld<TV, C>{in}, R);
      Cl.rhs[c] = (TV)v;
    }
    __syncthreads();
  }
  {  // coarsest
    const TailLevel<C, TV>& L = lv[last];
    Ld<TV, C> R{L.rhs};
    TV* out = sweep_target(L.p, L.t, coarse, 1);
    tail_sweep(L.g, LdZero<C>{}, R, out, omega);
    TV* in = out;
    for (int m = 2; m <= coarse; ++m) {
      out = sweep_target(L.p, L.t, coarse, m);
      tail_sweep(L.g, Ld<TV, C>{in}, R, out, omega);
      in = out;
    }
    cur[last] = in;
  }
  for (int l = last - 1; l >= first; --l) {
    const TailLevel<C, TV>& L = lv[l];
    const TailLevel<C, TV>& Cl = lv[l + 1];
    const int W = pre + post;
    Ld<TV, C> R{L.rhs};
    LdProlong<TV, TV, C> PP{cur[l], cur[l + 1], L.g.flags, Cl.g.nx, Cl.g.ny, Cl.g.nz, Cl.g.sx, Cl.g.sy, scale};
    TV* out = sweep_target(L.p, L.t, W, pre + 1);
    tail_sweep(L.g, PP, R, out, omega);
    TV* in = out;
    for (int m = pre + 2; m <= W; ++m) {
      out = sweep_target(L.p, L.t, W, m);
      tail_sweep(L.g, Ld<TV, C>{in}, R, out, omega);
      in = out;
    }
    cur[l] = in;
  }
}

template <typename C, typename TV>
__global__ void __launch_bounds__(kTailThreads) k_vcycle_tail(const TailArgs<C, TV>* args, int pre, int coarse,
                                                              int post, C omega, C scale) {
  tail_body<C, TV>(args->lv, args->first, args->last, pre, coarse, post, omega, scale);
}

template <typename T>
__device__ inline void block_copy(T* dst, const T* src, uint32_t n) {
  for (uint32_t c = threadIdx.x; c < n; c += blockDim.x) dst[c] = src[c];
}

// The image of the tail's flags and metrics, laid out as the tail workgroup holds it in LDS.
template <typename C>
__global__ void __launch_bounds__(kTailThreads) k_tail_pack(const TailArgs<C, float>* args, unsigned char* image) {
  const TailArgs<C, float>& A = *args;
  const TailLdsPlan& P = A.plan;
  unsigned char* at = image - P.off_image;
  for (int l = A.first; l <= A.last; ++l) {
    const OpGeo<C>& g = A.lv[l].g;
    block_copy(at + P.off_flags[l], g.flags, g.n);
    const uint32_t len[3] = {g.nx, g.ny, g.nz};
    for (int a = 0; a < 3; ++a) {
      block_copy(reinterpret_cast<C*>(at + P.off_cl[l][a]), g.cl[a], len[a]);
      block_copy(reinterpret_cast<C*>(at + P.off_ch[l][a]), g.ch[a], len[a]);
      block_copy(reinterpret_cast<float*>(at + P.off_wf[l][a]), g.wf[a], len[a]);
    }
  }
}

// A tail level as the workgroup sees it: LDS byte offsets.
template <typename C>
struct TailShape {
  uint32_t nx, ny, nz, n, sx, sy;
  uint32_t p, t, rhs, flags, cl[3], ch[3], wf[3];
  const float* fw;
  const double* diag;
  C outlet_add;
  int outlet;
};

// The shape of level l in scalar registers.
template <typename C>
__device__ inline TailShape<C> tail_shape(const TailShape<C>* shapes, int l) {
  static_assert(sizeof(TailShape<C>) % 4 == 0, "words");
  TailShape<C> S;
  const uint32_t* src = reinterpret_cast<const uint32_t*>(shapes + l);
  uint32_t* dst = reinterpret_cast<uint32_t*>(&S);
#pragma unroll
  for (uint32_t w = 0; w < sizeof(S) / 4; ++w) dst[w] = __builtin_amdgcn_readfirstlane(src[w]);
  return S;
}

// The cells of one level that a thread owns (c = base + thread + 1024 q), what does not change between
// the passes over it: position and open faces, and the diagonal (0 for an obstacle; cells whose diagonal
// is not positive hold 0).
constexpr int kTailQ = (int)kTailCells / kTailThreads;
template <typename C>
struct TailCells {
  uint32_t at[kTailQ];  // i | j << 16
  uint32_t kf[kTailQ];  // k | flags << 16
  C den[kTailQ];
};

// c / n for c < 2^20: the quotient's distance to the next integer, 0.5 / n, is far above its error
__device__ inline uint32_t small_div(uint32_t c, uint32_t n) { return (uint32_t)(((float)c + 0.5f) / (float)n); }

// Neighbour sum (in the order of nb_den) of the cell c at (i, j, k) with flags f, and its diagonal when
// DEN.  A closed face contributes an exact zero: coefficient 0 times the cell itself.
template <bool DEN, bool NB, typename C, typename TP>
__device__ inline void tail_nb(const unsigned char* smem, const TailShape<C>& L, uint32_t c, uint32_t ij, uint32_t kf,
                               const TP* p, C& nb, C& den) {
  const uint32_t pos[3] = {ij & 0xffffu, ij >> 16, kf & 0xffffu}, f = kf >> 16;
  const uint32_t stride[3] = {L.sx, L.sy, 1u};
  constexpr uint32_t lo_bit[3] = {kXm, kYm, kZm}, hi_bit[3] = {kXp, kYp, kZp};
  nb = (C)0;
  den = (C)0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const bool lo = f & lo_bit[a], hi = f & hi_bit[a];
    C cl = reinterpret_cast<const C*>(smem + L.cl[a])[pos[a]], ch = reinterpret_cast<const C*>(smem + L.ch[a])[pos[a]];
    const uint32_t cm = lo ? c - stride[a] : c, cp = hi ? c + stride[a] : c;
    if (L.fw) {
      cl *= (C)L.fw[c];
      ch *= (C)L.fw[cp];
    }
    cl = lo ? cl : (C)0;
    ch = hi ? ch : (C)0;
    if (NB) {
      nb += cl * (C)p[cm];
      nb += ch * (C)p[cp];
    }
    if (DEN) {
      den += cl;
      den += ch;
    }
  }
}

template <typename C>
__device__ inline void tail_setup(const unsigned char* smem, const TailShape<C>& L, uint32_t base, TailCells<C>& K) {
#pragma unroll
  for (int q = 0; q < kTailQ; ++q) {
    const uint32_t c = base + threadIdx.x + q * kTailThreads;
    K.at[q] = K.kf[q] = 0;
    K.den[q] = (C)0;
    if (c >= L.n) continue;
    const uint32_t ij = small_div(c, L.nz), k = c - ij * L.nz, i = small_div(ij, L.ny), j = ij - i * L.ny;
    const uint32_t f = smem[L.flags + c];
    K.at[q] = i | j << 16;
    K.kf[q] = k | f << 16;
    C nb, den;
    tail_nb<true, false>(smem, L, c, K.at[q], K.kf[q], (const float*)nullptr, nb, den);
    if (L.outlet && k == 0) den += L.outlet_add;
    if (L.diag) den += (C)L.diag[c];
    if (!(f & kObst)) K.den[q] = den;
  }
}

// out = one weighted-Jacobi update of p (ZERO: of the zero iterate).
template <bool ZERO, typename C, typename TP>
__device__ inline void tail_jacobi(const unsigned char* smem, const TailShape<C>& L, uint32_t base,
                                   const TailCells<C>& K, const TP* p, float* out, C omega) {
  const float* rhs = reinterpret_cast<const float*>(smem + L.rhs);
#pragma unroll
  for (int q = 0; q < kTailQ; ++q) {
    const uint32_t c = base + threadIdx.x + q * kTailThreads;
    if (c >= L.n) continue;
    C v = (C)0;
    if (K.den[q] > (C)0) {
      C nb, unused;
      tail_nb<false, !ZERO>(smem, L, c, K.at[q], K.kf[q], p, nb, unused);
      const C pc = ZERO ? (C)0 : (C)p[c];
      const C jac = (nb - (C)rhs[c]) / K.den[q];
      v = pc + omega * (jac - pc);
    }
    out[c] = (float)v;
  }
}

// Same V-cycle tail with every level in LDS, bound by the latency of its ~50 dependent passes.  A
// thread's cells keep their position and diagonal in registers over a level's passes, LDS is addressed as LDS (the level-pointer form compiled to flat loads), the residual is
// formed per fine cell before it is gathered, levels of at most 64 cells run in the first wavefront
// without barriers, and the masks and metrics arrive as one packed image: 107 -> 52 us per V-cycle at
// 64^3 in float64 (16^3 cells down), bit for bit the same.
template <typename C>
__global__ void __launch_bounds__(kTailThreads) k_vcycle_tail_lds(const TailArgs<C, float>* args,
                                                                  const unsigned char* image, int pre, int coarse,
                                                                  int post, C omega, C scale) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ TailShape<C> shapes[kMaxLevels];
  const TailArgs<C, float>& A = *args;
  const TailLdsPlan& P = A.plan;
  const int first = A.first, last = A.last, tid = threadIdx.x;
  for (uint32_t v = tid; v < P.image_bytes / 16; v += kTailThreads)
    reinterpret_cast<uint4*>(smem + P.off_image)[v] = reinterpret_cast<const uint4*>(image)[v];
  block_copy(reinterpret_cast<float*>(smem + P.off_rhs[first]), A.lv[first].rhs, A.lv[first].g.n);
  if (tid >= first && tid <= last) {
    const int l = tid;
    const OpGeo<C>& g = A.lv[l].g;
    TailShape<C> S;
    S.nx = g.nx; S.ny = g.ny; S.nz = g.nz; S.n = g.n; S.sx = g.sx; S.sy = g.sy;
    S.p = P.off_p[l]; S.t = P.off_t[l]; S.rhs = P.off_rhs[l]; S.flags = P.off_flags[l];
    for (int a = 0; a < 3; ++a) {
      S.cl[a] = P.off_cl[l][a];
      S.ch[a] = P.off_ch[l][a];
      S.wf[a] = P.off_wf[l][a];
    }
    S.fw = g.fw;
    S.diag = g.diag;
    S.outlet_add = g.outlet_add;
    S.outlet = g.outlet;
    shapes[l] = S;
  }
  __syncthreads();
  C* work = reinterpret_cast<C*>(smem + P.off_work);
  auto buf = [&](uint32_t off) { return reinterpret_cast<float*>(smem + off); };
  // end of a pass over a level of n cells: one wavefront's LDS accesses are in order by themselves
  auto sync = [](uint32_t n) {
    if (n <= 64) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
  };
  TailCells<C> K;
  // one pass of `f(base)` over a level's cells; levels beyond a thread's kTailQ cells set up per pass
  auto each = [&](const TailShape<C>& L, auto f) {
    if ((uint32_t)(tid & ~63) >= L.n) return;
    for (uint32_t base = 0; base < L.n; base += kTailCells) {
      if (L.n > kTailCells) tail_setup(smem, L, base, K);
      f(base);
    }
  };
  auto begin = [&](const TailShape<C>& L) {
    if (L.n <= kTailCells && (uint32_t)(tid & ~63) < L.n) tail_setup(smem, L, 0, K);
  };
  // where pass m of W over a level writes: the last one to p
  auto target = [](const TailShape<C>& L, int W, int m) { return (W - m) % 2 == 0 ? L.p : L.t; };
  const int W = pre + post;
  for (int l = first; l < last; ++l) {
    const TailShape<C> L = tail_shape(shapes, l);
    begin(L);
    uint32_t out = target(L, W, 1);
    each(L, [&](uint32_t base) { tail_jacobi<true>(smem, L, base, K, (const float*)nullptr, buf(out), omega); });
    sync(L.n);
    uint32_t in = out;
    for (int m = 2; m <= pre; ++m) {
      out = target(L, W, m);
      each(L, [&](uint32_t base) { tail_jacobi<false>(smem, L, base, K, (const float*)buf(in), buf(out), omega); });
      sync(L.n);
      in = out;
    }
    // residual of every fine cell into the other buffer, then the volume-weighted means
    const uint32_t res = in == L.p ? L.t : L.p;
    each(L, [&](uint32_t base) {
      const float *p = buf(in), *rhs = buf(L.rhs);
      float* r = buf(res);
#pragma unroll
      for (int q = 0; q < kTailQ; ++q) {
        const uint32_t c = base + tid + q * kTailThreads;
        if (c >= L.n || (K.kf[q] >> 16 & kObst)) continue;
        C nb, den;
        tail_nb<false, true>(smem, L, c, K.at[q], K.kf[q], p, nb, den);
        r[c] = (float)((C)rhs[c] - (nb - K.den[q] * (C)p[c]));
      }
    });
    sync(L.n);
    const TailShape<C> G = tail_shape(shapes, l + 1);
    for (uint32_t c = tid; c < G.n; c += kTailThreads) {
      C v = (C)0;
      if (!(smem[G.flags + c] & kObst)) {
        const uint32_t ij = small_div(c, G.nz), ck = c - ij * G.nz, ci = small_div(ij, G.ny), cj = ij - ci * G.ny;
        C rsum = (C)0, vsum = (C)0;
#pragma unroll
        for (int o = 0; o < 8; ++o) {
          const uint32_t fi = 2 * ci + (o >> 2), fj = 2 * cj + (o >> 1 & 1), fk = 2 * ck + (o & 1);
          if (fi < L.nx && fj < L.ny && fk < L.nz) {
            const uint32_t fc = fi * L.sx + fj * L.sy + fk;
            if (!(smem[L.flags + fc] & kObst)) {
              const C vol = (C)(buf(L.wf[0])[fi] * buf(L.wf[1])[fj] * buf(L.wf[2])[fk]);
              rsum += (C)buf(res)[fc] * vol;
              vsum += vol;
            }
          }
        }
        v = rsum / (vsum > (C)1.0e-30 ? vsum : (C)1.0e-30);
      }
      buf(G.rhs)[c] = (float)v;
    }
    sync(G.n);  // a level of at most 64 cells was written by the wavefront that continues with it
  }
  {  // coarsest
    const TailShape<C> L = tail_shape(shapes, last);
    begin(L);
    uint32_t out = target(L, coarse, 1);
    each(L, [&](uint32_t base) { tail_jacobi<true>(smem, L, base, K, (const float*)nullptr, buf(out), omega); });
    sync(L.n);
    uint32_t in = out;
    for (int m = 2; m <= coarse; ++m) {
      out = target(L, coarse, m);
      each(L, [&](uint32_t base) { tail_jacobi<false>(smem, L, base, K, (const float*)buf(in), buf(out), omega); });
      sync(L.n);
      in = out;
    }
  }
  for (int l = last - 1; l >= first; --l) {
    const TailShape<C> L = tail_shape(shapes, l), G = tail_shape(shapes, l + 1);
    if (L.n > 64 && G.n <= 64) __syncthreads();  // the first wavefront's levels are done
    begin(L);
    // the prolongated iterate, unrounded, then the sweeps
    const uint32_t fine = target(L, W, max(pre, 1));
    const uint32_t corr = l + 1 == last ? target(G, coarse, max(coarse, 1)) : target(G, W, max(W, pre + 1));
    for (uint32_t c = tid; c < L.n; c += kTailThreads) {
      C v = (C)buf(fine)[c];
      if (!(smem[L.flags + c] & kNotFree)) {
        const uint32_t ij = small_div(c, L.nz), k = c - ij * L.nz, i = small_div(ij, L.ny), j = ij - i * L.ny;
        const uint32_t ci = min(i >> 1, G.nx - 1), cj = min(j >> 1, G.ny - 1), ck = min(k >> 1, G.nz - 1);
        v += scale * (C)buf(corr)[ci * G.sx + cj * G.sy + ck];
      }
      work[c] = v;
    }
    sync(L.n);
    uint32_t out = target(L, W, pre + 1);
    each(L, [&](uint32_t base) { tail_jacobi<false>(smem, L, base, K, (const C*)work, buf(out), omega); });
    sync(L.n);
    uint32_t in = out;
    for (int m = pre + 2; m <= W; ++m) {
      out = target(L, W, m);
      each(L, [&](uint32_t base) { tail_jacobi<false>(smem, L, base, K, (const float*)buf(in), buf(out), omega); });
      sync(L.n);
      in = out;
    }
  }
  if (A.lv[first].g.n <= 64) __syncthreads();
  block_copy(A.lv[first].p, (const float*)(smem + P.off_p[first]), A.lv[first].g.n);
}

// ---------------------------------------------------------------------------
// Handle
// ---------------------------------------------------------------------------

struct LevelMem {
  uint32_t nx, ny, nz, n;
  uint8_t* flags = nullptr;
  uint8_t* vact = nullptr;
  float* vwraw = nullptr;
  float* fw = nullptr;
  double* diag = nullptr;
  double* cl[3] = {};
  double* ch[3] = {};
  float* clf[3] = {};
  float* chf[3] = {};
  float* wf[3] = {};
  double* wd[3] = {};
  float* df[3] = {};  // centre distances (float)
  double outlet_add = 0.0;
  // coarse-level V-cycle storage (levels >= 1), float
  float* p = nullptr;
  float* t = nullptr;
  float* rhs = nullptr;
};

// One level of the semi-coarsened hierarchy of the mixed V-cycle.  Level 0
// shares the main level-0 flags; e / rhs buffers are sized for float32 and
// hold fp16 when the level is stored in half precision.
struct MixLevel {
  uint32_t nx = 0, ny = 0, nz = 0, n = 0;
  uint8_t* flags = nullptr;
  float* cl[3] = {};   // coefficients / kappa
  float* ch[3] = {};
  float* wf[3] = {};   // float widths (restriction volumes)
  double* wd[3] = {};
  float outlet_add = 0.0f;  // 2 / w_z[0]^2 / kappa
  void* e = nullptr;
  void* e2 = nullptr;       // second iterate buffer of the fused sweeps (grid-launched levels, nz even)
  void* cur = nullptr;      // the level's iterate during a V-cycle: e or e2
  void* rhs = nullptr;      // unused on level 0 (the CG residual is the input)
  void* res = nullptr;      // residual scratch of the two-pass restriction (grid-launched levels)
  // transfer to level + 1 (fine side): parent, interpolation partner, parent weight
  int32_t* par[3] = {};
  int32_t* pnb[3] = {};
  float* pw[3] = {};
  // children in level - 1 (coarse side)
  int32_t* first[3] = {};
  int32_t* cnt[3] = {};
};

}  // namespace hfsi

struct hfsi_fluid {
  int L = 0;
  int tail_first = 0;
  int prec_mask = 0;
  bool uniform = true;
  bool has_vd = false, has_diag = false;
  hfsi::LevelMem lv[hfsi::kMaxLevels];
  std::vector<void*> allocs;
  size_t bytes = 0;
  // workspaces
  double* b = nullptr;     // float64 right-hand side
  double* r64 = nullptr;   // REF vectors
  double* d64 = nullptr;
  double* q64 = nullptr;
  double* z64 = nullptr;
  double* t64 = nullptr;
  float* r32 = nullptr;    // FP32 vectors
  float* d32 = nullptr;
  float* q32 = nullptr;
  float* z32 = nullptr;
  float* t32 = nullptr;
  double* partials = nullptr;
  unsigned int* counter = nullptr;
  double* totals = nullptr;
  hfsi::Scalars* scal = nullptr;
  hfsi::Scalars* host_scal = nullptr;  // pinned
  double* host_totals = nullptr;       // pinned
  void* tail_args_d = nullptr;  // TailArgs<double,float>
  void* tail_args_f = nullptr;  // TailArgs<float,float>
  unsigned char *tail_image_d = nullptr, *tail_image_f = nullptr;  // packed masks and metrics (k_tail_pack)
  uint32_t tail_lds_bytes_d = 0, tail_lds_bytes_f = 0;
  int tail_outlet = -1;  // outlet switch last written into both tail geometries (-1: none yet)
  // mixed-precision V-cycle (HFSI_PREC_MIXED)
  int ML = 0;
  int mix_tail_first = 0;
  uint32_t mix_tail_lds = 0;  // dynamic LDS bytes of k_mix_tail
  double mix_kappa = 1.0;
  uint32_t mix_half_min_cells = 1u << 20;  // levels with at least this many cells store fp16
  uint32_t mix_fused_min_cells = 1u << 21;  // fused two-colour sweeps (k_mix_sweep) on levels this large
  uint32_t mix_sweep_wgs = 1280;            // target workgroup count of a fused sweep (sets planes per chunk):
                                            // 5 resident per CU x 256 CUs, one round of workgroups
  hfsi::MixLevel ml[hfsi::kMixMaxLevels];
  void* mix_tail_args = nullptr;  // MixTailArgs (device)
  int mix_tail_outlet = -1;       // outlet switch the tail arguments were written for
  // float64 dense solve of the coarsest mixed level (at most kMixDenseMax cells): host copies of its
  // metrics, and per outlet switch the inverse of its V-weighted operator (null space shifted)
  std::vector<float> mixd_cl[3], mixd_ch[3], mixd_wf[3];
  float mixd_outlet_add = 0.0f;
  int mixd_m = 0;               // free cells of the coarsest level; 0: the tail sweeps it instead
  int32_t* mixd_idx = nullptr;  // [kMixDenseMax] cell of each free cell
  double* mixd_vol = nullptr;   // [kMixDenseMax] its volume
  double* mixd_inv[2] = {};     // [kMixDenseMax^2] row-major inverse, closed / z-min outlet
  // convergence monitor of the mixed solve: pinned ring of <r,r>_V values and their events
  double* mon_ring = nullptr;
  std::vector<hipEvent_t> mon_events;
  // live kernel timer: HIP events recorded on the launch stream around every
  // launch of one selected kernel (HFSI_TIMER_*), summed at flush/read time
  int timer_id = 0;
  std::vector<hipEvent_t> timer_events;
  int timer_used = 0;
  double timer_ms = 0.0;
  long timer_count = 0;
  // compiled pressure-interface couplings (hfsi_fluid_set_interface_couplings)
  hfsi::CoupleList cpl{};
  uint32_t cpl_n = 0, cpl_cap = 0;
  hfsi::CoupleStats* cpl_stats = nullptr;
  // BiCGSTAB fallback: shadow residual and s vectors (float64, allocated with the REF64 vectors)
  double* bi_rold = nullptr;
  double* bi_s = nullptr;
};

namespace hfsi {

template <typename T>
static int dalloc(hfsi_fluid* h, T** out, size_t count) {
  void* p = nullptr;
  size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
  HFSI_CHECK(hipMalloc(&p, bytes));
  h->allocs.push_back(p);
  h->bytes += bytes;
  *out = (T*)p;
  return HFSI_OK;
}

#define HFSI_TRY(expr)         \
  do {                         \
    int _rc = (expr);          \
    if (_rc != HFSI_OK) return _rc; \
  } while (0)

template <typename C>
static OpGeo<C> geo(const hfsi_fluid* h, int l, int outlet);

template <>
OpGeo<double> geo<double>(const hfsi_fluid* h, int l, int outlet) {
  const LevelMem& m = h->lv[l];
  OpGeo<double> g;
  g.nx = m.nx; g.ny = m.ny; g.nz = m.nz; g.n = m.n; g.sx = m.ny * m.nz; g.sy = m.nz;
  g.flags = m.flags;
  g.fw = h->has_vd ? m.fw : nullptr;
  g.diag = h->has_diag ? m.diag : nullptr;
  for (int a = 0; a < 3; ++a) {
    g.cl[a] = m.cl[a];
    g.ch[a] = m.ch[a];
    g.wf[a] = m.wf[a];
    g.wd[a] = m.wd[a];
  }
  g.outlet_add = m.outlet_add;
  g.outlet = outlet;
  return g;
}

template <>
OpGeo<float> geo<float>(const hfsi_fluid* h, int l, int outlet) {
  const LevelMem& m = h->lv[l];
  OpGeo<float> g;
  g.nx = m.nx; g.ny = m.ny; g.nz = m.nz; g.n = m.n; g.sx = m.ny * m.nz; g.sy = m.nz;
  g.flags = m.flags;
  g.fw = h->has_vd ? m.fw : nullptr;
  g.diag = h->has_diag ? m.diag : nullptr;
  for (int a = 0; a < 3; ++a) {
    g.cl[a] = m.clf[a];
    g.ch[a] = m.chf[a];
    g.wf[a] = m.wf[a];
    g.wd[a] = m.wd[a];
  }
  g.outlet_add = (float)m.outlet_add;
  g.outlet = outlet;
  return g;
}

static inline uint32_t blocks_for(uint32_t n) { return grid_blocks(n, kMaxGrid); }

template <typename Op>
static int launch_pointwise(hfsi_fluid* h, int l, Op op, hipStream_t st) {
  const LevelMem& m = h->lv[l];
  hipLaunchKernelGGL(k_pointwise<Op>, dim3(blocks_for(m.n)), dim3(kBlock), 0, st, m.n, m.flags, op);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

// d = z (- mean) + beta d, four cells per thread on float vectors.
template <typename TV>
static int launch_cgdir(hfsi_fluid* h, const TV* z, TV* d, const Scalars* sc, int rm, int first, hipStream_t st) {
  const LevelMem& m = h->lv[0];
  if (std::is_same<TV, float>::value && m.n % 4 == 0) {
    hipLaunchKernelGGL(k_cgdir4, dim3(blocks_for(m.n / 4)), dim3(kBlock), 0, st, m.n, m.flags,
                       reinterpret_cast<const float*>(z), reinterpret_cast<float*>(d), sc, rm, first);
    HFSI_LAUNCH_CHECK();
    return HFSI_OK;
  }
  return launch_pointwise(h, 0, OpCgDir<TV, TV>{z, d, sc, rm, first}, st);
}

// Combine the partials of a reducing launch of `nblocks` workgroups and run `fin`.
template <int NS, typename Fin>
static void finish_sums(hfsi_fluid* h, uint32_t nblocks, Fin fin, hipStream_t st, uint64_t maxmask = 0) {
  hipLaunchKernelGGL((k_finish_sums<NS, Fin>), dim3(1), dim3(kFinishThreads), 0, st, (const double*)h->partials,
                     nblocks, h->totals, fin, maxmask);
}

template <int NS, typename C, typename Op, typename Fin>
static int launch_sums(hfsi_fluid* h, const OpGeo<C>& g, Op op, Fin fin, hipStream_t st) {
  const uint32_t nb = blocks_for(g.n);
  hipLaunchKernelGGL((k_sums<NS, C, Op>), dim3(nb), dim3(kBlock), 0, st, g, op, h->partials);
  finish_sums<NS>(h, nb, fin, st);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

// out += scale * (C p) over the compiled interface couplings.
template <typename TP, typename TO>
static int launch_couple(hfsi_fluid* h, const TP* p, TO* out, double scale, hipStream_t st) {
  if (!h->cpl_n) return HFSI_OK;
  const uint32_t blocks = std::min<uint32_t>((h->cpl_n + kBlock - 1) / kBlock, kMaxGrid);
  hipLaunchKernelGGL((k_couple_apply<TP, TO>), dim3(blocks), dim3(kBlock), 0, st, h->cpl, h->cpl_n, p, out, scale);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

static int sync_scalars(hfsi_fluid* h, hipStream_t st) {
  HFSI_CHECK(hipMemcpyAsync(h->host_scal, h->scal, sizeof(Scalars), hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  return HFSI_OK;
}

static void timer_flush(hfsi_fluid* h) {
  if (h->timer_used == 0) return;
  (void)hipEventSynchronize(h->timer_events[h->timer_used - 1]);
  for (int i = 0; i + 1 < h->timer_used; i += 2) {
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, h->timer_events[i], h->timer_events[i + 1]) == hipSuccess) {
      h->timer_ms += ms;
      h->timer_count += 1;
    }
  }
  h->timer_used = 0;
}

static inline void timer_mark(hfsi_fluid* h, int id, hipStream_t st) {
  if (h->timer_id != id || h->timer_events.empty()) return;
  if (h->timer_used >= (int)h->timer_events.size()) timer_flush(h);
  (void)hipEventRecord(h->timer_events[h->timer_used++], st);
}

// ---------------------------------------------------------------------------
// V-cycle driver
// ---------------------------------------------------------------------------

static inline bool march_ok(const hfsi_fluid* h, int l) {
  const LevelMem& m = h->lv[l];
  return !h->has_vd && m.nz >= 4 && (m.nz % 4) == 0;
}

static inline uint32_t pick_ichunk(uint32_t nx, uint32_t per_plane_blocks) {
  uint32_t c = (nx * per_plane_blocks) / 2048u;
  c = c < 2 ? 2 : (c > 16 ? 16 : c);
  return c > nx ? nx : c;
}

static inline MarchGeo level_march_geo(const LevelMem& m) {
  MarchGeo g0 = march_geo(m.nx, m.ny, m.nz, 1);
  return march_geo(m.nx, m.ny, m.nz, pick_ichunk(m.nx, g0.kblocks * g0.jblocks));
}

// Marching sweep / apply on level l.  pc: coarse iterate of level l + 1 (prolongation).
template <typename C, typename TP, typename TR, typename TO, typename TQ, int MODE, bool DOTS, typename Fin>
static void launch_march(hfsi_fluid* h, int l, int outlet, const TP* p, const TR* rhs, C sign, TO* out, C omega,
                         const float* pc, C scale, const TQ* q, Fin fin, hipStream_t st) {
  const LevelMem& m = h->lv[l];
  MarchArgs<C, TP, TR, TO, TQ> a;
  a.m = level_march_geo(m);
  OpGeo<C> g = geo<C>(h, l, outlet);
  a.flags = m.flags;
  a.diag = g.diag;
  for (int ax = 0; ax < 3; ++ax) {
    a.cl[ax] = g.cl[ax];
    a.ch[ax] = g.ch[ax];
    a.wd[ax] = m.wd[ax];
  }
  a.outlet_add = g.outlet_add;
  a.outlet = outlet;
  a.omega = omega;
  a.rhs_sign = sign;
  a.p = p;
  a.rhs = rhs;
  a.out = out;
  a.pc = pc;
  if (l + 1 < h->L) {
    const LevelMem& c = h->lv[l + 1];
    a.cnx = c.nx; a.cny = c.ny; a.cnz = c.nz; a.csx = c.ny * c.nz; a.csy = c.nz;
  } else {
    a.cnx = a.cny = a.cnz = 1; a.csx = a.csy = 1;
  }
  a.scale = scale;
  a.q = q;
  a.partials = h->partials;
  a.counter = h->counter;
  a.totals = h->totals;
  hipLaunchKernelGGL((k_march<C, TP, TR, TO, TQ, MODE, DOTS>), dim3(march_grid(a.m)), dim3(256), 0, st, a);
  if (DOTS) finish_sums<march_sums<MODE>()>(h, march_grid(a.m), fin, st);
}

// The marching restriction where its columns fill the chip.
static bool march_restrict_pays(const hfsi_fluid* h, int l) { return march_ok(h, l) && h->lv[l].n > kRestrictTileMax; }

// Tile restriction l -> l + 1 (any grid).
template <typename TRes, typename C, typename P, typename R>
static void launch_restrict_tile(hfsi_fluid* h, int l, int outlet, P p, R rhs, hipStream_t st) {
  const OpGeo<C> c = geo<C>(h, l + 1, outlet);
  const uint32_t blocks = restrict_tiles(c.nx, kRestrictI) * restrict_tiles(c.ny, kRestrictJ) * restrict_tiles(c.nz, kRestrictK);
  hipLaunchKernelGGL((k_restrict_tile<TRes, C, P, R, float>), dim3(blocks), dim3(256), 0, st, geo<C>(h, l, outlet), p,
                     rhs, c, h->lv[l + 1].rhs);
}

template <typename C, typename TP, typename TR, typename TRes>
static void launch_march_restrict(hfsi_fluid* h, int l, int outlet, const TP* p, const TR* rhs, C sign,
                                  hipStream_t st) {
  const LevelMem& f = h->lv[l];
  const LevelMem& c = h->lv[l + 1];
  RestrictArgs<C, TP, TR, TRes> a;
  MarchGeo g0 = march_geo(c.nx, c.ny, f.nz, 1);
  a.m = march_geo(c.nx, c.ny, f.nz, pick_ichunk(c.nx, g0.kblocks * g0.jblocks));
  a.fnx = f.nx; a.fny = f.ny; a.fnz = f.nz; a.fsx = f.ny * f.nz; a.fsy = f.nz;
  a.cnx = c.nx; a.cny = c.ny; a.cnz = c.nz; a.csx = c.ny * c.nz; a.csy = c.nz;
  OpGeo<C> g = geo<C>(h, l, outlet);
  a.flags = f.flags;
  a.cflags = c.flags;
  a.diag = g.diag;
  for (int ax = 0; ax < 3; ++ax) {
    a.cl[ax] = g.cl[ax];
    a.ch[ax] = g.ch[ax];
    a.wf[ax] = f.wf[ax];
  }
  a.outlet_add = g.outlet_add;
  a.outlet = outlet;
  a.rhs_sign = sign;
  a.p = p;
  a.rhs = rhs;
  a.out = c.rhs;
  hipLaunchKernelGGL((k_march_restrict<C, TP, TR, TRes>), dim3(march_grid(a.m)), dim3(256), 0, st, a);
}

// Optional fusion of the PCG sums into the last level-0 post-smoothing sweep.
struct FusedDots {
  const void* q;
  Scalars* sc;
  int remove_mean, use_mg;
  bool done;
};

// Level-0 types: T0 storage of p/t at level 0, rhs0 loader R0 (Ld or LdNeg).
// Coarse levels are float storage with compute type C.
template <typename C, typename T0, typename R0>
static int run_vcycle(hfsi_fluid* h, T0* P0, T0* T0buf, R0 rhs0, bool zero_init, int pre, int coarse, int post,
                      int outlet, hipStream_t st, FusedDots* dots = nullptr) {
  using TR0 = typename R0::Storage;
  const int L = h->L;
  const C omega = (C)0.8f;  // f32 kernel argument in the reference
  const C scale = (C)(h->uniform ? 1.0f : 0.7f);
  const C sign0 = (C)R0::kSign;
  OpGeo<C> g0 = geo<C>(h, 0, outlet);
  if (dots) dots->done = false;
  if (L <= 1) {
    const int W = std::max(pre + post, coarse);
    if (!zero_init && (W % 2)) {
      set_error("level-0 smoothing count must be even for a warm start");
      return HFSI_ERR_ARG;
    }
    T0* in = P0;
    for (int m = 1; m <= W; ++m) {
      T0* out = sweep_target(P0, T0buf, W, m);
      if (m == 1 && zero_init)
        hipLaunchKernelGGL((k_jacobi<C, LdZero<C>, R0, T0>), dim3(blocks_for(g0.n)), dim3(kBlock), 0, st, g0,
                           LdZero<C>{}, rhs0, out, omega);
      else
        hipLaunchKernelGGL((k_jacobi<C, Ld<T0, C>, R0, T0>), dim3(blocks_for(g0.n)), dim3(kBlock), 0, st, g0,
                           Ld<T0, C>{in}, rhs0, out, omega);
      in = out;
    }
    HFSI_LAUNCH_CHECK();
    return HFSI_OK;
  }
  if (!zero_init && ((pre + post) % 2)) {
    set_error("V-cycle smoothing count must be even for a warm start");
    return HFSI_ERR_ARG;
  }
  const int W = pre + post;
  const int tail = h->tail_first;  // >= 1
  const bool m0 = march_ok(h, 0);
  // ---- level 0 down
  T0* in0 = P0;
  for (int m = 1; m <= pre; ++m) {
    T0* out = sweep_target(P0, T0buf, W, m);
    const bool from_zero = m == 1 && zero_init;
    if (m0) {
      if (from_zero)
        launch_march<C, T0, TR0, T0, T0, kModeFromZero, false>(h, 0, outlet, (const T0*)nullptr, rhs0.p, sign0, out,
                                                               omega, nullptr, scale, (const T0*)nullptr, FinNone{},
                                                               st);
      else {
        timer_mark(h, HFSI_TIMER_L0_SWEEP, st);
        launch_march<C, T0, TR0, T0, T0, kModeNormal, false>(h, 0, outlet, in0, rhs0.p, sign0, out, omega, nullptr,
                                                             scale, (const T0*)nullptr, FinNone{}, st);
        timer_mark(h, HFSI_TIMER_L0_SWEEP, st);
      }
    } else if (from_zero) {
      hipLaunchKernelGGL((k_jacobi<C, LdZero<C>, R0, T0>), dim3(blocks_for(g0.n)), dim3(kBlock), 0, st, g0,
                         LdZero<C>{}, rhs0, out, omega);
    } else {
      timer_mark(h, HFSI_TIMER_L0_SWEEP, st);
      hipLaunchKernelGGL((k_jacobi<C, Ld<T0, C>, R0, T0>), dim3(blocks_for(g0.n)), dim3(kBlock), 0, st, g0,
                         Ld<T0, C>{in0}, rhs0, out, omega);
      timer_mark(h, HFSI_TIMER_L0_SWEEP, st);
    }
    in0 = out;
  }
  timer_mark(h, HFSI_TIMER_L0_RESTRICT, st);
  if (march_restrict_pays(h, 0))
    launch_march_restrict<C, T0, TR0, T0>(h, 0, outlet, in0, rhs0.p, sign0, st);
  else
    launch_restrict_tile<T0, C>(h, 0, outlet, Ld<T0, C>{in0}, rhs0, st);
  timer_mark(h, HFSI_TIMER_L0_RESTRICT, st);
  // ---- grid-launched coarse levels down
  float* cur[kMaxLevels] = {};
  for (int l = 1; l < tail; ++l) {
    LevelMem& m = h->lv[l];
    OpGeo<C> g = geo<C>(h, l, outlet);
    const bool mk = march_ok(h, l);
    Ld<float, C> R{m.rhs};
    float* in = nullptr;
    for (int s = 1; s <= pre; ++s) {
      float* out = sweep_target(m.p, m.t, W, s);
      if (mk) {
        if (s == 1)
          launch_march<C, float, float, float, float, kModeFromZero, false>(
              h, l, outlet, (const float*)nullptr, m.rhs, (C)1, out, omega, nullptr, scale, (const float*)nullptr,
              FinNone{}, st);
        else
          launch_march<C, float, float, float, float, kModeNormal, false>(h, l, outlet, in, m.rhs, (C)1, out, omega,
                                                                          nullptr, scale, (const float*)nullptr,
                                                                          FinNone{}, st);
      } else if (s == 1) {
        hipLaunchKernelGGL((k_jacobi<C, LdZero<C>, Ld<float, C>, float>), dim3(blocks_for(g.n)), dim3(kBlock), 0,
                           st, g, LdZero<C>{}, R, out, omega);
      } else {
        hipLaunchKernelGGL((k_jacobi<C, Ld<float, C>, Ld<float, C>, float>), dim3(blocks_for(g.n)), dim3(kBlock),
                           0, st, g, Ld<float, C>{in}, R, out, omega);
      }
      in = out;
    }
    cur[l] = in;
    if (march_restrict_pays(h, l))
      launch_march_restrict<C, float, float, float>(h, l, outlet, in, m.rhs, (C)1, st);
    else
      launch_restrict_tile<float, C>(h, l, outlet, Ld<float, C>{in}, R, st);
  }
  // ---- tail: levels tail .. L-1 in one workgroup
  {
    const bool dbl = std::is_same<C, double>::value;
    const void* args = dbl ? h->tail_args_d : h->tail_args_f;
    const uint32_t lds = dbl ? h->tail_lds_bytes_d : h->tail_lds_bytes_f;
    if (lds > 0)
      hipLaunchKernelGGL((k_vcycle_tail_lds<C>), dim3(1), dim3(kTailThreads), lds, st,
                         (const TailArgs<C, float>*)args, dbl ? h->tail_image_d : h->tail_image_f, pre, coarse, post,
                         omega, scale);
    else
      hipLaunchKernelGGL((k_vcycle_tail<C, float>), dim3(1), dim3(kTailThreads), 0, st,
                         (const TailArgs<C, float>*)args, pre, coarse, post, omega, scale);
    cur[tail] = h->lv[tail].p;  // final smoothed value always lands in P
  }
  // ---- up through the grid-launched coarse levels
  for (int l = tail - 1; l >= 1; --l) {
    LevelMem& m = h->lv[l];
    LevelMem& mc = h->lv[l + 1];
    OpGeo<C> g = geo<C>(h, l, outlet);
    const bool mk = march_ok(h, l);
    Ld<float, C> R{m.rhs};
    float* out = sweep_target(m.p, m.t, W, pre + 1);
    if (mk) {
      launch_march<C, float, float, float, float, kModeProlong, false>(h, l, outlet, cur[l], m.rhs, (C)1, out, omega,
                                                                       cur[l + 1], scale, (const float*)nullptr,
                                                                       FinNone{}, st);
    } else {
      LdProlong<float, float, C> PP{cur[l], cur[l + 1], m.flags, mc.nx, mc.ny, mc.nz, mc.ny * mc.nz, mc.nz, scale};
      hipLaunchKernelGGL((k_jacobi<C, LdProlong<float, float, C>, Ld<float, C>, float>), dim3(blocks_for(g.n)),
                         dim3(kBlock), 0, st, g, PP, R, out, omega);
    }
    float* in = out;
    for (int s = pre + 2; s <= W; ++s) {
      out = sweep_target(m.p, m.t, W, s);
      if (mk)
        launch_march<C, float, float, float, float, kModeNormal, false>(h, l, outlet, in, m.rhs, (C)1, out, omega,
                                                                        nullptr, scale, (const float*)nullptr,
                                                                        FinNone{}, st);
      else
        hipLaunchKernelGGL((k_jacobi<C, Ld<float, C>, Ld<float, C>, float>), dim3(blocks_for(g.n)), dim3(kBlock), 0,
                           st, g, Ld<float, C>{in}, R, out, omega);
      in = out;
    }
    cur[l] = in;
  }
  // ---- level 0 up
  {
    LevelMem& mc = h->lv[1];
    T0* out = sweep_target(P0, T0buf, W, pre + 1);
    const bool fuse_last_prolong = dots && m0 && W == pre + 1;
    timer_mark(h, HFSI_TIMER_L0_PROLONG_SWEEP, st);
    if (m0) {
      if (fuse_last_prolong) {
        launch_march<C, T0, TR0, T0, T0, kModeProlong, true>(
            h, 0, outlet, in0, rhs0.p, sign0, out, omega, cur[1], scale, (const T0*)dots->q,
            FinDots5{dots->sc, dots->remove_mean, dots->use_mg}, st);
        dots->done = true;
      } else {
        launch_march<C, T0, TR0, T0, T0, kModeProlong, false>(h, 0, outlet, in0, rhs0.p, sign0, out, omega, cur[1],
                                                              scale, (const T0*)nullptr, FinNone{}, st);
      }
    } else {
      LdProlong<T0, float, C> PP{in0, cur[1], h->lv[0].flags, mc.nx, mc.ny, mc.nz, mc.ny * mc.nz, mc.nz, scale};
      hipLaunchKernelGGL((k_jacobi<C, LdProlong<T0, float, C>, R0, T0>), dim3(blocks_for(g0.n)), dim3(kBlock), 0, st,
                         g0, PP, rhs0, out, omega);
    }
    timer_mark(h, HFSI_TIMER_L0_PROLONG_SWEEP, st);
    T0* in = out;
    for (int s = pre + 2; s <= W; ++s) {
      out = sweep_target(P0, T0buf, W, s);
      const bool last = s == W;
      timer_mark(h, HFSI_TIMER_L0_SWEEP, st);
      if (m0) {
        if (last && dots) {
          launch_march<C, T0, TR0, T0, T0, kModeNormal, true>(h, 0, outlet, in, rhs0.p, sign0, out, omega, nullptr,
                                                             scale, (const T0*)dots->q,
                                                             FinDots5{dots->sc, dots->remove_mean, dots->use_mg}, st);
          dots->done = true;
        } else {
          launch_march<C, T0, TR0, T0, T0, kModeNormal, false>(h, 0, outlet, in, rhs0.p, sign0, out, omega, nullptr,
                                                              scale, (const T0*)nullptr, FinNone{}, st);
        }
      } else {
        hipLaunchKernelGGL((k_jacobi<C, Ld<T0, C>, R0, T0>), dim3(blocks_for(g0.n)), dim3(kBlock), 0, st, g0,
                           Ld<T0, C>{in}, rhs0, out, omega);
      }
      timer_mark(h, HFSI_TIMER_L0_SWEEP, st);
      in = out;
    }
  }
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

// ---------------------------------------------------------------------------
// PCG driver
// ---------------------------------------------------------------------------

// ---------------------------------------------------------------------------
// Mixed-precision V-cycle driver
// ---------------------------------------------------------------------------

static OpGeo<float> mix_geo(const hfsi_fluid* h, int l, int outlet) {
  const MixLevel& m = h->ml[l];
  OpGeo<float> g;
  g.nx = m.nx; g.ny = m.ny; g.nz = m.nz; g.n = m.n; g.sx = m.ny * m.nz; g.sy = m.nz;
  g.flags = m.flags;
  g.fw = nullptr;
  g.diag = nullptr;
  for (int a = 0; a < 3; ++a) {
    g.cl[a] = m.cl[a];
    g.ch[a] = m.ch[a];
    g.wf[a] = m.wf[a];
    g.wd[a] = m.wd[a];
  }
  g.outlet_add = m.outlet_add;
  g.outlet = outlet;
  return g;
}

static MixXfer mix_xfer(const hfsi_fluid* h, int l) {
  MixXfer x;
  for (int a = 0; a < 3; ++a) {
    x.par[a] = h->ml[l].par[a];
    x.pnb[a] = h->ml[l].pnb[a];
    x.pw[a] = h->ml[l].pw[a];
    x.first[a] = h->ml[l + 1].first[a];
    x.cnt[a] = h->ml[l + 1].cnt[a];
  }
  return x;
}

// fp16 storage for the large grid-launched levels; the workgroup tail is float.
static inline bool mix_half(const hfsi_fluid* h, int l) {
  return (l < h->mix_tail_first || h->ML == 1) && h->ml[l].n >= h->mix_half_min_cells;
}

static int write_mix_tail_args(hfsi_fluid* h, int outlet, hipStream_t st) {
  if (h->ML < 2 || h->mix_tail_outlet == outlet) return HFSI_OK;
  MixTailArgs A{};
  A.first = h->mix_tail_first;
  A.last = h->ML - 1;
  A.dense_m = h->mixd_m;
  A.dense_idx = h->mixd_idx;
  A.dense_vol = h->mixd_vol;
  A.dense_inv = h->mixd_inv[outlet ? 1 : 0];
  uint32_t n[kMixMaxLevels] = {};
  for (int l = A.first; l <= A.last; ++l) {
    A.lv[l].g = mix_geo(h, l, outlet);
    A.lv[l].e = (float*)h->ml[l].e;
    A.lv[l].rhs = (float*)h->ml[l].rhs;
    if (l < A.last) A.lv[l].x = mix_xfer(h, l);
    n[l] = A.lv[l].g.n;
  }
  mix_tail_lds_layout(n, A.first, A.last, A.lds_e, A.lds_rhs, A.lds_flags);
  HFSI_CHECK(hipMemcpyAsync(h->mix_tail_args, &A, sizeof(A), hipMemcpyHostToDevice, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  h->mix_tail_outlet = outlet;
  return HFSI_OK;
}

// Fused two-colour sweeps (k_mix_sweep) on grid-launched levels with a second
// iterate buffer (nz even) and at least mix_fused_min_cells cells; one launch
// per colour pass (k_mix_rb) elsewhere.
static inline bool mix_fused(const hfsi_fluid* h, const MixLevel& m) {
  return m.e2 != nullptr && m.n >= h->mix_fused_min_cells;
}

static SweepGeo mix_sweep_geo(const hfsi_fluid* h, const MixLevel& m) {
  SweepGeo sg;
  sg.kblocks = (m.nz + kSwTK - 1) / kSwTK;
  sg.jblocks = (m.ny + kSwTJ - 1) / kSwTJ;
  // planes per workgroup: about mix_sweep_wgs workgroups, 4..64 planes (each chunk recomputes 3 planes), a
  // multiple of kSwChunkAlign (the kernel's march is unrolled by that; one chunk of all planes also works)
  const uint64_t wgs = h->mix_sweep_wgs;
  uint32_t c = (uint32_t)(((uint64_t)m.nx * sg.kblocks * sg.jblocks + wgs / 2) / wgs);
  c = (c + kSwChunkAlign / 2) / kSwChunkAlign * kSwChunkAlign;
  c = c < 4 ? 4 : (c > 64 ? 64 : c);
  sg.ichunk = c > m.nx ? m.nx : c;
  sg.nblocks = sg.kblocks * sg.jblocks * ((m.nx + sg.ichunk - 1) / sg.ichunk);
  return sg;
}

template <typename TE, typename TR>
static void mix_rb_pass(hfsi_fluid* h, int l, int outlet, TE* e, const TR* rhs, const double* rs, int color,
                        bool from_zero, hipStream_t st) {
  const MixLevel& m = h->ml[l];
  const uint32_t npairs = m.nx * m.ny * ((m.nz + 1) / 2);
  OpGeo<float> g = mix_geo(h, l, outlet);
  if (from_zero) {
    hipLaunchKernelGGL((k_mix_rb<TE, TR, true>), dim3(blocks_for(npairs)), dim3(kBlock), 0, st, g, e, rhs, rs, color);
  } else {
    if (l == 0) timer_mark(h, HFSI_TIMER_MIX_RB, st);
    hipLaunchKernelGGL((k_mix_rb<TE, TR, false>), dim3(blocks_for(npairs)), dim3(kBlock), 0, st, g, e, rhs, rs,
                       color);
    if (l == 0) timer_mark(h, HFSI_TIMER_MIX_RB, st);
  }
}

// pre / post smoothing on level l: red then black (pre), black then red
// (post); the first pre-smoothing sweep starts from zero.  The iterate of the
// level is ml[l].cur (the fused sweeps alternate between e and e2).
template <typename TE, typename TR>
static void mix_smooth(hfsi_fluid* h, int l, int outlet, const TR* rhs, const double* rs, int sweeps, bool pre,
                       hipStream_t st) {
  MixLevel& m = h->ml[l];
  const int c0 = pre ? 0 : 1;
  if (mix_fused(h, m)) {
    const SweepGeo sg = mix_sweep_geo(h, m);
    const uint32_t grid = (sg.nblocks + HFSI_NXCD - 1) / HFSI_NXCD * HFSI_NXCD;
    OpGeo<float> g = mix_geo(h, l, outlet);
    for (int s = 0; s < sweeps; ++s) {
      TE* in = (TE*)m.cur;
      TE* out = (TE*)(m.cur == m.e ? m.e2 : m.e);
      if (pre && s == 0) {
        hipLaunchKernelGGL((k_mix_sweep<TE, TR, true>), dim3(grid), dim3(kSwThreads), 0, st, g, in, out, rhs, rs, c0,
                           sg);
      } else {
        if (l == 0) timer_mark(h, HFSI_TIMER_MIX_RB, st);
        hipLaunchKernelGGL((k_mix_sweep<TE, TR, false>), dim3(grid), dim3(kSwThreads), 0, st, g, in, out, rhs, rs,
                           c0, sg);
        if (l == 0) timer_mark(h, HFSI_TIMER_MIX_RB, st);
      }
      m.cur = out;
    }
    return;
  }
  for (int s = 0; s < sweeps; ++s) {
    mix_rb_pass<TE, TR>(h, l, outlet, (TE*)m.cur, rhs, rs, c0, pre && s == 0, st);
    mix_rb_pass<TE, TR>(h, l, outlet, (TE*)m.cur, rhs, rs, 1 - c0, false, st);
  }
}

// Residual of level l (stored at the level's own precision), then its
// volume-weighted restriction into the rhs of level l + 1.
template <typename TE, typename TR, typename TC>
static void mix_restrict(hfsi_fluid* h, int l, int outlet, const TR* rhs, const double* rs, hipStream_t st) {
  const MixLevel& f = h->ml[l];
  const MixLevel& c = h->ml[l + 1];
  TE* e = (TE*)f.cur;
  OpGeo<float> g = mix_geo(h, l, outlet);
  if (f.nz % 2 == 0)
    hipLaunchKernelGGL((k_mix_residual_pairs<TE, TR, TE>), dim3(blocks_for(f.n / 2)), dim3(kBlock), 0, st, g,
                       FastDiv::make(f.nz / 2), FastDiv::make(f.ny), (const TE*)e, rhs, rs, (TE*)f.res);
  else
    hipLaunchKernelGGL((k_mix_residual<TE, TR, TE>), dim3(blocks_for(f.n)), dim3(kBlock), 0, st, g, (const TE*)e,
                       rhs, rs, (TE*)f.res);
  hipLaunchKernelGGL((k_mix_restrict_res<TE, TC>), dim3(blocks_for(c.n)), dim3(kBlock), 0, st, g,
                     FastDiv::make(c.nz), FastDiv::make(c.ny), (const TE*)f.res, mix_xfer(h, l), c.n,
                     (const uint8_t*)c.flags, (TC*)c.rhs);
}

template <typename TF, typename TCo>
static void mix_prolong(hfsi_fluid* h, int l, int outlet, hipStream_t st) {
  const MixLevel& c = h->ml[l + 1];
  const MixLevel& f = h->ml[l];
  TF* ef = (TF*)f.cur;
  hipLaunchKernelGGL((k_mix_prolong<TF, TCo>), dim3(blocks_for(f.n)), dim3(kBlock), 0, st, mix_geo(h, l, outlet),
                     FastDiv::make(f.nz), FastDiv::make(f.ny), ef, mix_xfer(h, l), c.ny, c.nz,
                     (const uint8_t*)c.flags, (const TCo*)c.cur);
}

// Down-leg of level l (smoothing + restriction), with the storage types of l
// and l + 1 resolved at run time.
template <typename TE, typename TR>
static void mix_down(hfsi_fluid* h, int l, int outlet, const TR* rhs, const double* rs, int pre, hipStream_t st) {
  mix_smooth<TE, TR>(h, l, outlet, rhs, rs, pre, true, st);
  if (mix_half(h, l + 1))
    mix_restrict<TE, TR, __half>(h, l, outlet, rhs, rs, st);
  else
    mix_restrict<TE, TR, float>(h, l, outlet, rhs, rs, st);
}

template <typename TE, typename TR>
static void mix_up(hfsi_fluid* h, int l, int outlet, const TR* rhs, const double* rs, int post, hipStream_t st) {
  if (mix_half(h, l + 1))
    mix_prolong<TE, __half>(h, l, outlet, st);
  else
    mix_prolong<TE, float>(h, l, outlet, st);
  mix_smooth<TE, TR>(h, l, outlet, rhs, rs, post, false, st);
}

// One mixed V-cycle on A e = r0 * vin (scaled level operators); leaves the
// level-0 iterate in ml[0].cur (fp16 or float per mix_half(h, 0)).
static int run_mix_vcycle(hfsi_fluid* h, const float* r0, int pre, int coarse, int post, int outlet, hipStream_t st) {
  HFSI_TRY(write_mix_tail_args(h, outlet, st));
  const double* vin = (const double*)((const char*)h->scal + offsetof(Scalars, vin));
  for (int l = 0; l < h->ML; ++l) h->ml[l].cur = h->ml[l].e;
  const int T = h->ML > 1 ? h->mix_tail_first : 1;
  if (h->ML == 1) {
    if (mix_half(h, 0))
      mix_smooth<__half, float>(h, 0, outlet, r0, vin, coarse, true, st);
    else
      mix_smooth<float, float>(h, 0, outlet, r0, vin, coarse, true, st);
    HFSI_LAUNCH_CHECK();
    return HFSI_OK;
  }
  for (int l = 0; l < T; ++l) {
    const bool he = mix_half(h, l);
    if (l == 0) {
      if (he) mix_down<__half, float>(h, 0, outlet, r0, vin, pre, st);
      else mix_down<float, float>(h, 0, outlet, r0, vin, pre, st);
    } else if (he) {
      mix_down<__half, __half>(h, l, outlet, (const __half*)h->ml[l].rhs, nullptr, pre, st);
    } else {
      mix_down<float, float>(h, l, outlet, (const float*)h->ml[l].rhs, nullptr, pre, st);
    }
  }
  hipLaunchKernelGGL(k_mix_tail, dim3(1), dim3(kMixTailThreads), h->mix_tail_lds, st,
                     (const MixTailArgs*)h->mix_tail_args, pre, coarse, post);
  for (int l = T - 1; l >= 0; --l) {
    const bool he = mix_half(h, l);
    if (l == 0) {
      if (he) mix_up<__half, float>(h, 0, outlet, r0, vin, post, st);
      else mix_up<float, float>(h, 0, outlet, r0, vin, post, st);
    } else if (he) {
      mix_up<__half, __half>(h, l, outlet, (const __half*)h->ml[l].rhs, nullptr, post, st);
    } else {
      mix_up<float, float>(h, l, outlet, (const float*)h->ml[l].rhs, nullptr, post, st);
    }
  }
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

// z = M r (mixed V-cycle) with the NS PCG sums of z (FinDots3 / FinDots5).
template <int NS, typename Fin>
static int mix_precondition(hfsi_fluid* h, const float* r, const float* q, float* z, int pre, int coarse, int post,
                            int outlet, Fin fin, hipStream_t st) {
  HFSI_TRY(run_mix_vcycle(h, r, pre, coarse, post, outlet, st));
  OpGeo<double> g64 = geo<double>(h, 0, outlet);
  uint32_t nb = blocks_for(g64.n);
  if (g64.nz % 4 == 0) {
    nb = blocks_for(g64.n / 4);
    const FastDiv fq = FastDiv::make(g64.nz / 4), fy = FastDiv::make(g64.ny);
    if (mix_half(h, 0))
      hipLaunchKernelGGL((k_mix_finish4<NS, __half>), dim3(nb), dim3(kBlock), 0, st, g64, fq, fy,
                         (const __half*)h->ml[0].cur, r, q, z, h->scal, h->partials);
    else
      hipLaunchKernelGGL((k_mix_finish4<NS, float>), dim3(nb), dim3(kBlock), 0, st, g64, fq, fy,
                         (const float*)h->ml[0].cur, r, q, z, h->scal, h->partials);
  } else if (mix_half(h, 0)) {
    hipLaunchKernelGGL((k_mix_finish<NS, __half>), dim3(nb), dim3(kBlock), 0, st, g64, (const __half*)h->ml[0].cur,
                       r, q, z, h->scal, h->partials);
  } else {
    hipLaunchKernelGGL((k_mix_finish<NS, float>), dim3(nb), dim3(kBlock), 0, st, g64, (const float*)h->ml[0].cur, r,
                       q, z, h->scal, h->partials);
  }
  finish_sums<NS>(h, nb, fin, st);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

template <typename C, typename TV>
struct Vecs {
  TV *r, *d, *q, *z, *t;
};

template <typename C, typename TV>
static Vecs<C, TV> vecs(hfsi_fluid* h);
template <>
Vecs<double, double> vecs<double, double>(hfsi_fluid* h) {
  return {h->r64, h->d64, h->q64, h->z64, h->t64};
}
template <>
Vecs<float, float> vecs<float, float>(hfsi_fluid* h) {
  return {h->r32, h->d32, h->q32, h->z32, h->t32};
}

template <typename C, typename TV>
static int precondition(hfsi_fluid* h, bool use_mg, int pre, int coarse, int post, int outlet, hipStream_t st,
                        FusedDots* dots = nullptr) {
  Vecs<C, TV> v = vecs<C, TV>(h);
  if (dots) dots->done = false;
  if (use_mg)
    return run_vcycle<C, TV, LdNeg<TV, C>>(h, v.z, v.t, LdNeg<TV, C>{v.r}, true, pre, coarse, post, outlet, st,
                                           dots);
  OpGeo<C> g = geo<C>(h, 0, outlet);
  hipLaunchKernelGGL((k_jacobi_precond<C, TV, TV>), dim3(blocks_for(g.n)), dim3(kBlock), 0, st, g, v.r, v.z);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

template <typename C, typename TV>
static int solve_cg(hfsi_fluid* h, const float* div, const float* src, const double* iface, double* x,
                    const hfsi_cg_options& o, hfsi_cg_stats& S, hipStream_t st, bool mixed = false) {
  Vecs<C, TV> v = vecs<C, TV>(h);
  const int outlet = o.outlet_zmin ? 1 : 0;
  // interface couplings: the operator is the stencil plus the coupling list, so q = A d and
  // the true residual take an unfused stencil launch followed by the coupling pass
  const bool coupled = h->cpl_n > 0;
  const int rm = o.remove_mean ? 1 : 0;
  OpGeo<C> g = geo<C>(h, 0, outlet);
  OpGeo<double> g64 = geo<double>(h, 0, outlet);
  Scalars* sc = h->scal;
  const bool exact_checks = o.true_residual != 0;
  const int check_every = o.check_interval > 0 ? o.check_interval : 16;
  const int restart_every = o.restart_interval;
  const int max_it = std::max(1, o.max_iterations);
  const double tol = std::max(0.0, o.tolerance);
  std::memset(&S, 0, sizeof(S));
  S.initial_relative_residual = INFINITY;
  S.relative_residual = INFINITY;
  S.true_relative_residual = -1.0;

  // reset device scalars (keep the free volume of the current masks)
  {
    Scalars init{};
    HFSI_CHECK(hipMemcpyAsync(h->host_scal, h->scal, sizeof(Scalars), hipMemcpyDeviceToHost, st));
    HFSI_CHECK(hipStreamSynchronize(st));
    init.free_vol = h->host_scal->free_vol;
    *h->host_scal = init;
    HFSI_CHECK(hipMemcpyAsync(h->scal, h->host_scal, sizeof(Scalars), hipMemcpyHostToDevice, st));
  }
  // ---- right-hand side b = -(rhs0 - mean)
  const float scale = (float)o.rhs_scale;
  HFSI_TRY(launch_pointwise(h, 0, OpRhsNonFree{div, src, iface, h->b, scale}, st));
  HFSI_TRY(launch_sums<1>(h, g64, OpRhs{div, src, iface, h->b, scale, h->lv[0].flags}, FinBMean{sc, rm}, st));
  if (rm) S.mean_projection_count += 1;
  HFSI_TRY(launch_sums<1>(h, g64, OpBFinal{h->b, sc}, FinBNorm{sc}, st));
  HFSI_TRY(sync_scalars(h, st));
  const double b_norm = std::sqrt(std::max(h->host_scal->bnorm2, 0.0));
  S.b_norm = b_norm;
  if (!(b_norm > 1.0e-30)) {
    HFSI_TRY(launch_pointwise(h, 0, OpFill<double>{x, 0.0}, st));
    S.initial_relative_residual = 0.0;
    S.relative_residual = 0.0;
    S.true_relative_residual = 0.0;
    S.converged = 1;
    return HFSI_OK;
  }

  auto true_residual = [&](bool count_projection) -> int {
    hipLaunchKernelGGL((k_true_residual<TV>), dim3(blocks_for(g64.n)), dim3(kBlock), 0, st, g64, x, h->b, v.r,
                       h->partials);
    if (coupled) {
      HFSI_LAUNCH_CHECK();
      HFSI_TRY((launch_couple<double, TV>(h, x, v.r, -1.0, st)));
      HFSI_TRY(launch_sums<2>(h, g64, OpResidualSums<TV>{v.r}, FinMeanR{sc, rm}, st));
    } else {
      finish_sums<2>(h, blocks_for(g64.n), FinMeanR{sc, rm}, st);
    }
    HFSI_LAUNCH_CHECK();
    if (rm) {
      HFSI_TRY(launch_sums<1>(h, g64, OpSubMeans<TV>{nullptr, v.r, sc}, FinRR{sc}, st));
      HFSI_TRY(launch_pointwise(h, 0, OpZeroNonFree<TV>{nullptr, v.r}, st));
      if (count_projection) S.mean_projection_count += 1;
    }
    return HFSI_OK;
  };

  // ---- initial residual
  HFSI_TRY(true_residual(true));
  HFSI_TRY(sync_scalars(h, st));
  S.host_residual_checks += 1;
  double rel = std::sqrt(std::max(h->host_scal->rr, 0.0)) / b_norm;
  S.initial_relative_residual = rel;
  S.relative_residual = rel;
  if (rel * b_norm <= tol * b_norm) {
    S.converged = 1;
    return HFSI_OK;
  }
  bool use_mg = h->L > 1 && !o.interface_active &&
                (o.preconditioner == HFSI_PRECOND_MG || o.preconditioner == HFSI_PRECOND_MG_LIGHT ||
                 (o.preconditioner == HFSI_PRECOND_AUTO && !h->uniform));
  const bool light = o.preconditioner == HFSI_PRECOND_MG_LIGHT;
  const int pre = light ? 1 : 2, coarse = light ? 12 : 24, post = light ? 1 : 2;
  // mixed V-cycle: float32 CG vectors, no velocity-Dirichlet or interface terms
  bool use_mix = mixed && use_mg && std::is_same<TV, float>::value && h->ML >= 1 && !h->has_vd && !h->has_diag &&
                 h->cpl_n == 0;

  // coarsest mixed level: the float64 dense solve when it is set up (0), else
  // RB-GS sweeps (4, 8 and 24 sweeps give the same iteration counts)
  const int mix_coarse = h->mixd_m > 0 ? 0 : (light ? 4 : 8);
  const double kappa = h->mix_kappa;
  const int lag = std::min(std::max(0, o.monitor_lag), kMonRing - 1);
  auto mix_scale = [&]() -> int {
    hipLaunchKernelGGL(k_mix_scale_from_rr, dim3(1), dim3(64), 0, st, sc, kappa);
    HFSI_LAUNCH_CHECK();
    return HFSI_OK;
  };

  auto precond_and_rz = [&](bool project) -> int {
    if (use_mix) {
      HFSI_TRY(mix_scale());
      HFSI_TRY((mix_precondition<3>(h, (const float*)v.r, (const float*)v.q, (float*)v.z, pre, mix_coarse, post,
                                    outlet, FinDots3{sc, project ? rm : 0}, st)));
      S.vcycles += 1;
      if (project && rm) S.mean_projection_count += 1;
      return HFSI_OK;
    }
    HFSI_TRY((precondition<C, TV>(h, use_mg, pre, coarse, post, outlet, st)));
    if (use_mg) S.vcycles += 1;
    HFSI_TRY(launch_sums<3>(h, g64, OpDots3<TV, TV>{v.r, v.z}, FinDots3{sc, project ? rm : 0}, st));
    if (project && rm) S.mean_projection_count += 1;
    return HFSI_OK;
  };

  HFSI_TRY(precond_and_rz(true));
  HFSI_TRY(sync_scalars(h, st));
  double rz = h->host_scal->rz;
  if (!std::isfinite(rz) || std::fabs(rz) <= 1.0e-300) {
    use_mg = false;
    use_mix = false;
    HFSI_TRY(precond_and_rz(false));
    HFSI_TRY(sync_scalars(h, st));
    rz = h->host_scal->rz;
  }
  S.used_multigrid = use_mix ? 2 : (use_mg ? 1 : 0);
  if (!std::isfinite(rz) || rz <= 0.0) {
    S.breakdown_kind = HFSI_BREAKDOWN_INITIAL_DOT;
    return HFSI_OK;
  }
  HFSI_TRY(launch_cgdir<TV>(h, v.z, v.d, sc, rm, 1, st));

  // Convergence monitor (mixed solve, monitor_lag = L > 0): after each update of
  // x the float64 true residual norm of x (mean-free, not stored) goes to a pinned
  // ring slot.  At the end of iteration it -- its V-cycle already queued, so the
  // device stays busy -- the host reads the value of iteration it - L + 1: with
  // L = 1 the solve stops at the first iterate whose true residual meets the
  // tolerance; with L > 1 a hit forces a check at the next iteration.
  const bool monitor = use_mix && lag > 0 && h->mon_ring != nullptr;
  bool monitor_pending = false;
  int it = 0;
  while (it < max_it) {
    ++it;
    timer_mark(h, HFSI_TIMER_SPMV_DOT, st);
    if (coupled) {
      hipLaunchKernelGGL((k_apply<C, TV, TV>), dim3(blocks_for(g.n)), dim3(kBlock), 0, st, g, v.d, v.q);
      HFSI_LAUNCH_CHECK();
      HFSI_TRY((launch_couple<TV, TV>(h, v.d, v.q, 1.0, st)));
      HFSI_TRY(launch_sums<1>(h, g64, OpDot<TV, TV>{v.d, v.q}, FinDad{sc}, st));
    } else if (use_mix) {
      // q = A d with float64 arithmetic on the float32 d: for smooth d the stencil
      // sum den d - sum c d_nb cancels to a small fraction of den d, and float32
      // arithmetic would leave q -- and through r -= alpha q the recursive residual --
      // with errors that slow the convergence of the true residual (256^3 graded
      // sphere case: 15 iterations to 1e-8 against 11 with r recomputed each time)
      if (march_ok(h, 0))
        launch_march<double, TV, TV, TV, TV, kModeApply, true>(h, 0, outlet, v.d, (const TV*)nullptr, 1.0, v.q, 0.0,
                                                               nullptr, 0.0, (const TV*)nullptr, FinDad{sc}, st);
      else
        hipLaunchKernelGGL((k_spmv_dot<double, TV, TV>), dim3(blocks_for(g64.n)), dim3(kBlock), 0, st, g64, v.d, v.q,
                           h->partials);
    } else if (march_ok(h, 0)) {
      launch_march<C, TV, TV, TV, TV, kModeApply, true>(h, 0, outlet, v.d, (const TV*)nullptr, (C)1, v.q, (C)0,
                                                        nullptr, (C)0, (const TV*)nullptr, FinDad{sc}, st);
    } else {
      hipLaunchKernelGGL((k_spmv_dot<C, TV, TV>), dim3(blocks_for(g.n)), dim3(kBlock), 0, st, g, v.d, v.q,
                         h->partials);
    }
    timer_mark(h, HFSI_TIMER_SPMV_DOT, st);
    if (!coupled && !march_ok(h, 0)) finish_sums<1>(h, blocks_for(use_mix ? g64.n : g.n), FinDad{sc}, st);
    HFSI_LAUNCH_CHECK();
    const bool monitor_hit = monitor_pending;
    monitor_pending = false;
    if (use_mix) {
      timer_mark(h, HFSI_TIMER_CG_UPDATE, st);
      // (one cell per thread: a four-cell form with two 16-byte stores of x per thread measured slower)
      const uint32_t nbu = blocks_for(g64.n);
      hipLaunchKernelGGL(k_cg_update_rr, dim3(nbu), dim3(kBlock), 0, st, g64, x, (const float*)v.d, (float*)v.r,
                         (const float*)v.q, sc, h->partials);
      timer_mark(h, HFSI_TIMER_CG_UPDATE, st);
      finish_sums<1>(h, nbu, FinVScale{sc, kappa}, st);
      if (monitor) {
        const FinTrueMonitor fin{sc, rm, h->mon_ring + (it % kMonRing)};
        if (march_ok(h, 0)) {
          launch_march<double, double, double, double, double, kModeResidual, true>(
              h, 0, outlet, x, h->b, 1.0, (double*)nullptr, 0.0, nullptr, 0.0, (const double*)nullptr, fin, st);
        } else {
          hipLaunchKernelGGL((k_true_residual<float>), dim3(blocks_for(g64.n)), dim3(kBlock), 0, st, g64, x, h->b,
                             (float*)nullptr, h->partials);
          finish_sums<2>(h, blocks_for(g64.n), fin, st);
        }
        HFSI_CHECK(hipEventRecord(h->mon_events[it % kMonRing], st));
      }
      HFSI_LAUNCH_CHECK();
    } else {
      HFSI_TRY(launch_pointwise(h, 0, OpCgUpdate<TV, TV, TV>{x, v.d, v.r, v.q, sc}, st));
    }
    const bool project = rm && (it % 16 == 0);
    const bool check = (it % check_every == 0) || it == max_it || monitor_hit;
    if (project) {
      HFSI_TRY(launch_sums<2>(h, g64, OpSumsXR<TV>{x, v.r}, FinMeansXR{sc}, st));
      HFSI_TRY(launch_sums<1>(h, g64, OpSubMeans<TV>{x, v.r, sc}, FinRR{sc}, st));
      HFSI_TRY(launch_pointwise(h, 0, OpZeroNonFree<TV>{x, v.r}, st));
      S.mean_projection_count += 2;
    }
    S.iterations = it;
    if (check) {
      if (exact_checks) {
        HFSI_TRY(true_residual(true));
        S.true_residual_replacements += 1;
        if (use_mix) HFSI_TRY(mix_scale());
      } else if (!project) {
        HFSI_TRY(launch_sums<1>(h, g64, OpDot<TV, TV>{v.r, v.r}, FinRR{sc}, st));
      }
      HFSI_TRY(sync_scalars(h, st));
      S.host_residual_checks += 1;
      rel = std::sqrt(std::max(h->host_scal->rr, 0.0)) / b_norm;
      S.relative_residual = rel;
      if (rel <= tol) {
        S.converged = 1;
        break;
      }
      const int code = h->host_scal->code;
      bool restart = false;
      if (code != 0) {
        S.breakdown_dAd = h->host_scal->code_dAd;
        if (it >= max_it) {
          S.breakdown_kind = HFSI_BREAKDOWN_DEVICE_SCALAR;
          break;
        }
        restart = true;
      } else if (it < max_it && restart_every > 0 && it % restart_every == 0) {
        restart = true;
      }
      if (restart) {
        HFSI_TRY(true_residual(true));
        HFSI_TRY(sync_scalars(h, st));
        S.host_residual_checks += 1;
        rel = std::sqrt(std::max(h->host_scal->rr, 0.0)) / b_norm;
        S.relative_residual = rel;
        if (rel <= tol) {
          S.converged = 1;
          break;
        }
        HFSI_TRY(precond_and_rz(true));
        HFSI_TRY(sync_scalars(h, st));
        rz = h->host_scal->rz;
        if (std::isfinite(rz) && rz > 0.0) {
          HFSI_TRY(launch_cgdir<TV>(h, v.z, v.d, sc, rm, 1, st));
          Scalars fix = *h->host_scal;
          fix.code = 0;
          fix.code_dAd = 0.0;
          *h->host_scal = fix;
          HFSI_CHECK(hipMemcpyAsync(h->scal, h->host_scal, sizeof(Scalars), hipMemcpyHostToDevice, st));
          S.restart_count += 1;
          continue;
        }
        S.breakdown_kind = code != 0 ? HFSI_BREAKDOWN_DEVICE_SCALAR : HFSI_BREAKDOWN_RESTART_DOT;
        break;
      }
    }
    FusedDots fd{v.q, sc, rm, use_mg ? 1 : 0, false};
    if (use_mix) {
      HFSI_TRY((mix_precondition<5>(h, (const float*)v.r, (const float*)v.q, (float*)v.z, pre, mix_coarse, post,
                                    outlet, FinDots5{sc, rm, 1}, st)));
      fd.done = true;
    } else {
      HFSI_TRY((precondition<C, TV>(h, use_mg, pre, coarse, post, outlet, st, &fd)));
    }
    if (use_mg) S.vcycles += 1;
    if (rm) S.mean_projection_count += 1;
    if (!fd.done)
      HFSI_TRY(launch_sums<5>(h, g64, OpDots5<TV, TV, TV>{v.r, v.z, v.q}, FinDots5{sc, rm, use_mg ? 1 : 0}, st));
    HFSI_TRY(launch_cgdir<TV>(h, v.z, v.d, sc, rm, 0, st));
    if (monitor && it >= lag) {
      const int m = it - lag + 1;
      HFSI_CHECK(hipEventSynchronize(h->mon_events[m % kMonRing]));
      const double rel_m = std::sqrt(std::max(h->mon_ring[m % kMonRing], 0.0)) / b_norm;
      if (rel_m <= tol) {
        if (m == it) {
          // x is the iterate the monitor measured; the queued V-cycle does not touch it
          S.relative_residual = rel_m;
          S.converged = 1;
          break;
        }
        monitor_pending = true;
      }
    }
  }
  HFSI_TRY(sync_scalars(h, st));
  S.breakdown_code = h->host_scal->code;
  if (S.breakdown_code != 0 && S.breakdown_dAd == 0.0) S.breakdown_dAd = h->host_scal->code_dAd;
  if (o.true_residual_at_exit) {
    // float64 certificate ||b - A x||_V / ||b||_V (r is overwritten: the solve is over)
    HFSI_TRY(true_residual(false));
    HFSI_TRY(sync_scalars(h, st));
    double rr = h->host_scal->rr;
    S.true_relative_residual = std::sqrt(std::max(rr, 0.0)) / b_norm;
  }
  return HFSI_OK;
}

template <typename C>
static int write_tail_args(hfsi_fluid* h, void* dst, hipStream_t st) {
  TailArgs<C, float> A{};
  A.first = h->tail_first;
  A.last = h->L - 1;
  for (int l = 1; l < h->L; ++l) {
    A.lv[l].g = geo<C>(h, l, 0);
    A.lv[l].p = h->lv[l].p;
    A.lv[l].t = h->lv[l].t;
    A.lv[l].rhs = h->lv[l].rhs;
  }
  // LDS plan: the image (per level flags and the per-axis coefficient and width arrays), the prolongation
  // scratch, then per level p / t / rhs, all 16-byte aligned
  {
    auto al = [](uint32_t v) { return (v + 15u) & ~15u; };
    uint32_t off = 0;
    A.plan.off_image = off;
    for (int l = A.first; l <= A.last && l >= 1; ++l) {
      const LevelMem& m = h->lv[l];
      A.plan.off_flags[l] = off;
      off = al(off + m.n);
      const uint32_t len[3] = {m.nx, m.ny, m.nz};
      for (int a = 0; a < 3; ++a) {
        A.plan.off_cl[l][a] = off;
        off = al(off + (uint32_t)sizeof(C) * len[a]);
        A.plan.off_ch[l][a] = off;
        off = al(off + (uint32_t)sizeof(C) * len[a]);
        A.plan.off_wf[l][a] = off;
        off = al(off + 4 * len[a]);
      }
    }
    A.plan.image_bytes = off;
    A.plan.off_work = off;
    if (A.first < A.last) off = al(off + (uint32_t)sizeof(C) * h->lv[A.first].n);
    for (int l = A.first; l <= A.last && l >= 1; ++l) {
      A.plan.off_p[l] = off;
      off = al(off + 4 * h->lv[l].n);
      A.plan.off_t[l] = off;
      off = al(off + 4 * h->lv[l].n);
      A.plan.off_rhs[l] = off;
      off = al(off + 4 * h->lv[l].n);
    }
    A.plan.bytes = (h->L > 1 && off <= kTailLdsMax && h->lv[A.first].n < 65536) ? off : 0;
  }
  if (std::is_same<C, double>::value)
    h->tail_lds_bytes_d = A.plan.bytes;
  else
    h->tail_lds_bytes_f = A.plan.bytes;
  // the outlet flag is per solve: the tail reads outlet from lv[].g.outlet,
  // written below for both values by the solve entry (see set_tail_outlet)
  HFSI_CHECK(hipMemcpyAsync(dst, &A, sizeof(A), hipMemcpyHostToDevice, st));
  if (A.plan.bytes > 0) {
    unsigned char*& image = std::is_same<C, double>::value ? h->tail_image_d : h->tail_image_f;
    if (!image) HFSI_TRY(dalloc(h, &image, A.plan.image_bytes));  // the shapes never change
    hipLaunchKernelGGL(k_tail_pack<C>, dim3(1), dim3(kTailThreads), 0, st, (const TailArgs<C, float>*)dst, image);
    HFSI_LAUNCH_CHECK();
  }
  HFSI_CHECK(hipStreamSynchronize(st));
  return HFSI_OK;
}

// The tail geometry carries the outlet switch; refresh it when it changes (the copies and their
// synchronisation run only then: a run of solves with one outlet setting does neither).
static int set_tail_outlet(hfsi_fluid* h, int outlet, hipStream_t st) {
  if (h->tail_outlet == outlet) return HFSI_OK;
  using TAd = TailArgs<double, float>;
  using TLd = TailLevel<double, float>;
  using TAf = TailArgs<float, float>;
  using TLf = TailLevel<float, float>;
  using OGd = OpGeo<double>;
  using OGf = OpGeo<float>;
  for (int l = 1; l < h->L; ++l) {
    size_t off_d = offsetof(TAd, lv) + l * sizeof(TLd) + offsetof(TLd, g) + offsetof(OGd, outlet);
    size_t off_f = offsetof(TAf, lv) + l * sizeof(TLf) + offsetof(TLf, g) + offsetof(OGf, outlet);
    HFSI_CHECK(hipMemcpyAsync((char*)h->tail_args_d + off_d, &outlet, sizeof(int), hipMemcpyHostToDevice, st));
    HFSI_CHECK(hipMemcpyAsync((char*)h->tail_args_f + off_f, &outlet, sizeof(int), hipMemcpyHostToDevice, st));
  }
  HFSI_CHECK(hipStreamSynchronize(st));
  h->tail_outlet = outlet;
  return HFSI_OK;
}

}  // namespace hfsi

using namespace hfsi;

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" {

int hfsi_version(void) { return 1; }

const char* hfsi_last_error(void) { return g_last_error.c_str(); }

int hfsi_device_ok(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return 0;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, 0) != hipSuccess) return 0;
  return std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
}

// Semi-coarsened hierarchy of the mixed V-cycle from the level-0 float widths
// and float64 coefficients of the main operator.  With T_l = 2^l h_min (h_min:
// smallest level-0 width over all axes), along each axis cells i and i + 1 of
// level l merge when w_i + w_{i+1} <= 3 T_l, or always once the level's
// largest width is <= 2.5 T_l; coarsening stops when an axis has <= 3 cells or
// no pair merges.  On uniform grids this is the reference's 2:1 hierarchy.
static int build_mix_hierarchy(hfsi_fluid* h, const std::vector<float> wf0[3], const std::vector<double> cl0[3],
                               const std::vector<double> ch0[3]) {
  double hmin0 = 1e300;
  for (int a = 0; a < 3; ++a)
    for (float w : wf0[a]) hmin0 = std::min(hmin0, (double)w);
  if (!(hmin0 > 0.0)) {
    set_error("hfsi_fluid_create: non-positive cell width");
    return HFSI_ERR_ARG;
  }
  const double kappa = 1.0 / (hmin0 * hmin0);
  h->mix_kappa = kappa;
  struct HostLevel {
    std::vector<double> w[3], ctr[3];
    std::vector<int32_t> par[3], first[3], cnt[3];
  };
  std::vector<HostLevel> H(1);
  for (int a = 0; a < 3; ++a) H[0].w[a].assign(wf0[a].begin(), wf0[a].end());
  auto centres = [](HostLevel& L) {
    for (int a = 0; a < 3; ++a) {
      L.ctr[a].resize(L.w[a].size());
      double face = 0.0;
      for (size_t i = 0; i < L.w[a].size(); ++i) {
        L.ctr[a][i] = face + 0.5 * L.w[a][i];
        face += L.w[a][i];
      }
    }
  };
  centres(H[0]);
  while ((int)H.size() < kMixMaxLevels) {
    HostLevel& F = H.back();
    size_t mn = std::min(F.w[0].size(), std::min(F.w[1].size(), F.w[2].size()));
    if (mn <= 3) break;
    // nominal width of this level: the level-0 minimum doubled per level (an odd
    // leftover cell narrower than that does not hold the other pairs back)
    const double hmin = hmin0 * std::ldexp(1.0, (int)H.size() - 1);
    double hmax = 0.0;
    for (int a = 0; a < 3; ++a)
      for (double w : F.w[a]) hmax = std::max(hmax, w);
    // once every width is within kMixFullRatio of the nominal width, plain 2:1 coarsening
    const bool full = hmax <= kMixFullRatio * hmin;
    HostLevel Cn;
    bool any = false;
    for (int a = 0; a < 3; ++a) {
      const size_t n = F.w[a].size();
      F.par[a].assign(n, 0);
      for (size_t i = 0; i < n;) {
        const int32_t ci = (int32_t)Cn.w[a].size();
        Cn.first[a].push_back((int32_t)i);
        if (i + 1 < n && (full || F.w[a][i] + F.w[a][i + 1] <= kMixMergeRatio * hmin)) {
          Cn.w[a].push_back(F.w[a][i] + F.w[a][i + 1]);
          Cn.cnt[a].push_back(2);
          F.par[a][i] = F.par[a][i + 1] = ci;
          i += 2;
          any = true;
        } else {
          Cn.w[a].push_back(F.w[a][i]);
          Cn.cnt[a].push_back(1);
          F.par[a][i] = ci;
          i += 1;
        }
      }
    }
    if (!any) {
      for (int a = 0; a < 3; ++a) F.par[a].clear();
      break;
    }
    centres(Cn);
    H.push_back(std::move(Cn));
  }
  const int ML = (int)H.size();
  h->ML = ML;
  // mixed tail: the first level (>= 1) of at most kMixTailCells cells from which every coarser level
  // fits the tail kernel's LDS together (its iterates, right-hand sides and flags)
  h->mix_tail_first = ML > 1 ? ML - 1 : 0;
  h->mix_tail_lds = 0;
  if (ML > 1) {
    int dev = 0, max_lds = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) {
      set_error("hfsi_fluid_create: cannot query the device's LDS size");
      return HFSI_ERR_HIP;
    }
    const uint32_t budget = (uint32_t)max_lds > kMixTailStaticLds ? (uint32_t)max_lds - kMixTailStaticLds : 0u;
    uint32_t n[kMixMaxLevels] = {};
    for (int l = 1; l < ML; ++l) n[l] = (uint32_t)(H[l].w[0].size() * H[l].w[1].size() * H[l].w[2].size());
    for (int l = 1; l < ML; ++l) {
      if (n[l] <= kMixTailCells && mix_tail_lds_layout(n, l, ML - 1) <= budget) {
        h->mix_tail_first = l;
        break;
      }
    }
    h->mix_tail_lds = mix_tail_lds_layout(n, h->mix_tail_first, ML - 1);
    if (h->mix_tail_lds > budget ||
        hipFuncSetAttribute((const void*)k_mix_tail, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)h->mix_tail_lds) != hipSuccess) {
      set_error("hfsi_fluid_create: the coarsest multigrid levels do not fit the tail kernel's LDS");
      return HFSI_ERR_HIP;
    }
  }
  int rc = HFSI_OK;
  for (int l = 0; l < ML && rc == HFSI_OK; ++l) {
    HostLevel& L = H[l];
    MixLevel& m = h->ml[l];
    m.nx = (uint32_t)L.w[0].size();
    m.ny = (uint32_t)L.w[1].size();
    m.nz = (uint32_t)L.w[2].size();
    m.n = m.nx * m.ny * m.nz;
    if (l == 0) {
      m.flags = h->lv[0].flags;
    } else {
      rc |= dalloc(h, &m.flags, m.n);
      rc |= dalloc(h, (float**)&m.rhs, m.n);
    }
    rc |= dalloc(h, (float**)&m.e, m.n);
    m.cur = m.e;
    if (l + 1 < ML && (l < h->mix_tail_first || ML == 1)) rc |= dalloc(h, (float**)&m.res, m.n);
    if ((l < h->mix_tail_first || ML == 1) && m.nz % 2 == 0) rc |= dalloc(h, (float**)&m.e2, m.n);
    for (int a = 0; a < 3 && rc == HFSI_OK; ++a) {
      const size_t n = L.w[a].size();
      std::vector<float> cl(n, 0.0f), ch(n, 0.0f), wf(n);
      std::vector<double> wd(n);
      for (size_t i = 0; i < n; ++i) {
        wf[i] = (float)L.w[a][i];
        wd[i] = L.w[a][i];
        if (l == 0) {
          cl[i] = (float)(cl0[a][i] / kappa);
          ch[i] = (float)(ch0[a][i] / kappa);
        } else {
          if (i > 0) cl[i] = (float)(1.0 / (L.w[a][i] * (L.ctr[a][i] - L.ctr[a][i - 1])) / kappa);
          if (i + 1 < n) ch[i] = (float)(1.0 / (L.w[a][i] * (L.ctr[a][i + 1] - L.ctr[a][i])) / kappa);
        }
      }
      if (a == 2) m.outlet_add = (float)(2.0 / (L.w[2][0] * L.w[2][0]) / kappa);
      if (l == ML - 1 && ML > 1) {
        h->mixd_cl[a] = cl;
        h->mixd_ch[a] = ch;
        h->mixd_wf[a] = wf;
        if (a == 2) h->mixd_outlet_add = m.outlet_add;
      }
      rc |= dalloc(h, &m.cl[a], n);
      rc |= dalloc(h, &m.ch[a], n);
      rc |= dalloc(h, &m.wf[a], n);
      rc |= dalloc(h, &m.wd[a], n);
      if (rc != HFSI_OK) break;
      (void)hipMemcpy(m.cl[a], cl.data(), n * sizeof(float), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.ch[a], ch.data(), n * sizeof(float), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.wf[a], wf.data(), n * sizeof(float), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.wd[a], wd.data(), n * sizeof(double), hipMemcpyHostToDevice);
      if (l + 1 < ML) {
        // interpolation partner: the coarse neighbour on the side of the fine centre
        const HostLevel& Cn = H[l + 1];
        const int32_t cn = (int32_t)Cn.w[a].size();
        std::vector<int32_t> pnb(n);
        std::vector<float> pw(n);
        for (size_t i = 0; i < n; ++i) {
          const int32_t I = L.par[a][i];
          const double x = L.ctr[a][i], X = Cn.ctr[a][I];
          int32_t nb = I;
          double w = 1.0;
          if (std::fabs(x - X) > 1.0e-9 * L.w[a][i]) {
            const int32_t cand = x < X ? I - 1 : I + 1;
            if (cand >= 0 && cand < cn) {
              nb = cand;
              const double Xn = Cn.ctr[a][cand];
              w = (Xn - x) / (Xn - X);
            }
          }
          pnb[i] = nb;
          pw[i] = (float)w;
        }
        rc |= dalloc(h, &m.par[a], n);
        rc |= dalloc(h, &m.pnb[a], n);
        rc |= dalloc(h, &m.pw[a], n);
        if (rc != HFSI_OK) break;
        (void)hipMemcpy(m.par[a], L.par[a].data(), n * sizeof(int32_t), hipMemcpyHostToDevice);
        (void)hipMemcpy(m.pnb[a], pnb.data(), n * sizeof(int32_t), hipMemcpyHostToDevice);
        (void)hipMemcpy(m.pw[a], pw.data(), n * sizeof(float), hipMemcpyHostToDevice);
      }
      if (l > 0) {
        rc |= dalloc(h, &m.first[a], n);
        rc |= dalloc(h, &m.cnt[a], n);
        if (rc != HFSI_OK) break;
        (void)hipMemcpy(m.first[a], L.first[a].data(), n * sizeof(int32_t), hipMemcpyHostToDevice);
        (void)hipMemcpy(m.cnt[a], L.cnt[a].data(), n * sizeof(int32_t), hipMemcpyHostToDevice);
      }
    }
  }
  if (rc == HFSI_OK && ML > 1) rc |= dalloc(h, (char**)&h->mix_tail_args, sizeof(MixTailArgs));
  if (rc == HFSI_OK && ML > 1 && h->ml[ML - 1].n <= (uint32_t)kMixDenseMax) {
    rc |= dalloc(h, &h->mixd_idx, (size_t)kMixDenseMax);
    rc |= dalloc(h, &h->mixd_vol, (size_t)kMixDenseMax);
    rc |= dalloc(h, &h->mixd_inv[0], (size_t)kMixDenseMax * kMixDenseMax);
    rc |= dalloc(h, &h->mixd_inv[1], (size_t)kMixDenseMax * kMixDenseMax);
  }
  return rc;
}

// Inverse (row-major, float64) of the V-weighted operator S = V L of the
// coarsest mixed level over its free cells.  S is symmetric positive
// semidefinite; on every connected set of free cells without a z-min outlet
// row it has the constants as null space, shifted out by adding
// alpha 1 1^T (alpha = mean diagonal of the set / its size), which leaves
// the solution of a consistent right-hand side unchanged (the mean-free
// one).  Cholesky factorisation, then the inverse column by column.
static bool mix_dense_inverse(const hfsi_fluid* h, const std::vector<uint8_t>& fl, const std::vector<int32_t>& idx,
                              int outlet, std::vector<double>& inv) {
  const MixLevel& m = h->ml[h->ML - 1];
  const int nfree = (int)idx.size();
  std::vector<int32_t> pos(m.n, -1);
  for (int t = 0; t < nfree; ++t) pos[idx[t]] = t;
  std::vector<double> S((size_t)nfree * nfree, 0.0);
  auto vol = [&](uint32_t i, uint32_t j, uint32_t k) {
    return (double)h->mixd_wf[0][i] * (double)h->mixd_wf[1][j] * (double)h->mixd_wf[2][k];
  };
  for (int t = 0; t < nfree; ++t) {
    const uint32_t c = (uint32_t)idx[t];
    const uint32_t k = c % m.nz, j = (c / m.nz) % m.ny, i = c / (m.ny * m.nz);
    const uint8_t f = fl[c];
    const double V = vol(i, j, k);
    double den = 0.0;
    auto face = [&](uint8_t bit, double coef, int64_t nb) {
      if (!(f & bit)) return;
      den += coef;
      S[(size_t)t * nfree + pos[nb]] -= V * coef;
    };
    const int64_t sx = (int64_t)m.ny * m.nz, sy = m.nz;
    face(kXm, h->mixd_cl[0][i], (int64_t)c - sx);
    face(kXp, h->mixd_ch[0][i], (int64_t)c + sx);
    face(kYm, h->mixd_cl[1][j], (int64_t)c - sy);
    face(kYp, h->mixd_ch[1][j], (int64_t)c + sy);
    face(kZm, h->mixd_cl[2][k], (int64_t)c - 1);
    face(kZp, h->mixd_ch[2][k], (int64_t)c + 1);
    if (outlet && k == 0) den += h->mixd_outlet_add;
    S[(size_t)t * nfree + t] += V * den;
  }
  for (int a = 0; a < nfree; ++a)
    for (int b = a + 1; b < nfree; ++b) {
      const double v = 0.5 * (S[(size_t)a * nfree + b] + S[(size_t)b * nfree + a]);
      S[(size_t)a * nfree + b] = S[(size_t)b * nfree + a] = v;
    }
  // connected sets of free cells (open faces), shifted unless they hold an outlet row
  std::vector<int> comp(nfree, -1);
  int ncomp = 0;
  for (int t0 = 0; t0 < nfree; ++t0) {
    if (comp[t0] >= 0) continue;
    std::vector<int> stack{t0}, members;
    comp[t0] = ncomp;
    bool has_outlet = false;
    while (!stack.empty()) {
      const int t = stack.back();
      stack.pop_back();
      members.push_back(t);
      if (outlet && idx[t] % (int32_t)m.nz == 0) has_outlet = true;
      for (int u = 0; u < nfree; ++u)
        if (u != t && comp[u] < 0 && S[(size_t)t * nfree + u] != 0.0) {
          comp[u] = ncomp;
          stack.push_back(u);
        }
    }
    if (!has_outlet) {
      double dsum = 0.0;
      for (int t : members) dsum += S[(size_t)t * nfree + t];
      const double alpha = dsum / (double)members.size() / (double)members.size();
      for (int a : members)
        for (int b : members) S[(size_t)a * nfree + b] += alpha;
    }
    ++ncomp;
  }
  // Cholesky S = L L^T (lower triangle in place)
  for (int j = 0; j < nfree; ++j) {
    double d = S[(size_t)j * nfree + j];
    for (int q = 0; q < j; ++q) d -= S[(size_t)j * nfree + q] * S[(size_t)j * nfree + q];
    if (!(d > 0.0) || !std::isfinite(d)) return false;
    const double ljj = std::sqrt(d);
    S[(size_t)j * nfree + j] = ljj;
    for (int i = j + 1; i < nfree; ++i) {
      double v = S[(size_t)i * nfree + j];
      for (int q = 0; q < j; ++q) v -= S[(size_t)i * nfree + q] * S[(size_t)j * nfree + q];
      S[(size_t)i * nfree + j] = v / ljj;
    }
  }
  inv.assign((size_t)nfree * nfree, 0.0);
  std::vector<double> y(nfree);
  for (int col = 0; col < nfree; ++col) {
    for (int i = 0; i < nfree; ++i) {  // L y = e_col
      double v = i == col ? 1.0 : 0.0;
      for (int q = 0; q < i; ++q) v -= S[(size_t)i * nfree + q] * y[q];
      y[i] = v / S[(size_t)i * nfree + i];
    }
    for (int i = nfree - 1; i >= 0; --i) {  // L^T x = y
      double v = y[i];
      for (int q = i + 1; q < nfree; ++q) v -= S[(size_t)q * nfree + i] * y[q];
      y[i] = v / S[(size_t)i * nfree + i];
    }
    for (int i = 0; i < nfree; ++i) inv[(size_t)i * nfree + col] = y[i];
  }
  return true;
}

// After the masks change: the free cells of the coarsest mixed level and the
// two inverses (closed, outlet) of its dense solve.  mixd_m = 0 (the tail
// sweeps the level) when the level is too large or has no free cell.
static int build_mix_dense(hfsi_fluid* h, hipStream_t st) {
  h->mixd_m = 0;
  if (h->ML < 2 || !h->mixd_idx) return HFSI_OK;
  const MixLevel& m = h->ml[h->ML - 1];
  std::vector<uint8_t> fl(m.n);
  HFSI_CHECK(hipMemcpyAsync(fl.data(), m.flags, m.n, hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  std::vector<int32_t> idx;
  std::vector<double> vol;
  for (uint32_t c = 0; c < m.n; ++c) {
    if (fl[c] & kNotFree) continue;
    idx.push_back((int32_t)c);
    const uint32_t k = c % m.nz, j = (c / m.nz) % m.ny, i = c / (m.ny * m.nz);
    vol.push_back((double)h->mixd_wf[0][i] * (double)h->mixd_wf[1][j] * (double)h->mixd_wf[2][k]);
  }
  if (idx.empty()) return HFSI_OK;
  std::vector<double> inv0, inv1;
  if (!mix_dense_inverse(h, fl, idx, 0, inv0) || !mix_dense_inverse(h, fl, idx, 1, inv1)) return HFSI_OK;
  const size_t nf = idx.size();
  HFSI_CHECK(hipMemcpyAsync(h->mixd_idx, idx.data(), nf * sizeof(int32_t), hipMemcpyHostToDevice, st));
  HFSI_CHECK(hipMemcpyAsync(h->mixd_vol, vol.data(), nf * sizeof(double), hipMemcpyHostToDevice, st));
  HFSI_CHECK(hipMemcpyAsync(h->mixd_inv[0], inv0.data(), nf * nf * sizeof(double), hipMemcpyHostToDevice, st));
  HFSI_CHECK(hipMemcpyAsync(h->mixd_inv[1], inv1.data(), nf * nf * sizeof(double), hipMemcpyHostToDevice, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  h->mixd_m = (int)nf;
  return HFSI_OK;
}

static void axis_metrics(const std::vector<double>& w, double origin, std::vector<float>& wf,
                         std::vector<float>& df) {
  // centres by running faces (fluid.py:66-87); float32 storage like the reference's fields
  const size_t n = w.size();
  std::vector<double> centers(n);
  double face = origin;
  for (size_t i = 0; i < n; ++i) {
    centers[i] = face + 0.5 * w[i];
    face += w[i];
  }
  wf.resize(n);
  df.resize(n);
  for (size_t i = 0; i < n; ++i) {
    wf[i] = (float)w[i];
    df[i] = (float)(i == 0 ? w[0] : centers[i] - centers[i - 1]);
  }
}

int hfsi_fluid_create(hfsi_fluid** out, int32_t nx, int32_t ny, int32_t nz, const double* widths_x,
                      const double* widths_y, const double* widths_z, const double* origin3, int32_t precision_mask,
                      void* stream) {
  if (!out || nx < 1 || ny < 1 || nz < 1 || !widths_x || !widths_y || !widths_z) {
    set_error("hfsi_fluid_create: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if ((uint64_t)nx * ny * nz >= (1ull << 31)) {
    set_error("hfsi_fluid_create: grid too large for 32-bit cell indices");
    return HFSI_ERR_ARG;
  }
  if (!(precision_mask & (HFSI_PREC_REF64 | HFSI_PREC_FP32 | HFSI_PREC_MIXED)) ||
      (precision_mask & ~(HFSI_PREC_REF64 | HFSI_PREC_FP32 | HFSI_PREC_MIXED))) {
    set_error("hfsi_fluid_create: precision_mask must be a non-empty combination of HFSI_PREC_REF64, "
              "HFSI_PREC_FP32 and HFSI_PREC_MIXED");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  hfsi_fluid* h = new hfsi_fluid();
  h->prec_mask = precision_mask;
  double origin[3] = {0.0, 0.0, 0.0};
  if (origin3) std::memcpy(origin, origin3, sizeof(origin));
  // level shapes and widths (fluid.py:692-729)
  std::vector<std::vector<double>> W[kMaxLevels];
  std::vector<double> cur[3] = {std::vector<double>(widths_x, widths_x + nx),
                                std::vector<double>(widths_y, widths_y + ny),
                                std::vector<double>(widths_z, widths_z + nz)};
  // uniform test of the level-0 grid (fluid.py:150-162)
  h->uniform = true;
  for (int a = 0; a < 3; ++a) {
    double w0 = cur[a][0];
    double tolw = std::max(std::fabs(w0), 1.0) * 1.0e-12;
    for (double v : cur[a])
      if (std::fabs(v - w0) > tolw) h->uniform = false;
  }
  int L = 0;
  while (true) {
    W[L] = {cur[0], cur[1], cur[2]};
    ++L;
    size_t mn = std::min(cur[0].size(), std::min(cur[1].size(), cur[2].size()));
    if (mn <= 3 || L >= kMaxLevels) break;
    std::vector<double> nxt[3];
    bool same = true;
    for (int a = 0; a < 3; ++a) {
      size_t n = cur[a].size();
      size_t cn = std::max<size_t>(2, (n + 1) / 2);
      if (cn != n) same = false;
      for (size_t i = 0; i < n; i += 2) nxt[a].push_back(i + 1 < n ? cur[a][i] + cur[a][i + 1] : cur[a][i]);
      // coarse count follows max(2, (n+1)//2); pairwise sums give ceil(n/2) which equals it for n > 3
    }
    if (same) break;
    for (int a = 0; a < 3; ++a) cur[a] = nxt[a];
  }
  h->L = L;
  int rc = HFSI_OK;
  std::vector<float> wf0[3];
  std::vector<double> cl0[3], ch0[3];
  for (int l = 0; l < L && rc == HFSI_OK; ++l) {
    LevelMem& m = h->lv[l];
    m.nx = (uint32_t)W[l][0].size();
    m.ny = (uint32_t)W[l][1].size();
    m.nz = (uint32_t)W[l][2].size();
    m.n = m.nx * m.ny * m.nz;
    rc |= dalloc(h, &m.flags, m.n);
    rc |= dalloc(h, &m.vact, m.n);
    rc |= dalloc(h, &m.vwraw, m.n);
    rc |= dalloc(h, &m.fw, m.n);
    rc |= dalloc(h, &m.diag, m.n);
    for (int a = 0; a < 3; ++a) {
      std::vector<float> wf, df;
      axis_metrics(W[l][a], origin[a], wf, df);
      const size_t n = wf.size();
      std::vector<double> cl(n, 0.0), ch(n, 0.0), wd(n);
      std::vector<float> clf(n), chf(n);
      for (size_t i = 0; i < n; ++i) {
        wd[i] = (double)wf[i];
        if (i > 0) cl[i] = 1.0 / ((double)wf[i] * (double)df[i]);
        if (i + 1 < n) ch[i] = 1.0 / ((double)wf[i] * (double)df[i + 1]);
        clf[i] = (float)cl[i];
        chf[i] = (float)ch[i];
      }
      if (a == 2) m.outlet_add = 2.0 / ((double)wf[0] * (double)wf[0]);
      if (l == 0) {
        wf0[a] = wf;
        cl0[a] = cl;
        ch0[a] = ch;
      }
      rc |= dalloc(h, &m.cl[a], n);
      rc |= dalloc(h, &m.ch[a], n);
      rc |= dalloc(h, &m.clf[a], n);
      rc |= dalloc(h, &m.chf[a], n);
      rc |= dalloc(h, &m.wf[a], n);
      rc |= dalloc(h, &m.wd[a], n);
      rc |= dalloc(h, &m.df[a], n);
      if (rc != HFSI_OK) break;
      (void)hipMemcpy(m.cl[a], cl.data(), n * sizeof(double), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.ch[a], ch.data(), n * sizeof(double), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.clf[a], clf.data(), n * sizeof(float), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.chf[a], chf.data(), n * sizeof(float), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.wf[a], wf.data(), n * sizeof(float), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.wd[a], wd.data(), n * sizeof(double), hipMemcpyHostToDevice);
      (void)hipMemcpy(m.df[a], df.data(), n * sizeof(float), hipMemcpyHostToDevice);
    }
    if (l >= 1 && rc == HFSI_OK) {
      rc |= dalloc(h, &m.p, m.n);
      rc |= dalloc(h, &m.t, m.n);
      rc |= dalloc(h, &m.rhs, m.n);
    }
  }
  // tail start: first level (>= 1) whose size is at most kTailCells; the
  // coarsest level always runs in the tail
  h->tail_first = L > 1 ? L - 1 : 1;
  for (int l = 1; l < L; ++l)
    if (h->lv[l].n <= kTailCells) {
      h->tail_first = l;
      break;
    }
  const size_t n0 = h->lv[0].n;
  if (rc == HFSI_OK) {
    rc |= dalloc(h, &h->b, n0);
    rc |= dalloc(h, &h->t64, n0);  // level-0 smoother scratch of the standalone solvers
    if (precision_mask & HFSI_PREC_REF64) {
      rc |= dalloc(h, &h->r64, n0);
      rc |= dalloc(h, &h->d64, n0);
      rc |= dalloc(h, &h->q64, n0);
      rc |= dalloc(h, &h->z64, n0);
      rc |= dalloc(h, &h->bi_rold, n0);  // BiCGSTAB fallback vectors
      rc |= dalloc(h, &h->bi_s, n0);
    }
    if (precision_mask & (HFSI_PREC_FP32 | HFSI_PREC_MIXED)) {
      rc |= dalloc(h, &h->r32, n0);
      rc |= dalloc(h, &h->d32, n0);
      rc |= dalloc(h, &h->q32, n0);
      rc |= dalloc(h, &h->z32, n0);
      rc |= dalloc(h, &h->t32, n0);
    }
    rc |= dalloc(h, &h->partials, (size_t)kMaxPartials * 64);
    rc |= dalloc(h, &h->counter, 1);
    rc |= dalloc(h, &h->totals, 64);
    rc |= dalloc(h, &h->scal, 1);
    rc |= dalloc(h, &h->cpl_stats, 1);
  }
  if (rc == HFSI_OK) {
    if (hipHostMalloc((void**)&h->host_scal, sizeof(Scalars), hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc((void**)&h->host_totals, 64 * sizeof(double), hipHostMallocDefault) != hipSuccess) {
      set_error("hipHostMalloc failed");
      rc = HFSI_ERR_HIP;
    }
  }
  if (rc == HFSI_OK) {
    (void)hipMemset(h->counter, 0, sizeof(unsigned int));
    (void)hipMemset(h->scal, 0, sizeof(Scalars));
    // tail argument blocks (geometry pointers are fixed; the has_vd / has_diag
    // switches are refreshed by hfsi_fluid_set_masks)
    rc |= dalloc(h, (char**)&h->tail_args_d, sizeof(TailArgs<double, float>));
    rc |= dalloc(h, (char**)&h->tail_args_f, sizeof(TailArgs<float, float>));
  }
  if (rc == HFSI_OK && (precision_mask & HFSI_PREC_MIXED)) rc = build_mix_hierarchy(h, wf0, cl0, ch0);
  if (rc == HFSI_OK && (precision_mask & HFSI_PREC_MIXED)) {
    if (hipHostMalloc((void**)&h->mon_ring, kMonRing * sizeof(double), hipHostMallocDefault) != hipSuccess) {
      set_error("hipHostMalloc failed");
      rc = HFSI_ERR_HIP;
    }
    h->mon_events.assign(kMonRing, nullptr);
    for (int i = 0; i < kMonRing && rc == HFSI_OK; ++i)
      if (hipEventCreateWithFlags(&h->mon_events[i], hipEventDisableTiming) != hipSuccess) {
        set_error("hipEventCreate failed");
        rc = HFSI_ERR_HIP;
      }
  }
  if (rc == HFSI_OK) {
    (void)hipFuncSetAttribute((const void*)k_vcycle_tail_lds<double>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kTailLdsMax);
    (void)hipFuncSetAttribute((const void*)k_vcycle_tail_lds<float>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kTailLdsMax);
  }
  if (rc == HFSI_OK) {
    // Valid masks from the start (every cell free), so that no kernel can see
    // uninitialised open-face bits before the first hfsi_fluid_set_masks.
    for (int l = 0; l < L; ++l) {
      LevelMem& m = h->lv[l];
      (void)hipMemsetAsync(m.flags, 0, m.n, st);
      hipLaunchKernelGGL(k_open_bits, dim3(blocks_for(m.n)), dim3(kBlock), 0, st, m.nx, m.ny, m.nz, m.flags);
    }
    for (int l = 1; l < h->ML; ++l) {
      MixLevel& m = h->ml[l];
      (void)hipMemsetAsync(m.flags, 0, m.n, st);
      hipLaunchKernelGGL(k_open_bits, dim3(blocks_for(m.n)), dim3(kBlock), 0, st, m.nx, m.ny, m.nz, m.flags);
    }
    if (hipGetLastError() != hipSuccess) rc = HFSI_ERR_HIP;
    if (rc == HFSI_OK) rc = write_tail_args<double>(h, h->tail_args_d, st);
    if (rc == HFSI_OK) rc = write_tail_args<float>(h, h->tail_args_f, st);
    h->tail_outlet = -1;
  }
  if (rc != HFSI_OK) {
    hfsi_fluid_destroy(h);
    return rc;
  }
  HFSI_CHECK(hipStreamSynchronize(st));
  *out = h;
  return HFSI_OK;
}

int hfsi_fluid_destroy(hfsi_fluid* h) {
  if (!h) return HFSI_OK;
  (void)hipDeviceSynchronize();
  for (hipEvent_t e : h->timer_events) (void)hipEventDestroy(e);
  for (hipEvent_t e : h->mon_events)
    if (e) (void)hipEventDestroy(e);
  if (h->mon_ring) (void)hipHostFree(h->mon_ring);
  for (void* p : h->allocs) (void)hipFree(p);
  if (h->host_scal) (void)hipHostFree(h->host_scal);
  if (h->host_totals) (void)hipHostFree(h->host_totals);
  for (void* p : {(void*)h->cpl.a, (void*)h->cpl.b, (void*)h->cpl.ca, (void*)h->cpl.cb})
    if (p) (void)hipFree(p);
  delete h;
  return HFSI_OK;
}

int32_t hfsi_fluid_num_levels(const hfsi_fluid* h) { return h ? h->L : 0; }

int hfsi_fluid_level_shape(const hfsi_fluid* h, int32_t level, int32_t* shape3) {
  if (!h || !shape3 || level < 0 || level >= h->L) {
    set_error("hfsi_fluid_level_shape: invalid arguments");
    return HFSI_ERR_ARG;
  }
  shape3[0] = (int32_t)h->lv[level].nx;
  shape3[1] = (int32_t)h->lv[level].ny;
  shape3[2] = (int32_t)h->lv[level].nz;
  return HFSI_OK;
}

size_t hfsi_fluid_device_bytes(const hfsi_fluid* h) { return h ? h->bytes : 0; }

int hfsi_fluid_set_masks(hfsi_fluid* h, const int32_t* obstacle, const int32_t* vd_active, const float* vd_weight,
                         const double* iface_diag, void* stream) {
  if (!h || !obstacle) {
    set_error("hfsi_fluid_set_masks: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  h->has_vd = vd_active != nullptr;
  h->has_diag = iface_diag != nullptr;
  LevelMem& m0 = h->lv[0];
  hipLaunchKernelGGL(k_flags0, dim3(blocks_for(m0.n)), dim3(kBlock), 0, st, m0.n, obstacle, m0.flags);
  hipLaunchKernelGGL(k_open_bits, dim3(blocks_for(m0.n)), dim3(kBlock), 0, st, m0.nx, m0.ny, m0.nz, m0.flags);
  if (h->has_vd)
    hipLaunchKernelGGL(k_vd0, dim3(blocks_for(m0.n)), dim3(kBlock), 0, st, m0.n, vd_active, vd_weight, m0.vact,
                       m0.vwraw, m0.fw);
  if (h->has_diag) HFSI_CHECK(hipMemcpyAsync(m0.diag, iface_diag, m0.n * sizeof(double), hipMemcpyDeviceToDevice, st));
  for (int l = 1; l < h->L; ++l) {
    LevelMem& f = h->lv[l - 1];
    LevelMem& c = h->lv[l];
    CoarseMaskArgs a;
    a.fnx = f.nx; a.fny = f.ny; a.fnz = f.nz;
    a.cnx = c.nx; a.cny = c.ny; a.cnz = c.nz;
    a.fflags = f.flags;
    a.cflags = c.flags;
    a.fact = h->has_vd ? f.vact : nullptr;
    a.fwraw = f.vwraw;
    a.cact = h->has_vd ? c.vact : nullptr;
    a.cwraw = c.vwraw;
    a.cfw = c.fw;
    a.fdiag = h->has_diag ? f.diag : nullptr;
    a.cdiag = h->has_diag ? c.diag : nullptr;
    a.fwx = f.wf[0]; a.fwy = f.wf[1]; a.fwz = f.wf[2];
    hipLaunchKernelGGL(k_coarse_masks, dim3(blocks_for(c.n)), dim3(kBlock), 0, st, a);
    hipLaunchKernelGGL(k_open_bits, dim3(blocks_for(c.n)), dim3(kBlock), 0, st, c.nx, c.ny, c.nz, c.flags);
  }
  for (int l = 1; l < h->ML; ++l) {
    const MixLevel& f = h->ml[l - 1];
    const MixLevel& c = h->ml[l];
    hipLaunchKernelGGL(k_mix_coarse_flags, dim3(blocks_for(c.n)), dim3(kBlock), 0, st, c.nx, c.ny, c.nz, c.first[0],
                       c.cnt[0], c.first[1], c.cnt[1], c.first[2], c.cnt[2], f.ny, f.nz, (const uint8_t*)f.flags,
                       c.flags);
    hipLaunchKernelGGL(k_open_bits, dim3(blocks_for(c.n)), dim3(kBlock), 0, st, c.nx, c.ny, c.nz, c.flags);
  }
  h->mix_tail_outlet = -1;
  HFSI_LAUNCH_CHECK();
  HFSI_TRY(build_mix_dense(h, st));
  // free volume (V over free cells) into the device scalars
  OpGeo<double> g = geo<double>(h, 0, 0);
  HFSI_TRY(launch_sums<1>(h, g, OpVolume{}, FinFreeVol{h->scal}, st));
  HFSI_TRY(write_tail_args<double>(h, h->tail_args_d, st));
  HFSI_TRY(write_tail_args<float>(h, h->tail_args_f, st));
  h->tail_outlet = -1;  // the rewritten geometries carry the default switch
  return HFSI_OK;
}

int hfsi_fluid_mixed_levels(const hfsi_fluid* h, int32_t* half_levels) {
  if (!h) {
    set_error("hfsi_fluid_mixed_levels: invalid arguments");
    return -1;
  }
  if (half_levels) {
    int nh = 0;
    for (int l = 0; l < h->ML; ++l) nh += mix_half(h, l) ? 1 : 0;
    *half_levels = nh;
  }
  return h->ML;
}

int hfsi_fluid_mixed_level_shape(const hfsi_fluid* h, int32_t level, int32_t* shape3) {
  if (!h || !shape3 || level < 0 || level >= h->ML) {
    set_error("hfsi_fluid_mixed_level_shape: invalid arguments");
    return HFSI_ERR_ARG;
  }
  shape3[0] = (int32_t)h->ml[level].nx;
  shape3[1] = (int32_t)h->ml[level].ny;
  shape3[2] = (int32_t)h->ml[level].nz;
  return HFSI_OK;
}

int hfsi_fluid_mixed_set_half_min_cells(hfsi_fluid* h, int64_t min_cells) {
  if (!h || min_cells < 0) {
    set_error("hfsi_fluid_mixed_set_half_min_cells: invalid arguments");
    return HFSI_ERR_ARG;
  }
  h->mix_half_min_cells = (uint32_t)std::min<int64_t>(min_cells, (int64_t)UINT32_MAX);
  return HFSI_OK;
}

int hfsi_fluid_mixed_set_fused_min_cells(hfsi_fluid* h, int64_t min_cells) {
  if (!h || min_cells < 0) {
    set_error("hfsi_fluid_mixed_set_fused_min_cells: invalid arguments");
    return HFSI_ERR_ARG;
  }
  h->mix_fused_min_cells = (uint32_t)std::min<int64_t>(min_cells, (int64_t)UINT32_MAX);
  return HFSI_OK;
}

int hfsi_fluid_mixed_set_sweep_workgroups(hfsi_fluid* h, int64_t workgroups) {
  if (!h || workgroups < 1 || workgroups > (1 << 20)) {
    set_error("hfsi_fluid_mixed_set_sweep_workgroups: workgroups must be in [1, 2^20]");
    return HFSI_ERR_ARG;
  }
  h->mix_sweep_wgs = (uint32_t)workgroups;
  return HFSI_OK;
}

int hfsi_fluid_divergence(hfsi_fluid* h, const float* velocity, float* divergence, int32_t outlet_zmin,
                          void* stream) {
  if (!h || !velocity || !divergence) {
    set_error("hfsi_fluid_divergence: invalid arguments");
    return HFSI_ERR_ARG;
  }
  OpGeo<float> g = geo<float>(h, 0, outlet_zmin ? 1 : 0);
  hipLaunchKernelGGL(k_divergence, dim3(blocks_for(g.n)), dim3(kBlock), 0, (hipStream_t)stream, g, velocity,
                     divergence);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_fluid_apply(hfsi_fluid* h, const double* p, double* q, int32_t outlet_zmin, void* stream) {
  if (!h || !p || !q) {
    set_error("hfsi_fluid_apply: invalid arguments");
    return HFSI_ERR_ARG;
  }
  OpGeo<double> g = geo<double>(h, 0, outlet_zmin ? 1 : 0);
  hipLaunchKernelGGL((k_apply<double, double, double>), dim3(blocks_for(g.n)), dim3(kBlock), 0, (hipStream_t)stream,
                     g, p, q);
  HFSI_LAUNCH_CHECK();
  if (h->cpl_n) {
    const int rc = launch_couple<double, double>(h, p, q, 1.0, (hipStream_t)stream);
    if (rc != HFSI_OK) return rc;
  }
  return HFSI_OK;
}

// Coupling-list capacity: the list grows (reallocates) only when a call compiles more couplings than
// reserved; hfsi_fluid_reserve_couplings sets the capacity ahead for callers that cannot allocate.
static int reserve_couplings(hfsi_fluid* h, uint32_t count) {
  if (count <= h->cpl_cap) return HFSI_OK;
  for (void* p : {(void*)h->cpl.a, (void*)h->cpl.b, (void*)h->cpl.ca, (void*)h->cpl.cb})
    if (p) HFSI_CHECK(hipFree(p));
  h->cpl = CoupleList{};
  h->cpl_cap = 0;
  h->cpl_n = 0;
  HFSI_CHECK(hipMalloc((void**)&h->cpl.a, count * sizeof(uint32_t)));
  HFSI_CHECK(hipMalloc((void**)&h->cpl.b, count * sizeof(uint32_t)));
  HFSI_CHECK(hipMalloc((void**)&h->cpl.ca, count * sizeof(double)));
  HFSI_CHECK(hipMalloc((void**)&h->cpl.cb, count * sizeof(double)));
  h->cpl_cap = count;
  h->cpl.cap = count;
  return HFSI_OK;
}

int hfsi_fluid_reserve_couplings(hfsi_fluid* h, int64_t capacity) {
  if (!h || capacity < 0 || capacity > (int64_t)UINT32_MAX) {
    set_error("hfsi_fluid_reserve_couplings: invalid arguments");
    return HFSI_ERR_ARG;
  }
  HFSI_CHECK(hipDeviceSynchronize());  // the old list may still be read by queued work
  return reserve_couplings(h, (uint32_t)capacity);
}

int hfsi_fluid_set_interface_couplings(hfsi_fluid* h, const int32_t* obstacle, const hfsi_interface_fields* f,
                                       double* row_diagonal_density, double* report, void* stream) {
  if (!h || !obstacle || !f) {
    set_error("hfsi_fluid_set_interface_couplings: invalid arguments");
    return HFSI_ERR_ARG;
  }
  const LevelMem& m = h->lv[0];
  const bool rows = f->row_count > 0;
  if (rows ? (!f->row_owner || !f->row_neighbor || !f->row_transmissibility)
           : (f->slot_active && (!f->slot_neighbor || !f->slot_coefficient ||
                                 !f->extra_neighbor != !f->extra_coefficient))) {
    set_error("hfsi_fluid_set_interface_couplings: missing coupling array");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  if (!h->cpl_stats) {
    set_error("hfsi_fluid_set_interface_couplings: handle without coupling workspace");
    return HFSI_ERR_STATE;
  }
  CoupleSrc src{};
  src.nx = m.nx;
  src.ny = m.ny;
  src.nz = m.nz;
  src.n = m.n;
  src.obst = obstacle;
  for (int d = 0; d < 3; ++d) src.w[d] = m.wf[d];
  src.slot_active = f->slot_active;
  src.slot_nb = f->slot_neighbor;
  src.slot_coef = f->slot_coefficient;
  src.extra_nb = f->extra_neighbor;
  src.extra_coef = f->extra_coefficient;
  src.row_owner = f->row_owner;
  src.row_nb = f->row_neighbor;
  src.row_T = f->row_transmissibility;
  src.rows = rows ? (uint32_t)std::min<int64_t>(f->row_count, m.n) : 0;
  const bool any = rows || f->slot_active;
  const uint32_t work = rows ? src.rows : m.n;
  const uint32_t blocks = std::max<uint32_t>(1, std::min<uint32_t>((work + kBlock - 1) / kBlock, kMaxGrid));
  CoupleStats zero{};
  CoupleStats host{};
  HFSI_CHECK(hipMemcpyAsync(h->cpl_stats, &zero, sizeof(zero), hipMemcpyHostToDevice, st));
  if (row_diagonal_density) HFSI_CHECK(hipMemsetAsync(row_diagonal_density, 0, (size_t)m.n * sizeof(double), st));
  if (any) {
    hipLaunchKernelGGL((k_couple_build<false>), dim3(blocks), dim3(kBlock), 0, st, src, h->cpl, h->cpl_stats,
                       row_diagonal_density);
    HFSI_LAUNCH_CHECK();
  }
  HFSI_CHECK(hipMemcpyAsync(&host, h->cpl_stats, sizeof(host), hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  const uint32_t count = host.applied;
  if (count > h->cpl_cap) HFSI_TRY(reserve_couplings(h, count));
  h->cpl_n = 0;
  if (count) {
    HFSI_CHECK(hipMemcpyAsync(h->cpl_stats, &zero, sizeof(zero), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL((k_couple_build<true>), dim3(blocks), dim3(kBlock), 0, st, src, h->cpl, h->cpl_stats,
                       (double*)nullptr);
    HFSI_LAUNCH_CHECK();
    CoupleStats filled{};
    HFSI_CHECK(hipMemcpyAsync(&filled, h->cpl_stats, sizeof(filled), hipMemcpyDeviceToHost, st));
    HFSI_CHECK(hipStreamSynchronize(st));
    if (filled.applied != count) {
      set_error("hfsi_fluid_set_interface_couplings: coupling fields changed between the two passes");
      return HFSI_ERR_STATE;
    }
    h->cpl_n = count;
  }
  if (report) {
    report[0] = (double)host.active;
    report[1] = (double)host.invalid;
    report[2] = rows ? (double)std::max<int64_t>((int64_t)f->row_count - (int64_t)m.n, 0) : 0.0;
    report[3] = host.diag_integral;
    report[4] = host.active ? __builtin_bit_cast(double, host.tmax_bits) : 0.0;
    report[5] = (double)count;
  }
  return HFSI_OK;
}

int hfsi_fluid_interface_apply(hfsi_fluid* h, const double* p, double* out, double scale, void* stream) {
  if (!h || !p || !out) {
    set_error("hfsi_fluid_interface_apply: invalid arguments");
    return HFSI_ERR_ARG;
  }
  return launch_couple<double, double>(h, p, out, scale, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// BiCGSTAB fallback (_continue_pressure_poisson_fv_bicgstab, fluid.py:6264-6533)
// ---------------------------------------------------------------------------

namespace hfsi {

struct OpBiResidual {  // r = b - A x (obstacle == 1: 0), the axpby of fluid.py:4519-4531
  double* r;
  const double* b;
  const double* ax;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const { r[c] = (f & kObst) ? 0.0 : b[c] - ax[c]; }
};
struct OpBiReset {  // fluid.py:4614-4628
  const double* r;
  double *rold, *d, *ad, *s, *t;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const {
    rold[c] = (f & kObst) ? 0.0 : r[c];
    d[c] = 0.0;
    ad[c] = 0.0;
    s[c] = 0.0;
    t[c] = 0.0;
  }
};
struct OpBiDirection {  // fluid.py:4630-4638
  double* d;
  const double *r, *ad;
  double beta, omega;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const {
    d[c] = (f & kObst) ? 0.0 : r[c] + beta * (d[c] - omega * ad[c]);
  }
};
struct OpBiAlpha {  // fluid.py:4640-4650
  double* x;
  const double *z, *r, *ad;
  double* s;
  double alpha;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const {
    if (f & kObst) {
      x[c] = 0.0;
      s[c] = 0.0;
    } else {
      x[c] = x[c] + alpha * z[c];
      s[c] = r[c] - alpha * ad[c];
    }
  }
};
struct OpBiOmega {  // fluid.py:4652-4661
  double* x;
  const double *z, *s, *t;
  double* r;
  double omega;
  __device__ void operator()(uint32_t c, bool, uint8_t f) const {
    if (f & kObst) {
      x[c] = 0.0;
      r[c] = 0.0;
    } else {
      x[c] = x[c] + omega * z[c];
      r[c] = s[c] - omega * t[c];
    }
  }
};
struct OpSubConstant {  // field - mean on free cells, 0 elsewhere (fluid.py:4716-4722)
  double* f;
  double mean;
  __device__ void operator()(uint32_t c, bool free, uint8_t) const { f[c] = free ? f[c] - mean : 0.0; }
};
struct OpCopy64 {
  double* dst;
  const double* src;
  __device__ void operator()(uint32_t c, bool, uint8_t) const { dst[c] = src[c]; }
};
struct OpSumVol {
  const double* f;
  __device__ void operator()(uint32_t c, double V, double (&acc)[2]) const {
    acc[0] += f[c] * V;
    acc[1] += V;
  }
};

}  // namespace hfsi

int hfsi_fluid_solve_bicgstab(hfsi_fluid* h, const double* rhs, double* x, int32_t start_iteration,
                              int32_t max_iterations, double b_norm, int32_t outlet_zmin, double tolerance,
                              int32_t remove_mean, hfsi_cg_stats* S, void* stream) {
  if (!h || !x || !S || !h->r64) {
    set_error("hfsi_fluid_solve_bicgstab: invalid arguments (the handle needs the float64 CG vectors)");
    return HFSI_ERR_ARG;
  }
  const double* b = rhs ? rhs : h->b;
  hipStream_t st = (hipStream_t)stream;
  const LevelMem& m = h->lv[0];
  if (!h->bi_rold || !h->bi_s) {
    set_error("hfsi_fluid_solve_bicgstab: the handle has no float64 vectors (create it with HFSI_PREC_REF64)");
    return HFSI_ERR_STATE;
  }
  const int outlet = outlet_zmin ? 1 : 0;
  OpGeo<double> g = geo<double>(h, 0, outlet);
  double *r = h->r64, *d = h->d64, *ad = h->q64, *z = h->z64, *t = h->t64, *rold = h->bi_rold, *sv = h->bi_s;
  const int iters = std::max(1, (int)max_iterations);
  const double tol = std::max(0.0, tolerance);
  const double floor = 1.0e-300;
  S->breakdown_kind = HFSI_BREAKDOWN_NONE;
  S->converged = 0;

  auto wdot = [&](const double* a, const double* c2, double* out) -> int {
    HFSI_TRY(launch_sums<1>(h, g, OpDot<double, double>{a, c2}, FinStore{}, st));
    HFSI_CHECK(hipMemcpyAsync(h->host_totals, h->totals, sizeof(double), hipMemcpyDeviceToHost, st));
    HFSI_CHECK(hipStreamSynchronize(st));
    *out = h->host_totals[0];
    return HFSI_OK;
  };
  auto project = [&](double* f) -> int {
    if (!remove_mean) return HFSI_OK;
    HFSI_TRY(launch_sums<2>(h, g, OpSumVol{f}, FinStore{}, st));
    HFSI_CHECK(hipMemcpyAsync(h->host_totals, h->totals, 2 * sizeof(double), hipMemcpyDeviceToHost, st));
    HFSI_CHECK(hipStreamSynchronize(st));
    const double mean = h->host_totals[1] > 0.0 ? h->host_totals[0] / h->host_totals[1] : 0.0;
    HFSI_TRY(launch_pointwise(h, 0, OpSubConstant{f, mean}, st));
    S->mean_projection_count += 1;
    return HFSI_OK;
  };
  auto apply = [&](const double* p, double* q) -> int {
    hipLaunchKernelGGL((k_apply<double, double, double>), dim3(blocks_for(g.n)), dim3(kBlock), 0, st, g, p, q);
    HFSI_LAUNCH_CHECK();
    return launch_couple<double, double>(h, p, q, 1.0, st);
  };
  auto jacobi = [&](const double* src, double* dst) -> int {
    hipLaunchKernelGGL((k_jacobi_precond<double, double, double>), dim3(blocks_for(g.n)), dim3(kBlock), 0, st, g,
                       src, dst);
    HFSI_LAUNCH_CHECK();
    return HFSI_OK;
  };
  auto residual = [&]() -> int {  // r = b - A x, projected
    HFSI_TRY(apply(x, ad));
    HFSI_TRY(launch_pointwise(h, 0, OpBiResidual{r, b, ad}, st));
    return project(r);
  };
  auto reset = [&]() -> int { return launch_pointwise(h, 0, OpBiReset{r, rold, d, ad, sv, t}, st); };
  auto norm_check = [&](const double* v, int it, double& rel) -> int {
    double vv = 0.0;
    HFSI_TRY(wdot(v, v, &vv));
    S->host_residual_checks += 1;
    rel = std::sqrt(std::max(vv, 0.0)) / b_norm;
    if (it >= 0) S->iterations = start_iteration + it;
    S->relative_residual = rel;
    return HFSI_OK;
  };

  double rel = 0.0;
  HFSI_TRY(residual());
  HFSI_TRY(norm_check(r, -1, rel));
  if (rel <= tol) {
    S->converged = 1;
    return HFSI_OK;
  }
  HFSI_TRY(reset());
  double rho_prev = 1.0, alpha = 1.0, omega = 1.0;
  // a failed scalar restarts from the true residual (or from s for the omega scalars), or ends
  // the solve with its message on the last iteration
  auto restart_from_x = [&]() -> int {
    HFSI_TRY(residual());
    HFSI_TRY(reset());
    rho_prev = alpha = omega = 1.0;
    S->restart_count += 1;
    return HFSI_OK;
  };
  for (int it = 1; it <= iters; ++it) {
    double rho = 0.0;
    HFSI_TRY(wdot(rold, r, &rho));
    if (!std::isfinite(rho) || std::fabs(rho) <= floor) {
      if (it >= iters) {
        S->breakdown_kind = HFSI_BREAKDOWN_BICGSTAB_SHADOW;
        return HFSI_OK;
      }
      HFSI_TRY(residual());
      HFSI_TRY(norm_check(r, it, rel));
      if (rel <= tol) {
        S->converged = 1;
        return HFSI_OK;
      }
      HFSI_TRY(reset());
      rho_prev = alpha = omega = 1.0;
      S->restart_count += 1;
      continue;
    }
    double beta = 0.0;
    if (it > 1) {
      if (!std::isfinite(rho_prev) || std::fabs(rho_prev) <= floor || !std::isfinite(omega) ||
          std::fabs(omega) <= floor) {
        if (it >= iters) {
          S->breakdown_kind = HFSI_BREAKDOWN_BICGSTAB_RECURRENCE;
          return HFSI_OK;
        }
        HFSI_TRY(restart_from_x());
        continue;
      }
      beta = (rho / rho_prev) * (alpha / omega);
      if (!std::isfinite(beta)) {
        if (it >= iters) {
          S->breakdown_kind = HFSI_BREAKDOWN_BICGSTAB_BETA;
          return HFSI_OK;
        }
        HFSI_TRY(restart_from_x());
        continue;
      }
    }
    HFSI_TRY(launch_pointwise(h, 0, OpBiDirection{d, r, ad, beta, omega}, st));
    HFSI_TRY(jacobi(d, z));
    HFSI_TRY(project(z));
    HFSI_TRY(apply(z, ad));
    double den = 0.0;
    HFSI_TRY(wdot(rold, ad, &den));
    if (!std::isfinite(den) || std::fabs(den) <= floor) {
      if (it >= iters) {
        S->breakdown_kind = HFSI_BREAKDOWN_BICGSTAB_ALPHA_DEN;
        return HFSI_OK;
      }
      HFSI_TRY(restart_from_x());
      continue;
    }
    alpha = rho / den;
    if (!std::isfinite(alpha)) {
      if (it >= iters) {
        S->breakdown_kind = HFSI_BREAKDOWN_BICGSTAB_ALPHA;
        return HFSI_OK;
      }
      HFSI_TRY(restart_from_x());
      continue;
    }
    HFSI_TRY(launch_pointwise(h, 0, OpBiAlpha{x, z, r, ad, sv, alpha}, st));
    HFSI_TRY(project(sv));
    HFSI_TRY(norm_check(sv, it, rel));
    if (rel <= tol) {
      HFSI_TRY(launch_pointwise(h, 0, OpCopy64{r, sv}, st));
      S->converged = 1;
      return HFSI_OK;
    }
    HFSI_TRY(jacobi(sv, z));
    HFSI_TRY(project(z));
    HFSI_TRY(apply(z, t));
    double ts = 0.0, tt = 0.0;
    HFSI_TRY(wdot(t, sv, &ts));
    HFSI_TRY(wdot(t, t, &tt));
    const bool tt_bad = !std::isfinite(tt) || std::fabs(tt) <= floor;
    if (!tt_bad) omega = ts / tt;
    if (tt_bad || !std::isfinite(omega) || std::fabs(omega) <= floor) {
      if (it >= iters) {
        S->breakdown_kind = tt_bad ? HFSI_BREAKDOWN_BICGSTAB_OMEGA_DEN : HFSI_BREAKDOWN_BICGSTAB_OMEGA;
        return HFSI_OK;
      }
      HFSI_TRY(launch_pointwise(h, 0, OpCopy64{r, sv}, st));
      HFSI_TRY(project(r));
      HFSI_TRY(reset());
      rho_prev = alpha = omega = 1.0;
      S->restart_count += 1;
      continue;
    }
    HFSI_TRY(launch_pointwise(h, 0, OpBiOmega{x, z, sv, t, r, omega}, st));
    if (it % 16 == 0) {
      HFSI_TRY(project(x));
      HFSI_TRY(project(r));
    }
    HFSI_TRY(norm_check(r, it, rel));
    if (rel <= tol) {
      S->converged = 1;
      return HFSI_OK;
    }
    rho_prev = rho;
  }
  S->breakdown_kind = HFSI_BREAKDOWN_BICGSTAB_NOT_CONVERGED;
  return HFSI_OK;
}

int hfsi_fluid_diagonal(hfsi_fluid* h, double* diag, int32_t outlet_zmin, void* stream) {
  if (!h || !diag) {
    set_error("hfsi_fluid_diagonal: invalid arguments");
    return HFSI_ERR_ARG;
  }
  OpGeo<double> g = geo<double>(h, 0, outlet_zmin ? 1 : 0);
  hipLaunchKernelGGL(k_diagonal<double>, dim3(blocks_for(g.n)), dim3(kBlock), 0, (hipStream_t)stream, g, diag);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_fluid_weighted_dot(hfsi_fluid* h, const double* a, const double* b, double* out, void* stream) {
  if (!h || !a || !b || !out) {
    set_error("hfsi_fluid_weighted_dot: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  OpGeo<double> g = geo<double>(h, 0, 0);
  HFSI_TRY(launch_sums<1>(h, g, OpDot<double, double>{a, b}, FinNone{}, st));
  HFSI_CHECK(hipMemcpyAsync(h->host_totals, h->totals, sizeof(double), hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  *out = h->host_totals[0];
  return HFSI_OK;
}

int hfsi_fluid_vcycle(hfsi_fluid* h, const double* r, double* z, int32_t precision, int32_t pre, int32_t coarse,
                      int32_t post, int32_t outlet_zmin, void* stream) {
  if (!h || !r || !z || pre < 1 || coarse < (precision == HFSI_PREC_MIXED ? 0 : 1) || post < 1) {
    set_error("hfsi_fluid_vcycle: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if (!(h->prec_mask & precision)) {
    set_error("hfsi_fluid_vcycle: precision not enabled on this handle");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int outlet = outlet_zmin ? 1 : 0;
  HFSI_TRY(set_tail_outlet(h, outlet, st));
  if (precision == HFSI_PREC_REF64) {
    HFSI_TRY((run_vcycle<double, double, LdNeg<double, double>>(h, z, h->t64, LdNeg<double, double>{r}, true, pre,
                                                                 coarse, post, outlet, st)));
  } else if (precision == HFSI_PREC_FP32) {
    HFSI_TRY(launch_pointwise(h, 0, OpCopy<double, float>{r, h->r32}, st));
    HFSI_TRY((run_vcycle<float, float, LdNeg<float, float>>(h, h->z32, h->t32, LdNeg<float, float>{h->r32}, true,
                                                             pre, coarse, post, outlet, st)));
    HFSI_TRY(launch_pointwise(h, 0, OpCopy<float, double>{h->z32, z}, st));
  } else if (precision == HFSI_PREC_MIXED) {
    // z = M r with the scale taken from r itself (vin = 1 / RMS_V(r))
    HFSI_TRY(launch_pointwise(h, 0, OpCopy<double, float>{r, h->r32}, st));
    OpGeo<double> g64 = geo<double>(h, 0, outlet);
    HFSI_TRY(launch_sums<1>(h, g64, OpDot<float, float>{h->r32, h->r32}, FinVScale{h->scal, h->mix_kappa}, st));
    HFSI_TRY((mix_precondition<3>(h, h->r32, h->q32, h->z32, pre, coarse, post, outlet, FinNone{}, st)));
    HFSI_TRY(launch_pointwise(h, 0, OpCopy<float, double>{h->z32, z}, st));
  } else {
    set_error("hfsi_fluid_vcycle: unsupported precision");
    return HFSI_ERR_ARG;
  }
  return HFSI_OK;
}

int hfsi_fluid_solve_cg(hfsi_fluid* h, const float* divergence, const float* source, const double* iface_rhs,
                        double* pressure, const hfsi_cg_options* opt, hfsi_cg_stats* stats, void* stream) {
  if (!h || !divergence || !pressure || !opt) {
    set_error("hfsi_fluid_solve_cg: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if (!(h->prec_mask & opt->precision)) {
    set_error("hfsi_fluid_solve_cg: precision not enabled on this handle");
    return HFSI_ERR_ARG;
  }
  if (opt->preconditioner < 0 || opt->preconditioner > 3) {
    set_error("hfsi_fluid_solve_cg: unsupported preconditioner");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  HFSI_TRY(set_tail_outlet(h, opt->outlet_zmin ? 1 : 0, st));
  hfsi_cg_stats local;
  hfsi_cg_stats& S = stats ? *stats : local;
  if (opt->precision == HFSI_PREC_REF64)
    return solve_cg<double, double>(h, divergence, source, iface_rhs, pressure, *opt, S, st);
  if (opt->precision == HFSI_PREC_FP32)
    return solve_cg<float, float>(h, divergence, source, iface_rhs, pressure, *opt, S, st);
  if (opt->precision == HFSI_PREC_MIXED)
    return solve_cg<float, float>(h, divergence, source, iface_rhs, pressure, *opt, S, st, true);
  set_error("hfsi_fluid_solve_cg: unsupported precision");
  return HFSI_ERR_ARG;
}

int hfsi_fluid_solve_fv_jacobi(hfsi_fluid* h, const float* divergence, const float* source, const double* iface_rhs,
                               double* pressure, double rhs_scale, int32_t iterations, int32_t outlet_zmin,
                               void* stream) {
  if (!h || !divergence || !pressure || iterations < 0) {
    set_error("hfsi_fluid_solve_fv_jacobi: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int outlet = outlet_zmin ? 1 : 0;
  HFSI_TRY(launch_pointwise(h, 0, OpRhsLegacy{divergence, source, iface_rhs, h->b, (float)rhs_scale}, st));
  OpGeo<double> g = geo<double>(h, 0, outlet);
  Ld<double, double> R{h->b};
  double* in = pressure;
  for (int m = 0; m < iterations; ++m) {
    double* out = (in == pressure) ? h->t64 : pressure;
    hipLaunchKernelGGL((k_jacobi<double, Ld<double, double>, Ld<double, double>, double>), dim3(blocks_for(g.n)),
                       dim3(kBlock), 0, st, g, Ld<double, double>{in}, R, out, (double)0.8f);
    in = out;
  }
  HFSI_LAUNCH_CHECK();
  if (in != pressure) HFSI_CHECK(hipMemcpyAsync(pressure, in, g.n * sizeof(double), hipMemcpyDeviceToDevice, st));
  return HFSI_OK;
}

int hfsi_fluid_solve_fv_multigrid(hfsi_fluid* h, const float* divergence, const float* source,
                                  const double* iface_rhs, double* pressure, double rhs_scale, int32_t iterations,
                                  int32_t cycles, int32_t outlet_zmin, void* stream) {
  if (!h || !divergence || !pressure) {
    set_error("hfsi_fluid_solve_fv_multigrid: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int outlet = outlet_zmin ? 1 : 0;
  HFSI_TRY(set_tail_outlet(h, outlet, st));
  HFSI_TRY(launch_pointwise(h, 0, OpRhsLegacy{divergence, source, iface_rhs, h->b, (float)rhs_scale}, st));
  Ld<double, double> R{h->b};
  if (h->L <= 1) {
    int its = std::max(1, iterations);
    return hfsi_fluid_solve_fv_jacobi(h, divergence, source, iface_rhs, pressure, rhs_scale, its, outlet_zmin, stream);
  }
  int ncyc = cycles > 0 ? cycles : (h->uniform ? 12 : 24);
  for (int c = 0; c < ncyc; ++c)
    HFSI_TRY((run_vcycle<double, double, Ld<double, double>>(h, pressure, h->t64, R, false, 3, 36, 3, outlet, st)));
  if (!h->uniform)
    return hfsi_fluid_solve_fv_jacobi(h, divergence, source, iface_rhs, pressure, rhs_scale, std::max(1, iterations),
                                      outlet_zmin, stream);
  return HFSI_OK;
}

int hfsi_fluid_solve_legacy_jacobi(hfsi_fluid* h, const float* divergence, const float* source,
                                   const int32_t* obstacle, double* pressure, double rhs_scale, double inv_dx2,
                                   double inv_dy2, double inv_dz2, int32_t iterations, int32_t outlet_zmin,
                                   void* stream) {
  if (!h || !divergence || !obstacle || !pressure || iterations < 0) {
    set_error("hfsi_fluid_solve_legacy_jacobi: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  LevelMem& m = h->lv[0];
  LegacyArgs a;
  a.nx = m.nx; a.ny = m.ny; a.nz = m.nz;
  a.obst = obstacle;
  a.div = divergence;
  a.src = source;
  a.rhs_scale = (float)rhs_scale;
  a.ix2 = (float)inv_dx2;
  a.iy2 = (float)inv_dy2;
  a.iz2 = (float)inv_dz2;
  a.outlet = outlet_zmin ? 1 : 0;
  double* in = pressure;
  for (int it = 0; it < iterations; ++it) {
    double* out = (in == pressure) ? h->t64 : pressure;
    a.p = in;
    a.out = out;
    hipLaunchKernelGGL(k_legacy_jacobi, dim3(blocks_for(m.n)), dim3(kBlock), 0, st, a);
    in = out;
  }
  HFSI_LAUNCH_CHECK();
  if (in != pressure) HFSI_CHECK(hipMemcpyAsync(pressure, in, m.n * sizeof(double), hipMemcpyDeviceToDevice, st));
  return HFSI_OK;
}

int hfsi_fluid_subtract_gradient(hfsi_fluid* h, float* velocity, const double* pressure, const int32_t* vd_active,
                                 const float* vd_weight, const float* vd_value, float dt_over_rho,
                                 int32_t outlet_zmin, void* stream) {
  if (!h || !velocity || !pressure || (vd_active && !vd_weight)) {
    set_error("hfsi_fluid_subtract_gradient: invalid arguments");
    return HFSI_ERR_ARG;
  }
  GradArgs a;
  a.g = geo<double>(h, 0, outlet_zmin ? 1 : 0);
  a.u = velocity;
  a.p = pressure;
  a.dx = h->lv[0].df[0];
  a.dy = h->lv[0].df[1];
  a.dz = h->lv[0].df[2];
  a.vda = vd_active;
  a.vdw = vd_weight;
  a.vdv = vd_value;
  a.dt_over_rho = dt_over_rho;
  hipLaunchKernelGGL(k_subtract_gradient, dim3(blocks_for(a.g.n)), dim3(kBlock), 0, (hipStream_t)stream, a);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_fluid_wall_clamp(hfsi_fluid* h, float* velocity, int32_t outlet_zmin, void* stream) {
  if (!h || !velocity) {
    set_error("hfsi_fluid_wall_clamp: invalid arguments");
    return HFSI_ERR_ARG;
  }
  LevelMem& m = h->lv[0];
  uint32_t most = std::max(m.ny * m.nz, std::max(m.nx * m.nz, m.nx * m.ny));
  hipLaunchKernelGGL(k_wall_clamp, dim3((most + 255) / 256), dim3(256), 0, (hipStream_t)stream, m.nx, m.ny, m.nz,
                     velocity, outlet_zmin ? 1 : 0);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_fluid_predict(hfsi_fluid* h, const float* velocity_prev, const int32_t* obstacle, float* velocity,
                       const hfsi_axis_metrics* metrics, float dt_s, float nu_m2_s, int32_t scheme, void* stream) {
  if (!h || !velocity_prev || !obstacle || !velocity || !metrics) {
    set_error("hfsi_fluid_predict: invalid arguments");
    return HFSI_ERR_ARG;
  }
  const LevelMem& m = h->lv[0];
  const size_t bytes = (size_t)m.n * 3 * sizeof(float);
  const char* vp0 = (const char*)velocity_prev;
  const char* v0 = (const char*)velocity;
  if (vp0 < v0 + bytes && v0 < vp0 + bytes) {
    set_error("hfsi_fluid_predict: velocity and velocity_prev overlap");
    return HFSI_ERR_ARG;
  }
  if (!(dt_s > 0.0f) || !std::isfinite(dt_s) || !std::isfinite(nu_m2_s)) {
    set_error("hfsi_fluid_predict: dt_s must be positive and nu_m2_s finite");
    return HFSI_ERR_ARG;
  }
  if (scheme != HFSI_ADVECT_EULER && scheme != HFSI_ADVECT_RK2) {
    set_error("hfsi_fluid_predict: unsupported advection scheme");
    return HFSI_ERR_ARG;
  }
  if (m.nx < 2 || m.ny < 2 || m.nz < 2) {
    set_error("hfsi_fluid_predict: the predictor needs at least 2 cells along every axis");
    return HFSI_ERR_ARG;
  }
  if (m.n >= (1u << 31) || m.nx >= (1u << 24) || m.ny >= (1u << 24) || m.nz >= (1u << 24)) {
    set_error("hfsi_fluid_predict: grids of 2^31 cells or more, or 2^24 cells along an axis, are not supported");
    return HFSI_ERR_ARG;
  }
  PredictArgs a;
  a.nx = m.nx;
  a.ny = m.ny;
  a.nz = m.nz;
  a.n = m.n;
  a.fz = FastDiv::make(m.nz);
  a.fy = FastDiv::make(m.ny);
  for (int d = 0; d < 3; ++d) {
    if (!metrics->faces[d] || !metrics->centers[d] || !metrics->widths[d] || !metrics->center_distances[d]) {
      set_error("hfsi_fluid_predict: missing metric array");
      return HFSI_ERR_ARG;
    }
    a.face[d] = metrics->faces[d];
    a.centre[d] = metrics->centers[d];
    a.width[d] = metrics->widths[d];
    a.cdist[d] = metrics->center_distances[d];
  }
  a.vp = velocity_prev;
  a.obst = obstacle;
  a.v = velocity;
  a.dt = dt_s;
  a.nu = nu_m2_s;
  const uint32_t ncells = m.nx + m.ny + m.nz;
  const bool lds = ncells <= kPredictLdsMaxCells;
  const bool off32 = (uint64_t)m.n * 12 < (1ull << 32);
  const size_t shmem = lds ? (kPredictLdsTables * (size_t)ncells + (off32 ? m.nx : 0)) * sizeof(float) : 0;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid(blocks_for(m.n)), block(kBlock);
  timer_mark(h, HFSI_TIMER_PREDICT, st);
  const bool rk2 = scheme == HFSI_ADVECT_RK2;
  if (lds && off32) {
    if (rk2)
      hipLaunchKernelGGL((k_predict<true, true, uint32_t>), grid, block, shmem, st, a);
    else
      hipLaunchKernelGGL((k_predict<false, true, uint32_t>), grid, block, shmem, st, a);
  } else if (lds) {
    if (rk2)
      hipLaunchKernelGGL((k_predict<true, true, uint64_t>), grid, block, shmem, st, a);
    else
      hipLaunchKernelGGL((k_predict<false, true, uint64_t>), grid, block, shmem, st, a);
  } else if (off32) {
    if (rk2)
      hipLaunchKernelGGL((k_predict<true, false, uint32_t>), grid, block, shmem, st, a);
    else
      hipLaunchKernelGGL((k_predict<false, false, uint32_t>), grid, block, shmem, st, a);
  } else {
    if (rk2)
      hipLaunchKernelGGL((k_predict<true, false, uint64_t>), grid, block, shmem, st, a);
    else
      hipLaunchKernelGGL((k_predict<false, false, uint64_t>), grid, block, shmem, st, a);
  }
  HFSI_LAUNCH_CHECK();
  timer_mark(h, HFSI_TIMER_PREDICT, st);
  return HFSI_OK;
}

static bool guess_coarsens(const hfsi_fluid* h, int32_t coarsen) {
  const LevelMem& m = h->lv[0];
  return coarsen && m.nx % 2 == 0 && m.ny % 2 == 0 && m.nz % 2 == 0;
}

int hfsi_guess_features(hfsi_fluid* h, const float* divergence, int32_t coarsen, double net_min_width,
                        float* features, void* stream) {
  if (!h || !divergence || !features || !(net_min_width > 0.0) || (coarsen && !guess_coarsens(h, coarsen))) {
    set_error("hfsi_guess_features: invalid arguments (coarsening needs even grid dimensions)");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const OpGeo<double> g = geo<double>(h, 0, 0);
  const int cf = coarsen ? 2 : 1;
  const uint32_t cnx = g.nx / cf, cny = g.ny / cf, cnz = g.nz / cf, nc = cnx * cny * cnz;
  const uint32_t nb = blocks_for(nc);
  if (cf == 2)
    hipLaunchKernelGGL(k_guess_features<2>, dim3(nb), dim3(kBlock), 0, st, g, divergence, cny, cnz, nc,
                       1.0 / net_min_width, h->t64, features, h->partials);
  else
    hipLaunchKernelGGL(k_guess_features<1>, dim3(nb), dim3(kBlock), 0, st, g, divergence, cny, cnz, nc,
                       1.0 / net_min_width, h->t64, features, h->partials);
  finish_sums<2>(h, nb, FinGuessRms{h->scal}, st);
  hipLaunchKernelGGL(k_guess_normalise, dim3(blocks_for(nc)), dim3(kBlock), 0, st, nc, (const double*)h->t64, features,
                     (const Scalars*)h->scal);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_guess_pressure(hfsi_fluid* h, const float* net_out, const float* divergence, const float* source,
                        double rho_over_dt, double net_kappa, int32_t coarsen, int32_t outlet_zmin, double* pressure,
                        double* gamma_out, void* stream) {
  if (!h || !net_out || !divergence || !pressure || !(net_kappa > 0.0) ||
      (coarsen && !guess_coarsens(h, coarsen))) {
    set_error("hfsi_guess_pressure: invalid arguments (coarsening needs even grid dimensions)");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const OpGeo<double> g = geo<double>(h, 0, outlet_zmin ? 1 : 0);
  const int cf = coarsen ? 2 : 1;
  const uint32_t cny = g.ny / cf, cnz = g.nz / cf;
  const uint32_t nb = blocks_for(g.n);
  const double coef = -rho_over_dt / net_kappa;  // network units -> pressure, times the divergence RMS
  if (cf == 2)
    hipLaunchKernelGGL(k_guess_prolong<2>, dim3(nb), dim3(kBlock), 0, st, g, net_out, cny, cnz, coef,
                       (const Scalars*)h->scal, pressure, divergence, source, rho_over_dt, h->partials);
  else
    hipLaunchKernelGGL(k_guess_prolong<1>, dim3(nb), dim3(kBlock), 0, st, g, net_out, cny, cnz, coef,
                       (const Scalars*)h->scal, pressure, divergence, source, rho_over_dt, h->partials);
  const int remove_mean = outlet_zmin ? 0 : 1;
  finish_sums<3>(h, nb, FinGuessMean{h->scal}, st);
  hipLaunchKernelGGL(k_guess_center, dim3(nb), dim3(kBlock), 0, st, g, pressure, divergence, source, rho_over_dt,
                     (const Scalars*)h->scal, remove_mean, h->partials);
  finish_sums<1>(h, nb, FinGuessNum{h->scal}, st);
  hipLaunchKernelGGL(k_guess_energy, dim3(nb), dim3(kBlock), 0, st, g, (const double*)pressure, h->partials);
  finish_sums<1>(h, nb, FinGuessGamma{h->scal}, st);
  hipLaunchKernelGGL(k_guess_scale, dim3(nb), dim3(kBlock), 0, st, g.n, pressure, (const Scalars*)h->scal);
  HFSI_LAUNCH_CHECK();
  if (gamma_out) {
    HFSI_TRY(sync_scalars(h, st));
    *gamma_out = h->host_scal->g_gamma;
  }
  return HFSI_OK;
}

int hfsi_fluid_mark_sphere(hfsi_fluid* h, const float* center_x, const float* center_y, const float* center_z,
                           const float* centre3, float radius, int32_t* obstacle, void* stream) {
  if (!h || !center_x || !center_y || !center_z || !centre3 || !obstacle || !(radius > 0.0f)) {
    set_error("hfsi_fluid_mark_sphere: invalid arguments");
    return HFSI_ERR_ARG;
  }
  const LevelMem& m = h->lv[0];
  hipLaunchKernelGGL(k_mark_sphere, dim3(blocks_for(m.n)), dim3(kBlock), 0, (hipStream_t)stream, m.nx, m.ny, m.nz,
                     center_x, center_y, center_z, centre3[0], centre3[1], centre3[2], radius, obstacle);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

static VelocityRowArgs velocity_row_args(hfsi_fluid* h, float* velocity, const int32_t* obstacle, float rho) {
  const LevelMem& m = h->lv[0];
  VelocityRowArgs a{};
  a.nx = m.nx;
  a.ny = m.ny;
  a.nz = m.nz;
  a.u = velocity;
  a.obstacle = obstacle;
  a.wx = m.wf[0];
  a.wy = m.wf[1];
  a.wz = m.wf[2];
  a.rho = rho;
  a.partials = h->partials;
  return a;
}

// Copy `count` totals to the host report (synchronises).
static int read_totals(hfsi_fluid* h, double* out, int count, hipStream_t st) {
  HFSI_CHECK(hipMemcpyAsync(h->host_totals, h->totals, count * sizeof(double), hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  std::memcpy(out, h->host_totals, count * sizeof(double));
  if (!(out[2] >= 0.0)) out[2] = 0.0;  // no active cell: the max starts at zero
  return HFSI_OK;
}

int hfsi_fluid_apply_velocity_rows(hfsi_fluid* h, float* velocity, const int32_t* obstacle,
                                   const int32_t* vd_active, const float* vd_value, float rho, double* report6,
                                   void* stream) {
  if (!h || !velocity || !obstacle || !vd_active || !vd_value) {
    set_error("hfsi_fluid_apply_velocity_rows: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  VelocityRowArgs a = velocity_row_args(h, velocity, obstacle, rho);
  a.active = vd_active;
  a.value = vd_value;
  const uint32_t nb = blocks_for(h->lv[0].n);
  hipLaunchKernelGGL(k_velocity_rows, dim3(nb), dim3(kBlock), 0, st, a);
  if (!report6) {
    HFSI_LAUNCH_CHECK();
    return HFSI_OK;
  }
  finish_sums<kRowSlots>(h, nb, FinStore{}, st, kRowMaxMask);
  HFSI_LAUNCH_CHECK();
  return read_totals(h, report6, kRowSlots, st);
}

int hfsi_fluid_apply_velocity_constraints(hfsi_fluid* h, float* velocity, const int32_t* obstacle,
                                          const hfsi_velocity_constraints* c, float blend,
                                          float solid_mobility_ratio, float rho, double* primary_impulse3,
                                          double* secondary_impulse3, double* report12, void* stream) {
  if (!h || !velocity || !obstacle || !c || !c->sum || !c->weight || !c->primary_sum || !c->primary_weight ||
      !c->secondary_sum || !c->secondary_weight || !primary_impulse3 || !secondary_impulse3) {
    set_error("hfsi_fluid_apply_velocity_constraints: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if (!(blend >= 0.0f && blend <= 1.0f) || !std::isfinite(solid_mobility_ratio) || solid_mobility_ratio < 0.0f) {
    set_error("hfsi_fluid_apply_velocity_constraints: blend must be in [0, 1] and the solid mobility ratio "
              "finite and non-negative");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  VelocityRowArgs a = velocity_row_args(h, velocity, obstacle, rho);
  a.sum = c->sum;
  a.weight = c->weight;
  a.psum = c->primary_sum;
  a.pweight = c->primary_weight;
  a.ssum = c->secondary_sum;
  a.sweight = c->secondary_weight;
  volatile float one_plus = 1.0f + solid_mobility_ratio;  // float32, as on the device
  a.scale = blend / one_plus;
  const uint32_t nb = blocks_for(h->lv[0].n);
  hipLaunchKernelGGL(k_velocity_constraints, dim3(nb), dim3(kBlock), 0, st, a);
  finish_sums<kConSlots>(h, nb, FinConstraintImpulse{primary_impulse3, secondary_impulse3}, st, kRowMaxMask);
  HFSI_LAUNCH_CHECK();
  return report12 ? read_totals(h, report12, kConSlots, st) : HFSI_OK;
}

int hfsi_fluid_local_divergence_cleanup(hfsi_fluid* h, float* velocity, const float* divergence,
                                        const float* source, const int32_t* obstacle, const int32_t* vd_active,
                                        float dx, float dy, float dz, float relaxation, void* stream) {
  if (!h || !velocity || !divergence || !obstacle || !(dx > 0.0f) || !(dy > 0.0f) || !(dz > 0.0f) ||
      !(relaxation >= 0.0f && relaxation <= 1.0f)) {
    set_error("hfsi_fluid_local_divergence_cleanup: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if (!h->uniform) {
    set_error("hfsi_fluid_local_divergence_cleanup: non-uniform grid divergence cleanup is not available");
    return HFSI_ERR_ARG;
  }
  const LevelMem& m = h->lv[0];
  CleanupArgs a{};
  a.nx = m.nx;
  a.ny = m.ny;
  a.nz = m.nz;
  a.u = velocity;
  a.div = divergence;
  a.src = source;
  a.obstacle = obstacle;
  a.vda = vd_active;
  const float d[3] = {dx, dy, dz};
  for (int e = 0; e < 3; ++e) {
    volatile float dd = d[e] * d[e];  // float32 square, then a float32 reciprocal
    a.inv[e] = 1.0f / d[e];
    a.inv2[e] = 1.0f / dd;
  }
  a.relax = relaxation;
  hipLaunchKernelGGL(k_local_divergence_cleanup, dim3(blocks_for(m.n)), dim3(kBlock), 0, (hipStream_t)stream, a);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_fluid_kernel_timer(hfsi_fluid* h, int32_t kernel_id) {
  if (!h || kernel_id < 0 || kernel_id > HFSI_TIMER_PREDICT) {
    set_error("hfsi_fluid_kernel_timer: invalid arguments");
    return HFSI_ERR_ARG;
  }
  timer_flush(h);
  h->timer_id = kernel_id;
  h->timer_ms = 0.0;
  h->timer_count = 0;
  if (kernel_id != 0 && h->timer_events.empty()) {
    h->timer_events.resize(4096);
    for (hipEvent_t& e : h->timer_events) HFSI_CHECK(hipEventCreate(&e));
  }
  return HFSI_OK;
}

int hfsi_fluid_kernel_timer_read(hfsi_fluid* h, int64_t* launches, double* total_ms) {
  if (!h || !launches || !total_ms) {
    set_error("hfsi_fluid_kernel_timer_read: invalid arguments");
    return HFSI_ERR_ARG;
  }
  timer_flush(h);
  *launches = h->timer_count;
  *total_ms = h->timer_ms;
  return HFSI_OK;
}

int hfsi_fluid_divergence_report(hfsi_fluid* h, const float* divergence, const float* source,
                                 const double* iface_div, const int32_t* vd_active, int32_t outlet_zmin,
                                 double* out54, void* stream) {
  if (!h || !divergence || !out54) {
    set_error("hfsi_fluid_divergence_report: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  ReportArgs a;
  a.g = geo<float>(h, 0, outlet_zmin ? 1 : 0);
  a.div = divergence;
  a.src = source;
  a.idiv = iface_div;
  a.vda = vd_active;
  a.partials = h->partials;
  a.counter = h->counter;
  a.totals = h->totals;
  const uint32_t nb = std::min(blocks_for(a.g.n), std::max(kReportBlocks, blocks_for(a.g.n / 16)));
  hipLaunchKernelGGL(k_div_report, dim3(nb), dim3(kBlock), 0, st, a);
  hipLaunchKernelGGL(k_finish_report, dim3(kReportSlots), dim3(kFinishThreads), 0, st, (const double*)h->partials, nb,
                     h->totals);
  HFSI_LAUNCH_CHECK();
  HFSI_CHECK(hipMemcpyAsync(h->host_totals, h->totals, 54 * sizeof(double), hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  std::memcpy(out54, h->host_totals, 54 * sizeof(double));
  return HFSI_OK;
}

}  // extern "C"
