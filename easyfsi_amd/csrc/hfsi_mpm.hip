// libhfsi: neo-Hookean MLS/APIC MPM particle <-> grid transfers for gfx950.
//
// One step (simulation_core/neo_hookean_mpm.py:695-959), atomic path:
//   k_mpm_clear      grid mass / momentum / force := 0
//   k_mpm_p2g        SVD clamp of F, first Piola stress, affine momentum,
//                    27-node quadratic B-spline scatter (hardware fp32 atomics)
//   k_mpm_grid       v = p/m + dt f/m, transfer snapshot, damping
//   k_mpm_g2p        27-node gather, APIC C, x += dt v, F <- (I + dt C) F,
//                    surface normal / area update
//   k_mpm_radial     centroid-relative radial stretch diagnostics
// Binned path (default): particles binned by block of 4^3 or 8^3 nodes; P2G as a per-particle
// pass (k_mpm_p2g_prepare, k_mpm_p2g_prepare_svd) and a per-cell scatter into
// LDS tiles (k_mpm_p2g_fine or k_mpm_p2g_cells, k_mpm_p2g_force); the grid update gathers the tiles
// (k_mpm_grid_gather); G2P from an LDS velocity tile per block (k_mpm_g2p_binned)
// with its report sums in a pass of their own (k_mpm_g2p_sums).
// The report quantities are reduced deterministically (workgroup partials,
// combined in workgroup order by a one-workgroup finish launch); the final
// 34-value report snapshot is assembled on the device.
#include <hip/hip_runtime.h>

#include <cmath>
#include <algorithm>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/hfsi.h"
#include "hfsi_common.hpp"

namespace hfsi {

constexpr double kMinSigma = 1.0e-2;
constexpr double kMaxSigma = 1.0e2;

// ---------------------------------------------------------------------------
// 3x3 helpers (float64)
// ---------------------------------------------------------------------------

struct M3 {
  double a[3][3];
};

__device__ inline M3 mmul(const M3& A, const M3& B) {
  M3 C;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C.a[i][j] = A.a[i][0] * B.a[0][j] + A.a[i][1] * B.a[1][j] + A.a[i][2] * B.a[2][j];
  return C;
}

__device__ inline M3 mtrans(const M3& A) {
  M3 T;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) T.a[i][j] = A.a[j][i];
  return T;
}

__device__ inline double mdet(const M3& A) {
  return A.a[0][0] * (A.a[1][1] * A.a[2][2] - A.a[1][2] * A.a[2][1]) -
         A.a[0][1] * (A.a[1][0] * A.a[2][2] - A.a[1][2] * A.a[2][0]) +
         A.a[0][2] * (A.a[1][0] * A.a[2][1] - A.a[1][1] * A.a[2][0]);
}

// inverse transpose (cofactor matrix / det)
__device__ inline M3 minv_t(const M3& A, double det) {
  M3 R;
  const double id = 1.0 / det;
  R.a[0][0] = (A.a[1][1] * A.a[2][2] - A.a[1][2] * A.a[2][1]) * id;
  R.a[0][1] = (A.a[1][2] * A.a[2][0] - A.a[1][0] * A.a[2][2]) * id;
  R.a[0][2] = (A.a[1][0] * A.a[2][1] - A.a[1][1] * A.a[2][0]) * id;
  R.a[1][0] = (A.a[0][2] * A.a[2][1] - A.a[0][1] * A.a[2][2]) * id;
  R.a[1][1] = (A.a[0][0] * A.a[2][2] - A.a[0][2] * A.a[2][0]) * id;
  R.a[1][2] = (A.a[0][1] * A.a[2][0] - A.a[0][0] * A.a[2][1]) * id;
  R.a[2][0] = (A.a[0][1] * A.a[1][2] - A.a[0][2] * A.a[1][1]) * id;
  R.a[2][1] = (A.a[0][2] * A.a[1][0] - A.a[0][0] * A.a[1][2]) * id;
  R.a[2][2] = (A.a[0][0] * A.a[1][1] - A.a[0][1] * A.a[1][0]) * id;
  return R;
}

// SVD F = U diag(s) V^T with U, V proper rotations, |s0| >= |s1| >= |s2| and
// the sign of det F carried by s2.  Method: cyclic Jacobi eigen-decomposition
// of the symmetric F^T F (V and s^2), eigenvalues sorted descending, then a
// Givens QR factorisation F V = U R whose rotations keep det U = +1; s is the
// diagonal of R (the structure of McAdams et al., "Computing the singular
// value decomposition of 3x3 matrices with minimal branching and elementary
// floating point operations", 2011, here with exact rotations in float64).
__device__ inline void svd3(const M3& F, M3& U, double s[3], M3& V) {
  M3 A = mmul(mtrans(F), F);
  M3 W;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) W.a[i][j] = i == j ? 1.0 : 0.0;
  for (int sweep = 0; sweep < 12; ++sweep) {
    double off = A.a[0][1] * A.a[0][1] + A.a[0][2] * A.a[0][2] + A.a[1][2] * A.a[1][2];
    double diag = A.a[0][0] * A.a[0][0] + A.a[1][1] * A.a[1][1] + A.a[2][2] * A.a[2][2];
    if (off <= 1.0e-32 * diag || off == 0.0) break;
#pragma unroll
    for (int pq = 0; pq < 3; ++pq) {
      const int p = pq == 2 ? 1 : 0;
      const int q = pq == 0 ? 1 : 2;
      const double apq = A.a[p][q];
      if (apq == 0.0) continue;
      const double theta = (A.a[q][q] - A.a[p][p]) / (2.0 * apq);
      const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
      const double c = 1.0 / sqrt(t * t + 1.0);
      const double sn = t * c;
      // A <- J^T A J, J rotation in the (p, q) plane
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double akp = A.a[k][p], akq = A.a[k][q];
        A.a[k][p] = c * akp - sn * akq;
        A.a[k][q] = sn * akp + c * akq;
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double apk = A.a[p][k], aqk = A.a[q][k];
        A.a[p][k] = c * apk - sn * aqk;
        A.a[q][k] = sn * apk + c * aqk;
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double wkp = W.a[k][p], wkq = W.a[k][q];
        W.a[k][p] = c * wkp - sn * wkq;
        W.a[k][q] = sn * wkp + c * wkq;
      }
    }
  }
  // sort eigenvalues descending (columns of W follow)
  double lam[3] = {A.a[0][0], A.a[1][1], A.a[2][2]};
  int idx[3] = {0, 1, 2};
  if (lam[idx[0]] < lam[idx[1]]) { int t = idx[0]; idx[0] = idx[1]; idx[1] = t; }
  if (lam[idx[1]] < lam[idx[2]]) { int t = idx[1]; idx[1] = idx[2]; idx[2] = t; }
  if (lam[idx[0]] < lam[idx[1]]) { int t = idx[0]; idx[0] = idx[1]; idx[1] = t; }
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) V.a[i][j] = W.a[i][idx[j]];
  if (mdet(V) < 0.0) {
    V.a[0][2] = -V.a[0][2];
    V.a[1][2] = -V.a[1][2];
    V.a[2][2] = -V.a[2][2];
  }
  // Givens QR of B = F V: rows (0,1), (0,2), (1,2)
  M3 B = mmul(F, V);
  M3 Q;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) Q.a[i][j] = i == j ? 1.0 : 0.0;
  const int ri[3] = {0, 0, 1}, rj[3] = {1, 2, 2}, col[3] = {0, 0, 1};
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    const int i = ri[g], j = rj[g], k = col[g];
    const double a = B.a[i][k], b = B.a[j][k];
    const double r = sqrt(a * a + b * b);
    double c = 1.0, sn = 0.0;
    if (r > 0.0) {
      c = a / r;
      sn = b / r;
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double bi = B.a[i][m], bj = B.a[j][m];
      B.a[i][m] = c * bi + sn * bj;
      B.a[j][m] = -sn * bi + c * bj;
    }
    // Q <- Q G^T
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double qi = Q.a[m][i], qj = Q.a[m][j];
      Q.a[m][i] = c * qi + sn * qj;
      Q.a[m][j] = -sn * qi + c * qj;
    }
  }
  U = Q;
  s[0] = B.a[0][0];
  s[1] = B.a[1][1];
  s[2] = B.a[2][2];
}

// ---------------------------------------------------------------------------
// Kernel arguments
// ---------------------------------------------------------------------------

struct MpmArgs {
  // particles (caller-owned)
  float* x;
  float* v;
  float* C;
  float* F;
  const float* mass;
  const float* volume;
  const float* rest_x;
  const int32_t* fixed;
  const int32_t* region;
  const float* f_ext;
  float* normal;
  const float* rest_normal;
  float* area;
  const float* rest_area;
  int32_t count;
  // grid (caller-owned)
  float* gm;
  float* gv;
  float* gf;
  int32_t nx, ny, nz;
  float bmin[3];
  float dx[3];
  float dt, mu, lambda, damping;
  int32_t primary, secondary;
  // reductions: workgroup partials stored slot-major, partials[slot * pstride + prow0 + workgroup]
  double* partials;
  uint32_t prow0, pstride;
  unsigned int* counter;
  double* totals;   // per-stage totals
  double* report;   // 34 packed values (device)
};

// Stage totals layout
enum {
  T_PMOM = 0,    // 3
  T_FEXT = 3,    // 3
  T_MASS = 6,
  T_VOL = 7,
  T_PSQ = 8,
  T_MAXJ = 9,    // max
  T_CLAMP = 10,
  T_OOB = 11,
  T_TRANS = 12,  // 3
  T_GMOM = 15,   // 3
  T_ACTIVE = 18,
  T_MAXV = 19,   // max
  T_PDISP = 20,  // 3
  T_PVEL = 23,   // 3
  T_SDISP = 26,  // 3
  T_SVEL = 29,   // 3
  T_PCNT = 32,
  T_SCNT = 33,
  T_CCUR = 34,   // 3
  T_CREST = 37,  // 3
  T_CCNT = 40,
  T_RSUM = 41,
  T_RCNT = 42,
  T_RMAX = 43,   // max
  T_COUNT = 44   // the two doubles after the step's totals hold the layered surface's region masses
};

// max-reduced slots of each stage (relative to the stage's first total)
constexpr uint64_t kP2gMax = 1ull << T_MAXJ;
constexpr uint64_t kGridMax = 1ull << 7;
constexpr uint64_t kRadialMax = 1ull << 2;

// Workgroup partials, slot-major: the finishing workgroup reads each slot's rows contiguously.
template <int NS>
__device__ inline void mpm_partials(double (&v)[NS], const MpmArgs& a, uint32_t row, double* lds, uint64_t maxmask) {
  block_reduce<NS>(v, lds, maxmask);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) a.partials[(size_t)s * a.pstride + row] = v[s];
  }
}

// Combine nrows slot-major partial rows.  The partials come from every XCD,
// so each load misses this XCD's L2: a thread issues the loads of kMpmFinishRows rows (t, t + 512,
// ...) before adding them in row order, so that up to 2048 rows take one memory round trip; the
// thread sums are then combined by the workgroup tree (a fixed order).
constexpr int kMpmFinishThreads = 512;
constexpr int kMpmFinishRows = 4;

template <int NS>
__device__ inline void finish_rows(const double* partials, uint32_t nrows, uint32_t stride, double* totals,
                                   uint64_t maxmask, double* lds) {
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = ((maxmask >> s) & 1) ? -INFINITY : 0.0;
  for (uint32_t b0 = threadIdx.x; b0 < nrows; b0 += kMpmFinishRows * kMpmFinishThreads) {
    double p[kMpmFinishRows][NS];
#pragma unroll
    for (int r = 0; r < kMpmFinishRows; ++r) {
      const uint32_t b = b0 + (uint32_t)r * kMpmFinishThreads;
#pragma unroll
      for (int s = 0; s < NS; ++s)
        p[r][s] = b < nrows ? partials[(size_t)s * stride + b] : (((maxmask >> s) & 1) ? -INFINITY : 0.0);
    }
#pragma unroll
    for (int r = 0; r < kMpmFinishRows; ++r)
#pragma unroll
      for (int s = 0; s < NS; ++s) acc[s] = ((maxmask >> s) & 1) ? fmax(acc[s], p[r][s]) : acc[s] + p[r][s];
  }
  block_reduce<NS>(acc, lds, maxmask);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) totals[s] = acc[s];
  }
}

// One table of partial rows, then the finaliser.
template <int NS, typename Fin>
__global__ void __launch_bounds__(kMpmFinishThreads) k_mpm_finish(const double* partials, uint32_t nrows,
                                                                   uint32_t stride, double* totals, Fin fin,
                                                                   uint64_t maxmask) {
  __shared__ double lds[NS * (kMpmFinishThreads / 64)];
  finish_rows<NS>(partials, nrows, stride, totals, maxmask, lds);
  if (threadIdx.x == 0) fin(totals);
}

// Totals 0..40 of a step: the scatter's, the grid update's and the gather's tables, one workgroup
// each.  A table takes 6 us, nearly all of it latency (one workgroup, two memory round trips), and
// nothing reads a total before the radial stretch: three launches in the step's chain became one.
struct StageRows {
  const double* partials;
  uint32_t nrows;
};

__global__ void __launch_bounds__(kMpmFinishThreads) k_mpm_finish_stages(StageRows p2g, StageRows grid, StageRows g2p,
                                                                          double* totals) {
  __shared__ double lds[21 * (kMpmFinishThreads / 64)];
  if (blockIdx.x == 0)
    finish_rows<12>(p2g.partials, p2g.nrows, p2g.nrows, totals, kP2gMax, lds);
  else if (blockIdx.x == 1)
    finish_rows<8>(grid.partials, grid.nrows, grid.nrows, totals + T_TRANS, kGridMax, lds);
  else
    finish_rows<21>(g2p.partials, g2p.nrows, g2p.nrows, totals + T_PDISP, 0ull, lds);
}

__device__ inline void grid_coord(const MpmArgs& a, const float* xp, float X[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) X[d] = (xp[d] - a.bmin[d]) / a.dx[d];
}

// Written as the negation of "inside" so that a NaN coordinate counts as out
// of bounds and never reaches the node-index computation.
__device__ inline bool stencil_oob(const MpmArgs& a, const float X[3]) {
  const bool inside = X[0] >= 0.5f && X[0] < (float)a.nx - 1.5f && X[1] >= 0.5f && X[1] < (float)a.ny - 1.5f &&
                      X[2] >= 0.5f && X[2] < (float)a.nz - 1.5f;
  return !inside;
}

__device__ inline void bspline(float f, float w[3]) {
  w[0] = 0.5f * (1.5f - f) * (1.5f - f);
  w[1] = 0.75f - (f - 1.0f) * (f - 1.0f);
  w[2] = 0.5f * (f - 0.5f) * (f - 0.5f);
}


// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock) k_mpm_clear(uint32_t n, float* gm, float* gv, float* gf) {
  HFSI_CELL_LOOP(n) {
    gm[c] = 0.0f;
    gv[3 * (size_t)c + 0] = 0.0f;
    gv[3 * (size_t)c + 1] = 0.0f;
    gv[3 * (size_t)c + 2] = 0.0f;
    gf[3 * (size_t)c + 0] = 0.0f;
    gf[3 * (size_t)c + 1] = 0.0f;
    gf[3 * (size_t)c + 2] = 0.0f;
  }
}

// P2G (neo_hookean_mpm.py:712-801).  Totals 0..11.
//
// Per particle: the SVD clamp of F (persisted when it changed), the first
// Piola stress of the clamped F and the affine momentum, plus the report
// sums; the 27-node scatter is done by the caller (global atomics, or LDS
// atomics into a block tile in the binned path).
struct P2gPart {
  bool inb;
  int base[3];
  float X[3], fx[3], w[3][3];
  float m, mom[3], aff[3][3], fe[3];
};

// Stencil base node, offset from it and quadratic B-spline weights of grid coordinates X.
__device__ inline void p2g_stencil(const float (&X)[3], P2gPart& q) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q.X[d] = X[d];
    q.base[d] = (int)floorf(X[d] - 0.5f);
    q.fx[d] = X[d] - (float)q.base[d];
    bspline(q.fx[d], q.w[d]);
  }
}

// SVD = false: a particle whose F needs the SVD clamp is left untouched (no sums, no F store) and
// false is returned, so that the caller can defer it to a pass that carries the SVD code (which
// would otherwise set the register count of the common path).
template <bool SVD = true>
__device__ inline bool p2g_prepare(const MpmArgs& a, uint32_t p, double (&acc)[12], P2gPart& q) {
  float X[3];
  grid_coord(a, a.x + 3 * (size_t)p, X);
  p2g_stencil(X, q);
  M3 F;
  const float* Fp_in = a.F + 9 * (size_t)p;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) F.a[i][j] = (double)Fp_in[3 * i + j];
  const double detF = mdet(F);
  const double raw_J = (double)(float)detF;
  // Singular values inside [kMinSigma, kMaxSigma] with det F > 0 leave F unchanged (no clamp, no
  // reflection: U diag(sigma) V^T = F), and they are there when sigma_max <= ||F||_F <= kMaxSigma and
  // sigma_min = det F / (sigma_mid sigma_max) >= det F / ||F||_F^2 >= kMinSigma: then the SVD is skipped.
  double fro2 = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) fro2 += F.a[i][j] * F.a[i][j];
  const bool inside = detF > 0.0 && fro2 <= kMaxSigma * kMaxSigma && detF >= kMinSigma * fro2;
  if (!SVD && !inside) return false;
  bool clamped = false;
  M3 Fc = F;
  if (SVD && !inside) {
    M3 U, V;
    double sig[3];
    svd3(F, U, sig, V);
    double sc[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      sc[d] = fmin(fmax(fabs(sig[d]), kMinSigma), kMaxSigma);
      if (fabs(sc[d] - sig[d]) > 1.0e-6) clamped = true;
    }
    if (mdet(mmul(U, mtrans(V))) < 0.0) {
      clamped = true;
      U.a[0][2] = -U.a[0][2];
      U.a[1][2] = -U.a[1][2];
      U.a[2][2] = -U.a[2][2];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        Fc.a[i][j] = U.a[i][0] * sc[0] * V.a[j][0] + U.a[i][1] * sc[1] * V.a[j][1] + U.a[i][2] * sc[2] * V.a[j][2];
    if (mdet(Fc) <= 0.0) {
      clamped = true;
      Fc.a[0][2] = -Fc.a[0][2];
      Fc.a[1][2] = -Fc.a[1][2];
      Fc.a[2][2] = -Fc.a[2][2];
    }
    if (raw_J <= 0.0) clamped = true;
  }
  // float32 state: the stress uses the stored (rounded) corrected F
  M3 Fs;
  float* Fp_out = a.F + 9 * (size_t)p;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      float fv = (float)Fc.a[i][j];
      Fs.a[i][j] = (double)fv;
      if (clamped) Fp_out[3 * i + j] = fv;
    }
  const double J = mdet(Fs);
  const M3 FinvT = minv_t(Fs, J);
  const double lnJ = log(J);
  M3 Pk;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      Pk.a[i][j] = (double)a.mu * (Fs.a[i][j] - FinvT.a[i][j]) + (double)a.lambda * lnJ * FinvT.a[i][j];
  const M3 PFt = mmul(Pk, mtrans(Fs));
  const float m_p = a.mass[p];
  const float vol_p = a.volume[p];
  const bool fixed = a.fixed && a.fixed[p] != 0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double inv = 4.0 / ((double)a.dx[j] * (double)a.dx[j]);
      const double stress = -(double)a.dt * (double)vol_p * PFt.a[i][j] * inv;
      q.aff[i][j] = fixed ? 0.0f : (float)(stress + (double)m_p * (double)a.C[9 * (size_t)p + 3 * i + j]);
    }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q.mom[d] = fixed ? 0.0f : m_p * a.v[3 * (size_t)p + d];
    q.fe[d] = (fixed || !a.f_ext) ? 0.0f : a.f_ext[3 * (size_t)p + d];
  }
  q.m = m_p;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    acc[T_PMOM + d] += q.mom[d];
    acc[T_FEXT + d] += q.fe[d];
  }
  acc[T_MASS] += m_p;
  acc[T_VOL] += vol_p;
  acc[T_PSQ] += (double)q.mom[0] * q.mom[0] + (double)q.mom[1] * q.mom[1] + (double)q.mom[2] * q.mom[2];
  acc[T_MAXJ] = fmax(acc[T_MAXJ], fabs(J));
  acc[T_CLAMP] += clamped ? 1.0 : 0.0;
  q.inb = !stencil_oob(a, X);
  if (!q.inb) acc[T_OOB] += 1.0;
  return true;
}

// A prepared particle staged for the binned scatter as four float4: grid coordinates and mass,
// momentum and aff[0][0], then aff[0][1], aff[0][2], aff[1][0], aff[1][1], then aff[1][2] and row 2.
// The scatter rebuilds the stencil from the stored coordinates with the same arithmetic as the
// preparation, so a staged particle scatters exactly what an unstaged one does.
__device__ inline void p2g_stage(float4* s, const P2gPart& q) {
  s[0] = make_float4(q.X[0], q.X[1], q.X[2], q.m);
  s[1] = make_float4(q.mom[0], q.mom[1], q.mom[2], q.aff[0][0]);
  s[2] = make_float4(q.aff[0][1], q.aff[0][2], q.aff[1][0], q.aff[1][1]);
  s[3] = make_float4(q.aff[1][2], q.aff[2][0], q.aff[2][1], q.aff[2][2]);
}

__device__ inline void p2g_unstage(const float4 (&s)[4], P2gPart& q) {
  const float X[3] = {s[0].x, s[0].y, s[0].z};
  p2g_stencil(X, q);
  q.inb = true;
  q.m = s[0].w;
  q.mom[0] = s[1].x;
  q.mom[1] = s[1].y;
  q.mom[2] = s[1].z;
  q.aff[0][0] = s[1].w;
  q.aff[0][1] = s[2].x;
  q.aff[0][2] = s[2].y;
  q.aff[1][0] = s[2].z;
  q.aff[1][1] = s[2].w;
  q.aff[1][2] = s[3].x;
  q.aff[2][0] = s[3].y;
  q.aff[2][1] = s[3].z;
  q.aff[2][2] = s[3].w;
#pragma unroll
  for (int d = 0; d < 3; ++d) q.fe[d] = 0.0f;
}

// The 27 node contributions of a particle: node(ox, oy, oz) gets mass wt m,
// momentum wt (m v + aff dpos) and force wt f_ext.
template <typename Sink>
__device__ inline void p2g_scatter(const MpmArgs& a, const P2gPart& q, Sink sink) {
#pragma unroll
  for (int ox = 0; ox < 3; ++ox)
#pragma unroll
    for (int oy = 0; oy < 3; ++oy)
#pragma unroll
      for (int oz = 0; oz < 3; ++oz) {
        const float wt = q.w[0][ox] * q.w[1][oy] * q.w[2][oz];
        const float dp0 = ((float)ox - q.fx[0]) * a.dx[0];
        const float dp1 = ((float)oy - q.fx[1]) * a.dx[1];
        const float dp2 = ((float)oz - q.fx[2]) * a.dx[2];
        float md[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) md[d] = wt * (q.mom[d] + (q.aff[d][0] * dp0 + q.aff[d][1] * dp1 + q.aff[d][2] * dp2));
        sink(ox, oy, oz, wt * q.m, md, wt);
      }
}

__global__ void __launch_bounds__(kBlock) k_mpm_p2g(MpmArgs a) {
  constexpr int NS = 12;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const uint32_t n = (uint32_t)a.count;
  const uint32_t sx = (uint32_t)a.ny * a.nz, sy = a.nz;
  HFSI_CELL_LOOP(n) {
    P2gPart q;
    p2g_prepare(a, c, acc, q);
    if (!q.inb) continue;
    p2g_scatter(a, q, [&](int ox, int oy, int oz, float mw, const float (&md)[3], float wt) {
      const uint32_t node = (uint32_t)(q.base[0] + ox) * sx + (uint32_t)(q.base[1] + oy) * sy + (uint32_t)(q.base[2] + oz);
      atomicAdd(&a.gm[node], mw);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        atomicAdd(&a.gv[3 * (size_t)node + d], md[d]);
        if (q.fe[d] != 0.0f) atomicAdd(&a.gf[3 * (size_t)node + d], wt * q.fe[d]);
      }
    });
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, kP2gMax);
}

// ---------------------------------------------------------------------------
// Cell-binned P2G: particles are bucketed by the block of EDGE^3 nodes of their stencil base node; one
// workgroup sums a block's particles cell by cell into a tile of (EDGE + 2)^3 nodes in LDS, and the
// grid update gathers every node from the tiles that cover it (or, without tile buffers, the tile is
// added to the grid with one global atomic per touched node value instead of 27 x 7 per particle).
// ---------------------------------------------------------------------------

// Blocks of 8^3 nodes have 2.0 tile nodes per cell, and their 512 cells can be ordered by particle
// count before lanes take them; but a small body has too few of them: 32^3 particles span 27 to 64, and
// one workgroup's chain of steps sets the time (scatter 66 us, gather 35 us).  Blocks of 4^3 (3.4 tile
// nodes per cell, a wavefront's lanes are a block's cells) are eight times as many: 12 and 11 us.  The
// whole step, loaded, with 4^3 against 8^3 blocks (us):
//   16^3 particles 77 / 89, 32^3 at 4.6 per cell 81 / 163 and at 1.4 80 / 99, 50^3 at 5.2 115 / 244 and at
//   2.2 118 / 156, 64^3 at 4.6 151 / 229 and at 2.4 168 / 213, 80^3 at 9.0 213 / 370 and at 2.4 236 / 246,
//   100^3 at 9.0 364 / 535 but at 2.2 442 / 387, 128^3 at 4.6 738 / 707.
// The line lies where the sparse body's two times meet, by the state's particle capacity (the tile
// buffers' layout hangs on it).
constexpr int kFineEdge = 4, kCoarseEdge = 8;
constexpr int64_t kFineParticles = 1 << 19;

template <int EDGE>
struct Tile {
  static constexpr int kEdge = EDGE + 2;  // stencil reach of a block
  static constexpr int kNodes = kEdge * kEdge * kEdge;
  static constexpr int kCells = EDGE * EDGE * EDGE;
  // components of a block's tile: mass, momentum (3), external force (3)
  static constexpr size_t kStride = (size_t)7 * kNodes;
};

// Grids of up to this many blocks of 8^3 nodes get tile buffers (28 KB per 8^3 block, 6 KB per 4^3
// block, for as many blocks as can hold particles at once: the smaller of the block and the particle
// count); larger grids flush tiles with global atomics.
constexpr size_t kMaxTileBlocks = 65536;
// Grids are taken up to this many blocks of 8^3 nodes (per-block tables of 4 MB each, 32 MB at 4^3).
constexpr size_t kMaxBlocks = 1u << 20;

struct BinArgs {
  int32_t edge;            // nodes per block edge: kFineEdge or kCoarseEdge
  int32_t nbx, nby, nbz;   // block grid
  int32_t* key;            // per particle: block, or -1 when out of bounds
  int32_t* rank;           // per particle: slot within its block
  int32_t* count;          // per block
  int32_t* offset;         // per active block: its first entry of sorted
  int32_t* slot;           // per active block: its place in the active list
  int32_t* sorted;         // particles ordered by block
  int32_t* cell;           // per in-bounds particle: its stencil base cell within its block
  int32_t* scell;          // cell of each entry of sorted
  int32_t* active;         // blocks with particles (unordered)
  int32_t* nactive;
  int32_t* nsorted;        // entries of sorted handed out to active blocks
  int32_t* oob;            // out-of-bounds particles (unordered)
  int32_t* noob;
  int32_t* svd;            // particles whose F takes the SVD clamp this step (unordered)
  int32_t* nsvd;
  // tile path: every active block stores its whole tile (plain stores) and the grid update gathers each
  // node from the (up to 8) tiles that cover it, in a fixed order
  float* tiles;            // [active block][component][tile node], or nullptr (atomic flush)
  float4* stage;           // per particle: the prepared scatter operands (p2g_stage), 4 float4
  int32_t* need_stamp;     // per block: stamp of the step that last listed it
  int32_t* need_list;      // blocks with nodes a tile covers: the active blocks and their +1 neighbours
  int32_t* nneed;
  int32_t stamp;           // this step's stamp (never 0: need_stamp starts at 0)
  int32_t has_force;       // particles carry an external force (force components stored)
  int32_t* block_force;    // per active block: its tile holds force components (some particle has a force)
  int32_t* prev_need;      // the previous step's need list: every grid node outside it is zero
  int32_t* nprev;
  int32_t reset_prev;      // the grid was cleared whole this step: forget the previous list
};

__global__ void k_bin_clear(BinArgs b) {
  const int32_t nb = b.nbx * b.nby * b.nbz;
  for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nb; i += gridDim.x * blockDim.x) b.count[i] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *b.nactive = 0;
    *b.nsorted = 0;
    *b.noob = 0;
    *b.nsvd = 0;
    if (b.nneed) *b.nneed = 0;
    if (b.nprev && b.reset_prev) *b.nprev = 0;
  }
}

// Lists of the active blocks and of the blocks whose nodes their tiles cover (an active block and its
// +1 neighbours, so a block is needed when it or one of its seven -1 neighbours is active), and the
// ranges of `sorted`, one thread per block.  The counts of all eight blocks are loaded at once and a
// workgroup takes its places in the three lists with one atomic each, so the pass is two memory round
// trips long at any number of active blocks: 125 blocks of a 64^3-node grid took 7.5 us by marking
// neighbours from the active list through an exchange each, after two scan launches over the blocks.
constexpr int kListBlocks = 1024;  // blocks per workgroup: runs of the lists that keep neighbours together

__global__ void __launch_bounds__(kListBlocks) k_bin_lists(BinArgs b) {
  constexpr int kWaves = kListBlocks / 64;
  __shared__ int32_t wave_total[3][kWaves], first[3];
  const int32_t nblk = b.nbx * b.nby * b.nbz;
  const int32_t k = (int32_t)(blockIdx.x * kListBlocks + threadIdx.x);
  const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
  int32_t cnt = 0;
  bool need = false;
  if (k < nblk) {
    cnt = b.count[k];
    need = cnt > 0;
    if (b.need_list) {
      const int32_t bx = k / (b.nby * b.nbz), by = (k / b.nbz) % b.nby, bz = k % b.nbz;
      int32_t any = 0;
#pragma unroll
      for (int e = 1; e < 8; ++e) {
        const int ex = e >> 2, ey = (e >> 1) & 1, ez = e & 1;
        const bool in = bx >= ex && by >= ey && bz >= ez;
        any |= b.count[in ? k - (ex * b.nby + ey) * b.nbz - ez : k];
      }
      need = need || any > 0;
    }
  }
  const uint64_t below = (1ull << lane) - 1ull;
  const uint64_t actives = __builtin_amdgcn_ballot_w64(cnt > 0), needs = __builtin_amdgcn_ballot_w64(need);
  int32_t incl = cnt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t y = __shfl_up(incl, off, 64);
    if (lane >= off) incl += y;
  }
  if (lane == 63) {
    wave_total[0][wave] = (int32_t)__builtin_popcountll(actives);
    wave_total[1][wave] = incl;
    wave_total[2][wave] = (int32_t)__builtin_popcountll(needs);
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    int32_t sum = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int32_t t = wave_total[threadIdx.x][w];
      wave_total[threadIdx.x][w] = sum;
      sum += t;
    }
    int32_t* counter = threadIdx.x == 0 ? b.nactive : threadIdx.x == 1 ? b.nsorted : b.nneed;
    first[threadIdx.x] = sum > 0 && counter ? atomicAdd(counter, sum) : 0;
  }
  __syncthreads();
  if (cnt > 0) {
    const int32_t slot = first[0] + wave_total[0][wave] + (int32_t)__builtin_popcountll(actives & below);
    b.active[slot] = k;
    b.slot[k] = slot;
    b.offset[k] = first[1] + wave_total[1][wave] + incl - cnt;
  }
  if (need && b.need_list) {
    b.need_list[first[2] + wave_total[2][wave] + (int32_t)__builtin_popcountll(needs & below)] = k;
    b.need_stamp[k] = b.stamp;
  }
}

// Key and rank of every particle.  The lanes of a wavefront with the same block take
// their ranks from one atomic (the lowest such lane adds the group's size; every lane adds its
// position among the group's lanes); the out-of-bounds lanes of a wavefront reserve their slots of the out-of-bounds list with
// one atomic.  The loop over chunks is uniform across the workgroup, so every lane takes part in
// the ballots.
template <int EDGE>
__global__ void __launch_bounds__(kBlock) k_bin_count(MpmArgs a, BinArgs b) {
  const uint32_t n = (uint32_t)a.count;
  const int lane = (int)(threadIdx.x & 63u);
  const uint64_t below = (1ull << lane) - 1ull;
  const ChunkRange cr = xcd_chunks((n + kBlock - 1) / kBlock);
  for (uint32_t ch = cr.first; ch < cr.end; ch += cr.step) {
    const uint32_t c = ch * kBlock + threadIdx.x;
    const bool valid = c < n;
    int32_t k = -1;
    bool out = false;
    if (valid) {
      float X[3];
      grid_coord(a, a.x + 3 * (size_t)c, X);
      out = stencil_oob(a, X);
      if (!out) {
        const int sx = (int)floorf(X[0] - 0.5f), sy = (int)floorf(X[1] - 0.5f), sz = (int)floorf(X[2] - 0.5f);
        const int bx = sx / EDGE, by = sy / EDGE, bz = sz / EDGE;
        k = (bx * b.nby + by) * b.nbz + bz;
        b.cell[c] = ((sx - bx * EDGE) * EDGE + (sy - by * EDGE)) * EDGE + (sz - bz * EDGE);
      }
    }
    const uint64_t outs = __builtin_amdgcn_ballot_w64(valid && out);
    if (outs) {
      const int first = __builtin_ctzll(outs);
      int32_t slot = 0;
      if (lane == first) slot = atomicAdd(b.noob, (int32_t)__builtin_popcountll(outs));
      slot = __shfl(slot, first, 64);
      if (valid && out) b.oob[slot + __builtin_popcountll(outs & below)] = (int32_t)c;
    }
    // group the lanes by block (register work only), then every group's lowest lane takes the
    // group's ranks with one atomic, all groups' atomics in flight together
    uint64_t todo = __builtin_amdgcn_ballot_w64(k >= 0);
    uint64_t group = 0ull;
    int leader = lane;
    while (todo) {
      const int first = __builtin_ctzll(todo);
      const int32_t kl = __shfl(k, first, 64);
      const uint64_t same = __builtin_amdgcn_ballot_w64(k == kl) & todo;
      if ((same >> lane) & 1ull) {
        group = same;
        leader = first;
      }
      todo &= ~same;
    }
    int32_t first_rank = 0;
    if (k >= 0 && lane == leader) first_rank = atomicAdd(&b.count[k], (int32_t)__builtin_popcountll(group));
    first_rank = __shfl(first_rank, leader, 64);
    const int32_t r = first_rank + (int32_t)__builtin_popcountll(group & below);
    if (valid) {
      b.key[c] = k;
      if (k >= 0) b.rank[c] = r;
    }
  }
}

__global__ void __launch_bounds__(kBlock) k_bin_scatter(int32_t n, BinArgs b) {
  HFSI_CELL_LOOP((uint32_t)n) {
    const int32_t k = b.key[c];
    if (k >= 0) {
      const int32_t pos = b.offset[k] + b.rank[c];
      b.sorted[pos] = (int32_t)c;
      b.scell[pos] = b.cell[c];
    }
  }
}

// Binned P2G scatter of one block of 8^3 nodes, a stencil-base cell at a time (no floating-point atomics).  LDS
// float atomics run at about 1/30 of the rate of integer ones on gfx950 (a probe measured ~190 cycles
// per wavefront instruction per CU with distinct addresses, against ~6 for u32), so the block's
// particles are added with plain read-modify-writes instead:
//   - each wavefront accumulates mass and momentum into a tile of its own (float4 per node);
//   - a chunk of the block's particles is ordered by base cell (u32 LDS atomics give each particle a
//     slot in its cell, a scan of the 512 cell counts the cells' ranges), and the occupied cells are
//     listed by particle count, largest first (a counting sort), so that the 64 cells a wavefront
//     takes together hold similar numbers of particles;
//   - each lane sums the 27 node contributions of its cell's particles in registers (they share the
//     cell's stencil), then adds the sums to the tile.  The lanes' cells are distinct, so for every
//     stencil offset their nodes are distinct, and a compiler barrier after each update keeps a
//     lane's 27 updates in program order (LDS operations of one wavefront complete in issue order):
//     no update reads a node before the wavefront's previous update of it has been written.
// The tile is read and written once per occupied cell and stencil node rather than once per
// particle.  The per-particle operands come staged by k_mpm_p2g_prepare (64 B per particle), and a
// lane loads its next particle's while it adds the current one.  The wavefront tiles are summed in
// wavefront order into the block's tile.  External forces are accumulated by k_mpm_p2g_force.  Two
// wavefronts per workgroup keep a workgroup's LDS (two 16 KB tiles and the cell tables) under 40 KB,
// so that four workgroups share a CU.
constexpr int kP2gThreads = 128;
constexpr int kP2gWaves = kP2gThreads / 64;
constexpr int kP2gChunk = 1024;                      // particles of a block ordered per pass
constexpr int kP2gPerThread = kP2gChunk / kP2gThreads;
constexpr int kBlockCells = Tile<kCoarseEdge>::kCells;
constexpr int kCellsPerThread = kBlockCells / kP2gThreads;
constexpr int kCountBuckets = 8;                     // cells by particle count: >= 8, 7, ..., 1
constexpr size_t kP2gTileBytes = (size_t)kP2gWaves * Tile<kCoarseEdge>::kNodes * sizeof(float4);  // dynamic LDS
static_assert(kP2gWaves == 2 && kBlockCells % kP2gThreads == 0, "the cell scan assumes two wavefronts");
static_assert(kP2gChunk < 65536 && kBlockCells < 65536, "cell ranges and lists are 16-bit");

__device__ inline uint32_t count_bucket(uint32_t c) {
  return c >= (uint32_t)kCountBuckets ? 0u : (uint32_t)kCountBuckets - c;
}

__device__ inline void tile_add(float4* tile, int li, float mw, const float (&md)[3]) {
  float4 t = tile[li];
  t.x += mw;
  t.y += md[0];
  t.z += md[1];
  t.w += md[2];
  tile[li] = t;
  __asm__ __volatile__("" ::: "memory");
}

// First half of the binned P2G, over every particle in particle order: the stress and the affine
// momentum (p2g_prepare), staged for k_mpm_p2g_cells, and the report sums 0..11 (out-of-bounds
// particles included; they are staged too but never scattered).  Particles whose F needs the SVD
// clamp are listed for k_mpm_p2g_prepare_svd instead.
__global__ void __launch_bounds__(kBlock) k_mpm_p2g_prepare(MpmArgs a, BinArgs b) {
  constexpr int NS = 12;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const int lane = (int)(threadIdx.x & 63u);
  HFSI_CELL_LOOP((uint32_t)a.count) {
    P2gPart q;
    const bool done = p2g_prepare<false>(a, c, acc, q);
    if (done) p2g_stage(b.stage + 4 * (size_t)c, q);
    const uint64_t defer = __builtin_amdgcn_ballot_w64(!done);
    if (defer) {
      const int first = __builtin_ctzll(defer);
      int32_t slot = 0;
      if (lane == first) slot = atomicAdd(b.nsvd, (int32_t)__builtin_popcountll(defer));
      slot = __shfl(slot, first, 64);
      if (!done) b.svd[slot + __builtin_popcountll(defer & ((1ull << lane) - 1ull))] = (int32_t)c;
    }
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, kP2gMax);
}

// The listed particles of k_mpm_p2g_prepare with the SVD clamp of F (persisted when it changed).
__global__ void __launch_bounds__(kBlock) k_mpm_p2g_prepare_svd(MpmArgs a, BinArgs b) {
  constexpr int NS = 12;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const int32_t n = *b.nsvd;
  for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t p = (uint32_t)b.svd[i];
    P2gPart q;
    p2g_prepare(a, p, acc, q);
    p2g_stage(b.stage + 4 * (size_t)p, q);
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, kP2gMax);
}

__device__ inline void load_stage(const float4* stage, int32_t p, float4 (&s)[4]) {
  const float4* src = stage + 4 * (size_t)p;
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = src[i];
}

// A block's wavefront tiles, summed in wavefront order, to its tile buffer or onto the grid.
template <int EDGE, int WAVES>
__device__ inline void flush_tiles(const MpmArgs& a, const BinArgs& b, uint32_t ab, int ox0, int oy0, int oz0,
                                   const float4* wave_tiles) {
  constexpr int kNodes = Tile<EDGE>::kNodes, kEdge = Tile<EDGE>::kEdge;
  const uint32_t sx = (uint32_t)a.ny * a.nz, sy = a.nz;
  for (int i = threadIdx.x; i < kNodes; i += 64 * WAVES) {
    float4 v = wave_tiles[i];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      const float4 u = wave_tiles[w * kNodes + i];
      v.x += u.x;
      v.y += u.y;
      v.z += u.z;
      v.w += u.w;
    }
    if (b.tiles) {
      float* T = b.tiles + (size_t)ab * Tile<EDGE>::kStride;
      T[i] = v.x;
      T[kNodes + i] = v.y;
      T[2 * kNodes + i] = v.z;
      T[3 * kNodes + i] = v.w;
      continue;
    }
    const int gx = ox0 + i / (kEdge * kEdge), gy = oy0 + (i / kEdge) % kEdge, gz = oz0 + i % kEdge;
    if (gx >= a.nx || gy >= a.ny || gz >= a.nz) continue;
    const uint32_t node = (uint32_t)gx * sx + (uint32_t)gy * sy + (uint32_t)gz;
    if (v.x != 0.0f) atomicAdd(&a.gm[node], v.x);
    if (v.y != 0.0f) atomicAdd(&a.gv[3 * (size_t)node + 0], v.y);
    if (v.z != 0.0f) atomicAdd(&a.gv[3 * (size_t)node + 1], v.z);
    if (v.w != 0.0f) atomicAdd(&a.gv[3 * (size_t)node + 2], v.w);
  }
}

__global__ void __launch_bounds__(kP2gThreads, 2) k_mpm_p2g_cells(MpmArgs a, BinArgs b) {
  extern __shared__ float4 wave_tiles[];  // [kP2gWaves][Tile<kCoarseEdge>::kNodes]: mass, momentum
  __shared__ uint32_t cell_count[kBlockCells];
  __shared__ uint16_t cell_start[kBlockCells];  // first entry of each cell in order
  __shared__ uint16_t cell_list[kBlockCells];   // occupied cells, largest count first
  __shared__ uint32_t bucket_count[kCountBuckets];
  __shared__ uint32_t bucket_start[kCountBuckets + 1];
  __shared__ uint32_t wave0_total;
  __shared__ int32_t order[kP2gChunk];          // the chunk's particles by cell
  const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63u);
  float4* tile = wave_tiles + (size_t)wave * Tile<kCoarseEdge>::kNodes;
  const ChunkRange cr = xcd_chunks((uint32_t)*b.nactive);
  for (uint32_t ab = cr.first; ab < cr.end; ab += cr.step) {
    const int32_t k = b.active[ab];
    const int ox0 = (k / (b.nby * b.nbz)) * kCoarseEdge, oy0 = ((k / b.nbz) % b.nby) * kCoarseEdge,
              oz0 = (k % b.nbz) * kCoarseEdge;
    for (int i = threadIdx.x; i < kP2gWaves * Tile<kCoarseEdge>::kNodes; i += kP2gThreads) wave_tiles[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    const int32_t beg = b.offset[k], cnt = b.count[k];
    for (int32_t c0 = 0; c0 < cnt; c0 += kP2gChunk) {
      const int32_t n = min(kP2gChunk, cnt - c0);
      for (int i = threadIdx.x; i < kBlockCells; i += kP2gThreads) cell_count[i] = 0u;
      if (threadIdx.x < kCountBuckets) bucket_count[threadIdx.x] = 0u;
      __syncthreads();
      uint32_t slot[kP2gPerThread];
#pragma unroll
      for (int j = 0; j < kP2gPerThread; ++j) {
        const int t = (int)threadIdx.x + j * kP2gThreads;
        slot[j] = 0u;
        if (t < n) {
          const uint32_t cl = (uint32_t)b.scell[beg + c0 + t];
          slot[j] = (cl << 16) | atomicAdd(&cell_count[cl], 1u);
        }
      }
      __syncthreads();
      // cell ranges: exclusive scan of the counts (kCellsPerThread consecutive cells per thread),
      // and each occupied cell's rank within its count bucket
      const int cell0 = (int)threadIdx.x * kCellsPerThread;
      uint32_t cc[kCellsPerThread], brank[kCellsPerThread], run = 0u;
#pragma unroll
      for (int i = 0; i < kCellsPerThread; ++i) {
        cc[i] = cell_count[cell0 + i];
        run += cc[i];
        brank[i] = cc[i] > 0u ? atomicAdd(&bucket_count[count_bucket(cc[i])], 1u) : 0u;
      }
      uint32_t incl = run;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
      }
      if (wave == 0 && lane == 63) wave0_total = incl;
      __syncthreads();
      uint32_t pre = incl - run + (wave == 1 ? wave0_total : 0u);
#pragma unroll
      for (int i = 0; i < kCellsPerThread; ++i) {
        cell_start[cell0 + i] = (uint16_t)pre;
        pre += cc[i];
      }
      if (threadIdx.x == 0) {
        uint32_t s0 = 0u;
        for (int q = 0; q < kCountBuckets; ++q) {
          bucket_start[q] = s0;
          s0 += bucket_count[q];
        }
        bucket_start[kCountBuckets] = s0;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kCellsPerThread; ++i)
        if (cc[i] > 0u) cell_list[bucket_start[count_bucket(cc[i])] + brank[i]] = (uint16_t)(cell0 + i);
#pragma unroll
      for (int j = 0; j < kP2gPerThread; ++j) {
        const int t = (int)threadIdx.x + j * kP2gThreads;
        if (t < n) order[cell_start[slot[j] >> 16] + (slot[j] & 0xffffu)] = b.sorted[beg + c0 + t];
      }
      __syncthreads();
      const uint32_t ncells = bucket_start[kCountBuckets];
      for (uint32_t g0 = (uint32_t)wave * 64u; g0 < ncells; g0 += kP2gThreads) {
        const uint32_t li = g0 + (uint32_t)lane;
        const int cl = li < ncells ? (int)cell_list[li] : -1;
        const uint32_t np = cl >= 0 ? cell_count[cl] : 0u, s = cl >= 0 ? (uint32_t)cell_start[cl] : 0u;
        float acc[27][4];
#pragma unroll
        for (int o = 0; o < 27; ++o) acc[o][0] = acc[o][1] = acc[o][2] = acc[o][3] = 0.0f;
        float4 cur[4] = {};
        if (np > 0u) load_stage(b.stage, order[s], cur);
        for (uint32_t i = 0; i < np; ++i) {
          float4 nxt[4] = {};
          if (i + 1u < np) load_stage(b.stage, order[s + i + 1u], nxt);
          P2gPart q;
          p2g_unstage(cur, q);
          p2g_scatter(a, q, [&](int ox, int oy, int oz, float mw, const float (&md)[3], float) {
            float* t = acc[(ox * 3 + oy) * 3 + oz];
            t[0] += mw;
            t[1] += md[0];
            t[2] += md[1];
            t[3] += md[2];
          });
#pragma unroll
          for (int r = 0; r < 4; ++r) cur[r] = nxt[r];
        }
        if (np > 0u) {
          const int lx = cl / (kCoarseEdge * kCoarseEdge), ly = (cl / kCoarseEdge) % kCoarseEdge, lz = cl % kCoarseEdge;
#pragma unroll
          for (int ox = 0; ox < 3; ++ox)
#pragma unroll
            for (int oy = 0; oy < 3; ++oy)
#pragma unroll
              for (int oz = 0; oz < 3; ++oz) {
                const float* t = acc[(ox * 3 + oy) * 3 + oz];
                const float md[3] = {t[1], t[2], t[3]};
                tile_add(tile, ((lx + ox) * Tile<kCoarseEdge>::kEdge + (ly + oy)) * Tile<kCoarseEdge>::kEdge + (lz + oz), t[0], md);
              }
        }
      }
      __syncthreads();  // the cell tables and order are rewritten by the next chunk
    }
    flush_tiles<kCoarseEdge, kP2gWaves>(a, b, ab, ox0, oy0, oz0, wave_tiles);
    __syncthreads();  // the wave tiles are cleared for the next block
  }
}

// The same scatter of one block of 4^3 nodes: lane c of a wavefront takes cell c, over all chunks, so
// the cells need no ordering by count and a cell's sums reach the tile once.  The bound is the chain
// of dependent steps of a cell's particles, hence three wavefronts on a block, one per plane ox of
// the stencil: the chain is a third as long, and 36 sums per lane instead of 108 let four wavefronts
// share a SIMD.  The second and third wavefront's operand loads hit the cache.  (Staging a chunk's
// operands in LDS in cell order instead was 1 us faster for 32^3 particles and 11 us slower for 100^3.)
// 32^3 particles, 4.6 per cell: 66 us with 8^3 blocks, 12.3 us.
constexpr int kFineWaves = 3;
constexpr int kFineThreads = 64 * kFineWaves;
constexpr int kFinePerThread = 5;
constexpr int kFineChunk = kFinePerThread * kFineThreads;  // particles of a block ordered per pass
static_assert(Tile<kFineEdge>::kCells == 64, "a block's cells are the lanes of a wavefront");
static_assert(kFineChunk < 65536, "a particle's place in its cell is kept in 16 bits");

// The contributions of a particle to plane ox of its stencil (p2g_scatter's arithmetic).
template <typename Sink>
__device__ inline void p2g_scatter_plane(const MpmArgs& a, const P2gPart& q, int ox, Sink sink) {
  const float w0 = ox == 0 ? q.w[0][0] : ox == 1 ? q.w[0][1] : q.w[0][2];
  const float dp0 = ((float)ox - q.fx[0]) * a.dx[0];
#pragma unroll
  for (int oy = 0; oy < 3; ++oy)
#pragma unroll
    for (int oz = 0; oz < 3; ++oz) {
      const float wt = w0 * q.w[1][oy] * q.w[2][oz];
      const float dp1 = ((float)oy - q.fx[1]) * a.dx[1];
      const float dp2 = ((float)oz - q.fx[2]) * a.dx[2];
      float md[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) md[d] = wt * (q.mom[d] + (q.aff[d][0] * dp0 + q.aff[d][1] * dp1 + q.aff[d][2] * dp2));
      sink(oy, oz, wt * q.m, md);
    }
}

__global__ void __launch_bounds__(kFineThreads, 4) k_mpm_p2g_fine(MpmArgs a, BinArgs b) {
  __shared__ float4 wave_tiles[kFineWaves * Tile<kFineEdge>::kNodes];  // mass, momentum
  __shared__ uint32_t cell_count[Tile<kFineEdge>::kCells];
  __shared__ uint32_t cell_start[Tile<kFineEdge>::kCells];  // first entry of each cell in order
  __shared__ int32_t order[kFineChunk];          // the chunk's particles by cell
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
  float4* tile = wave_tiles + wave * Tile<kFineEdge>::kNodes;
  const ChunkRange cr = xcd_chunks((uint32_t)*b.nactive);
  for (uint32_t ab = cr.first; ab < cr.end; ab += cr.step) {
    const int32_t k = b.active[ab];
    const int ox0 = (k / (b.nby * b.nbz)) * kFineEdge, oy0 = ((k / b.nbz) % b.nby) * kFineEdge,
              oz0 = (k % b.nbz) * kFineEdge;
    for (int i = threadIdx.x; i < kFineWaves * Tile<kFineEdge>::kNodes; i += kFineThreads) wave_tiles[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    const int32_t beg = b.offset[k], cnt = b.count[k];
    float acc[9][4];
#pragma unroll
    for (int o = 0; o < 9; ++o) acc[o][0] = acc[o][1] = acc[o][2] = acc[o][3] = 0.0f;
    for (int32_t c0 = 0; c0 < cnt; c0 += kFineChunk) {
      const int32_t n = min(kFineChunk, cnt - c0);
      if (threadIdx.x < Tile<kFineEdge>::kCells) cell_count[threadIdx.x] = 0u;
      __syncthreads();
      uint32_t place[kFinePerThread];
      int32_t part[kFinePerThread];
#pragma unroll
      for (int j = 0; j < kFinePerThread; ++j) {
        const int t = (int)threadIdx.x + j * kFineThreads;
        place[j] = t < n ? (uint32_t)b.scell[beg + c0 + t] : 0u;
        part[j] = t < n ? b.sorted[beg + c0 + t] : 0;
      }
#pragma unroll
      for (int j = 0; j < kFinePerThread; ++j) {
        const int t = (int)threadIdx.x + j * kFineThreads;
        if (t < n) place[j] = (place[j] << 16) | atomicAdd(&cell_count[place[j]], 1u);
      }
      __syncthreads();
      // every wavefront scans the 64 counts: lane c keeps the range of cell c
      const uint32_t np = cell_count[lane];
      uint32_t incl = np;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
      }
      const uint32_t s = incl - np;
      if (wave == 0) cell_start[lane] = s;
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kFinePerThread; ++j) {
        const int t = (int)threadIdx.x + j * kFineThreads;
        if (t < n) order[cell_start[place[j] >> 16] + (place[j] & 0xffffu)] = part[j];
      }
      __syncthreads();
      float4 cur[4] = {};
      if (np > 0u) load_stage(b.stage, order[s], cur);
      for (uint32_t i = 0; i < np; ++i) {
        float4 nxt[4] = {};
        if (i + 1u < np) load_stage(b.stage, order[s + i + 1u], nxt);
        P2gPart q;
        p2g_unstage(cur, q);
        p2g_scatter_plane(a, q, wave, [&](int oy, int oz, float mw, const float (&md)[3]) {
          float* t = acc[oy * 3 + oz];
          t[0] += mw;
          t[1] += md[0];
          t[2] += md[1];
          t[3] += md[2];
        });
#pragma unroll
        for (int r = 0; r < 4; ++r) cur[r] = nxt[r];
      }
      __syncthreads();  // the cell tables and order are rewritten by the next chunk
    }
    {
      const int lx = lane / (kFineEdge * kFineEdge), ly = (lane / kFineEdge) % kFineEdge, lz = lane % kFineEdge;
#pragma unroll
      for (int oy = 0; oy < 3; ++oy)
#pragma unroll
        for (int oz = 0; oz < 3; ++oz) {
          const float* t = acc[oy * 3 + oz];
          const float md[3] = {t[1], t[2], t[3]};
          tile_add(tile, ((lx + wave) * Tile<kFineEdge>::kEdge + (ly + oy)) * Tile<kFineEdge>::kEdge + (lz + oz), t[0], md);
        }
    }
    __syncthreads();
    flush_tiles<kFineEdge, kFineWaves>(a, b, ab, ox0, oy0, oz0, wave_tiles);
    __syncthreads();  // the wave tiles are cleared for the next block
  }
}

// External-force part of the binned P2G: f += w f_ext over the 27 nodes of every particle with a
// non-zero force (fixed particles carry none), LDS atomics into a block tile.  A block without
// such particles writes no force components and is flagged so that the grid update skips them.
template <int EDGE>
__global__ void __launch_bounds__(kBlock) k_mpm_p2g_force(MpmArgs a, BinArgs b) {
  constexpr int kNodes = Tile<EDGE>::kNodes, kEdge = Tile<EDGE>::kEdge;
  __shared__ float tf[3][kNodes];
  __shared__ int32_t any;
  const uint32_t sx = (uint32_t)a.ny * a.nz, sy = a.nz;
  const ChunkRange cr = xcd_chunks((uint32_t)*b.nactive);
  for (uint32_t ab = cr.first; ab < cr.end; ab += cr.step) {
    const int32_t k = b.active[ab];
    const int ox0 = (k / (b.nby * b.nbz)) * EDGE, oy0 = ((k / b.nbz) % b.nby) * EDGE,
              oz0 = (k % b.nbz) * EDGE;
    if (threadIdx.x == 0) any = 0;
    for (int i = threadIdx.x; i < kNodes; i += kBlock) tf[0][i] = tf[1][i] = tf[2][i] = 0.0f;
    __syncthreads();
    const int32_t beg = b.offset[k], cnt = b.count[k];
    for (int32_t t = threadIdx.x; t < cnt; t += kBlock) {
      const uint32_t p = (uint32_t)b.sorted[beg + t];
      if (a.fixed && a.fixed[p] != 0) continue;
      const float fe[3] = {a.f_ext[3 * (size_t)p], a.f_ext[3 * (size_t)p + 1], a.f_ext[3 * (size_t)p + 2]};
      if (fe[0] == 0.0f && fe[1] == 0.0f && fe[2] == 0.0f) continue;
      any = 1;
      float X[3], w[3][3];
      int base[3];
      grid_coord(a, a.x + 3 * (size_t)p, X);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        base[d] = (int)floorf(X[d] - 0.5f);
        bspline(X[d] - (float)base[d], w[d]);
      }
      const int lx = base[0] - ox0, ly = base[1] - oy0, lz = base[2] - oz0;
#pragma unroll
      for (int ox = 0; ox < 3; ++ox)
#pragma unroll
        for (int oy = 0; oy < 3; ++oy)
#pragma unroll
          for (int oz = 0; oz < 3; ++oz) {
            const float wt = w[0][ox] * w[1][oy] * w[2][oz];
            const int li = ((lx + ox) * kEdge + (ly + oy)) * kEdge + (lz + oz);
#pragma unroll
            for (int d = 0; d < 3; ++d)
              if (fe[d] != 0.0f) atomicAdd(&tf[d][li], wt * fe[d]);
          }
    }
    __syncthreads();
    if (any) {
      if (b.tiles) {
        float* T = b.tiles + (size_t)ab * Tile<EDGE>::kStride;
        for (int i = threadIdx.x; i < kNodes; i += kBlock) {
#pragma unroll
          for (int d = 0; d < 3; ++d) T[(4 + d) * kNodes + i] = tf[d][i];
        }
      } else {
        for (int i = threadIdx.x; i < kNodes; i += kBlock) {
          const int tz = i % kEdge, ty = (i / kEdge) % kEdge, tx = i / (kEdge * kEdge);
          const int gx = ox0 + tx, gy = oy0 + ty, gz = oz0 + tz;
          if (gx >= a.nx || gy >= a.ny || gz >= a.nz) continue;
          const uint32_t node = (uint32_t)gx * sx + (uint32_t)gy * sy + (uint32_t)gz;
#pragma unroll
          for (int d = 0; d < 3; ++d)
            if (tf[d][i] != 0.0f) atomicAdd(&a.gf[3 * (size_t)node + d], tf[d][i]);
        }
      }
    }
    if (threadIdx.x == 0 && b.block_force) b.block_force[ab] = any;
    __syncthreads();  // the tile and the flag are reused by the next block
  }
}

// Blocks of the previous step's need list that this step does not list: zero their nodes (every
// node outside the need list is zero, and the grid update rewrites every node of the listed blocks).
// A wavefront takes 64 nodes of a block: units first, first + step, ... of the list.
template <int EDGE>
__device__ inline void clear_stale(const MpmArgs& a, const BinArgs& b, uint32_t first, uint32_t step) {
  constexpr uint32_t kUnits = Tile<EDGE>::kCells / 64;
  const uint32_t n = (uint32_t)*b.nprev * kUnits;
  for (uint32_t w = first; w < n; w += step) {
    const int32_t B = b.prev_need[w / kUnits];
    if (b.need_stamp[B] == b.stamp) continue;
    const int t = (int)(w % kUnits * 64 + (threadIdx.x & 63u));
    const int gx = (B / (b.nby * b.nbz)) * EDGE + t / (EDGE * EDGE), gy = ((B / b.nbz) % b.nby) * EDGE + (t / EDGE) % EDGE,
              gz = (B % b.nbz) * EDGE + t % EDGE;
    if (gx >= a.nx || gy >= a.ny || gz >= a.nz) continue;
    const size_t node = ((size_t)gx * a.ny + gy) * a.nz + gz;
    a.gm[node] = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      a.gv[3 * node + d] = 0.0f;
      a.gf[3 * node + d] = 0.0f;
    }
  }
}

// Grid update (neo_hookean_mpm.py:803-817).  Totals 12..19.
__global__ void __launch_bounds__(kBlock) k_mpm_grid(MpmArgs a) {
  constexpr int NS = 8;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const uint32_t n = (uint32_t)a.nx * a.ny * a.nz;
  HFSI_CELL_LOOP(n) {
    const float m = a.gm[c];
    if (!(m > 1.0e-20f)) continue;
    float v[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      v[d] = a.gv[3 * (size_t)c + d] / m;
      v[d] += a.dt * a.gf[3 * (size_t)c + d] / m;
      acc[d] += (double)(m * v[d]);
      v[d] *= a.damping;
      a.gv[3 * (size_t)c + d] = v[d];
      acc[3 + d] += (double)(m * v[d]);
    }
    acc[6] += 1.0;
    acc[7] = fmax(acc[7], (double)sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, kGridMax);
}

// Grid update of the tile path: every node of a listed block sums the tiles
// that cover it (its own block's and, within 2 nodes of a low face, the lower
// neighbours'), in a fixed order, then updates as k_mpm_grid and writes mass,
// velocity and force.  Nodes of listed blocks without mass get the raw sums
// (zero), as the cleared grid has.  Totals 12..19.  One wavefront per 64 nodes of a block; the
// (up to) eight tiles' values are loaded together and added afterwards, so that a node costs one
// memory round trip after the list's, not eight.  The last kStaleGroups workgroups clear the nodes
// of the blocks that only the previous step listed.
constexpr uint32_t kStaleGroups = 64;

template <int EDGE>
__global__ void __launch_bounds__(kBlock) k_mpm_grid_gather(MpmArgs a, BinArgs b) {
  constexpr int NS = 8;
  constexpr int kWaves = kBlock / 64, kNodes = Tile<EDGE>::kNodes, kEdge = Tile<EDGE>::kEdge;
  constexpr uint32_t kUnits = Tile<EDGE>::kCells / 64;
  __shared__ double lds[NS * (kBlock / 64)];
  const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63u);
  const uint32_t groups = gridDim.x - kStaleGroups;
  if (blockIdx.x >= groups) {
    clear_stale<EDGE>(a, b, (blockIdx.x - groups) * kWaves + (uint32_t)wave, kStaleGroups * kWaves);
    return;
  }
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const uint32_t nneed = (uint32_t)*b.nneed * kUnits;
  const ChunkRange cr = xcd_chunks((nneed + kWaves - 1) / kWaves, groups);
  for (uint32_t ch = cr.first; ch < cr.end; ch += cr.step) {
    const uint32_t w = ch * kWaves + (uint32_t)wave;
    if (w >= nneed) break;
    const int32_t B = b.need_list[w / kUnits];
    const int t = (int)(w % kUnits) * 64 + lane;
    const int lx = t / (EDGE * EDGE), ly = (t / EDGE) % EDGE, lz = t % EDGE;
    const int32_t bx = B / (b.nby * b.nbz), by = (B / b.nbz) % b.nby, bz = B % b.nbz;
    const int gx = bx * EDGE + lx, gy = by * EDGE + ly, gz = bz * EDGE + lz;
    if (gx >= a.nx || gy >= a.ny || gz >= a.nz) continue;
    int32_t slot[8];  // of the covering tile, or -1
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ex = e >> 2, ey = (e >> 1) & 1, ez = e & 1;
      const bool in = bx >= ex && by >= ey && bz >= ez;
      const int32_t k = in ? B - (ex * b.nby + ey) * b.nbz - ez : B;
      const bool covers = in && (!ex || lx < 2) && (!ey || ly < 2) && (!ez || lz < 2) && b.count[k] > 0;
      slot[e] = covers ? b.slot[k] : -1;
    }
    float tv[8][4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ex = e >> 2, ey = (e >> 1) & 1, ez = e & 1;
      const int ti = ((lx + ex * EDGE) * kEdge + (ly + ey * EDGE)) * kEdge + (lz + ez * EDGE);
#pragma unroll
      for (int c = 0; c < 4; ++c) tv[e][c] = 0.0f;
      if (slot[e] >= 0) {
        const float* T = b.tiles + (size_t)slot[e] * Tile<EDGE>::kStride + ti;
#pragma unroll
        for (int c = 0; c < 4; ++c) tv[e][c] = T[c * kNodes];
      }
    }
    float f[3] = {0.0f, 0.0f, 0.0f};
    if (b.has_force) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int ex = e >> 2, ey = (e >> 1) & 1, ez = e & 1;
        const int ti = ((lx + ex * EDGE) * kEdge + (ly + ey * EDGE)) * kEdge + (lz + ez * EDGE);
        if (slot[e] < 0 || !b.block_force[slot[e]]) continue;
        const float* T = b.tiles + (size_t)slot[e] * Tile<EDGE>::kStride + ti;
#pragma unroll
        for (int d = 0; d < 3; ++d) f[d] += T[(4 + d) * kNodes];
      }
    }
    float m = 0.0f, p[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      m += tv[e][0];
#pragma unroll
      for (int d = 0; d < 3; ++d) p[d] += tv[e][1 + d];
    }
    const size_t node = ((size_t)gx * a.ny + gy) * a.nz + gz;
    a.gm[node] = m;
    float v[3] = {p[0], p[1], p[2]};
    if (m > 1.0e-20f) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        v[d] = p[d] / m;
        v[d] += a.dt * f[d] / m;
        acc[d] += (double)(m * v[d]);
        v[d] *= a.damping;
        acc[3 + d] += (double)(m * v[d]);
      }
      acc[6] += 1.0;
      acc[7] = fmax(acc[7], (double)sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      a.gv[3 * node + d] = v[d];
      a.gf[3 * node + d] = f[d];
    }
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, kGridMax);
}

__device__ inline void update_surface(const MpmArgs& a, uint32_t p) {
  if (!a.rest_area) return;
  const float ra = a.rest_area[p];
  const float* rn = a.rest_normal + 3 * (size_t)p;
  if (!(ra > 0.0f) || !(sqrtf(rn[0] * rn[0] + rn[1] * rn[1] + rn[2] * rn[2]) > 1.0e-12f)) return;
  M3 F;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) F.a[i][j] = (double)a.F[9 * (size_t)p + 3 * i + j];
  const double J = mdet(F);
  if (!(J > 1.0e-12)) return;
  const M3 FiT = minv_t(F, J);
  double av[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) av[i] = J * (FiT.a[i][0] * rn[0] + FiT.a[i][1] * rn[1] + FiT.a[i][2] * rn[2]);
  const double s = sqrt(av[0] * av[0] + av[1] * av[1] + av[2] * av[2]);
  if (!(s > 1.0e-12)) return;
#pragma unroll
  for (int i = 0; i < 3; ++i) a.normal[3 * (size_t)p + i] = (float)(av[i] / s);
  a.area[p] = (float)((double)ra * s);
}

__device__ inline void g2p_report(const MpmArgs& a, uint32_t p, double (&acc)[21]);

// The part of a particle's G2P that needs no grid: the reset of a fixed particle and the surface.
__device__ inline void g2p_rest(const MpmArgs& a, uint32_t p, bool fixed) {
  if (fixed) {
    float* vp = a.v + 3 * (size_t)p;
    float* Cp = a.C + 9 * (size_t)p;
    float* Fp = a.F + 9 * (size_t)p;
#pragma unroll
    for (int d = 0; d < 3; ++d) vp[d] = 0.0f;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      Cp[i] = 0.0f;
      Fp[i] = (i % 4 == 0) ? 1.0f : 0.0f;
    }
  }
  update_surface(a, p);
}

// G2P of one particle (neo_hookean_mpm.py:819-874) with the grid velocity of node base + (ox, oy, oz)
// from vel(base, ox, oy, oz, out[3]); with SUMS, its report totals 20..40 into acc (g2p_report).
template <bool SUMS, typename Vel>
__device__ inline void g2p_particle(const MpmArgs& a, uint32_t p, double (&acc)[21], Vel vel) {
  float* xp = a.x + 3 * (size_t)p;
  float X[3];
  grid_coord(a, xp, X);
  const bool fixed = a.fixed && a.fixed[p] != 0;
  if (!stencil_oob(a, X)) {
    int base[3];
    float fx[3], w[3][3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      base[d] = (int)floorf(X[d] - 0.5f);
      fx[d] = X[d] - (float)base[d];
      bspline(fx[d], w[d]);
    }
    float nv[3] = {0.0f, 0.0f, 0.0f};
    float nC[3][3] = {};
    const float s0 = 4.0f / (a.dx[0] * a.dx[0]), s1 = 4.0f / (a.dx[1] * a.dx[1]), s2 = 4.0f / (a.dx[2] * a.dx[2]);
#pragma unroll
    for (int ox = 0; ox < 3; ++ox)
#pragma unroll
      for (int oy = 0; oy < 3; ++oy)
#pragma unroll
        for (int oz = 0; oz < 3; ++oz) {
          const float wt = w[0][ox] * w[1][oy] * w[2][oz];
          const float g0 = s0 * ((float)ox - fx[0]) * a.dx[0];
          const float g1 = s1 * ((float)oy - fx[1]) * a.dx[1];
          const float g2 = s2 * ((float)oz - fx[2]) * a.dx[2];
          float gvn[3];
          vel(base, ox, oy, oz, gvn);
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const float gvd = gvn[d];
            nv[d] += wt * gvd;
            nC[d][0] += wt * gvd * g0;
            nC[d][1] += wt * gvd * g1;
            nC[d][2] += wt * gvd * g2;
          }
        }
    if (!fixed) {
      float* vp = a.v + 3 * (size_t)p;
      float* Cp = a.C + 9 * (size_t)p;
      float* Fp = a.F + 9 * (size_t)p;
      float Fo[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) Fo[i] = Fp[i];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        vp[d] = nv[d];
        xp[d] = xp[d] + a.dt * nv[d];
#pragma unroll
        for (int e = 0; e < 3; ++e) Cp[3 * d + e] = nC[d][e];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          float acc_f = 0.0f;
#pragma unroll
          for (int k = 0; k < 3; ++k) acc_f += ((i == k ? 1.0f : 0.0f) + a.dt * nC[i][k]) * Fo[3 * k + j];
          Fp[3 * i + j] = acc_f;
        }
    }
  }
  g2p_rest(a, p, fixed);
  if (SUMS) g2p_report(a, p, acc);
}

// Report sums 20..40 of one particle after its G2P update: the region displacement and velocity
// sums and counts, and the current and rest position sums of the particles inside the grid.
__device__ inline void g2p_report(const MpmArgs& a, uint32_t p, double (&acc)[21]) {
  // every load first (one memory round trip), then the sums
  float xp[3], rx[3], vp[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    xp[d] = a.x[3 * (size_t)p + d];
    rx[d] = a.rest_x[3 * (size_t)p + d];
    vp[d] = a.v[3 * (size_t)p + d];
  }
  const int region = a.region ? a.region[p] : 0;
  float Xn[3];
  grid_coord(a, xp, Xn);
  if (!stencil_oob(a, Xn)) {
    int slot = -1;
    if (region == a.primary)
      slot = 0;
    else if (region == a.secondary)
      slot = 1;
    // region sums by select (a register array indexed by the slot would live in scratch memory)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double disp = (double)(xp[d] - rx[d]), vel = (double)vp[d];
      acc[d] += slot == 0 ? disp : 0.0;
      acc[3 + d] += slot == 0 ? vel : 0.0;
      acc[6 + d] += slot == 1 ? disp : 0.0;
      acc[9 + d] += slot == 1 ? vel : 0.0;
    }
    acc[12] += slot == 0 ? 1.0 : 0.0;
    acc[13] += slot == 1 ? 1.0 : 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      acc[14 + d] += (double)xp[d];
      acc[17 + d] += (double)rx[d];
    }
    acc[20] += 1.0;
  }
}

// G2P over all particles, grid velocities from global memory.  Totals 20..40.
__global__ void __launch_bounds__(kBlock) k_mpm_g2p(MpmArgs a) {
  constexpr int NS = 21;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  const uint32_t n = (uint32_t)a.count;
  const uint32_t sx = (uint32_t)a.ny * a.nz, sy = a.nz;
  auto vel = [&](const int (&base)[3], int ox, int oy, int oz, float (&out)[3]) {
    const uint32_t node = (uint32_t)(base[0] + ox) * sx + (uint32_t)(base[1] + oy) * sy + (uint32_t)(base[2] + oz);
#pragma unroll
    for (int d = 0; d < 3; ++d) out[d] = a.gv[3 * (size_t)node + d];
  };
  HFSI_CELL_LOOP(n) { g2p_particle<true>(a, c, acc, vel); }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, 0ull);
}

// G2P of the binned path: per active block, the grid velocities its particles' stencils reach
// are staged in LDS and the block's particles gather from there.  The last kOobGroups workgroups take
// the out-of-bounds particles (no gather: fixed-particle reset and surface update; they stay outside
// the grid, so they add nothing to the report sums).  The report sums are k_mpm_g2p_sums'.
constexpr uint32_t kOobGroups = 16;

template <int EDGE>
__global__ void __launch_bounds__(kBlock, 4) k_mpm_g2p_binned(MpmArgs a, BinArgs b) {
  constexpr int kNodes = Tile<EDGE>::kNodes, kEdge = Tile<EDGE>::kEdge;
  __shared__ float tv[3][kNodes];
  double none[21];  // report sums: k_mpm_g2p_sums
  const uint32_t sx = (uint32_t)a.ny * a.nz, sy = a.nz;
  const uint32_t groups = gridDim.x - kOobGroups;
  if (blockIdx.x >= groups) {
    const int32_t n = *b.noob;
    for (int32_t i = (int32_t)((blockIdx.x - groups) * kBlock + threadIdx.x); i < n; i += (int32_t)kOobGroups * kBlock) {
      const uint32_t p = (uint32_t)b.oob[i];
      g2p_rest(a, p, a.fixed && a.fixed[p] != 0);
    }
    return;
  }
  const ChunkRange cr = xcd_chunks((uint32_t)*b.nactive, groups);
  for (uint32_t ab = cr.first; ab < cr.end; ab += cr.step) {
    const int32_t k = b.active[ab];
    const int ox0 = (k / (b.nby * b.nbz)) * EDGE, oy0 = ((k / b.nbz) % b.nby) * EDGE,
              oz0 = (k % b.nbz) * EDGE;
    for (int i = threadIdx.x; i < kNodes; i += kBlock) {
      const int tz = i % kEdge, ty = (i / kEdge) % kEdge, tx = i / (kEdge * kEdge);
      const int gx = ox0 + tx, gy = oy0 + ty, gz = oz0 + tz;
      const bool inside = gx < a.nx && gy < a.ny && gz < a.nz;
      const size_t node = inside ? (size_t)gx * sx + (size_t)gy * sy + (size_t)gz : 0;
#pragma unroll
      for (int d = 0; d < 3; ++d) tv[d][i] = inside ? a.gv[3 * node + d] : 0.0f;
    }
    __syncthreads();
    auto vel = [&](const int (&base)[3], int ox, int oy, int oz, float (&out)[3]) {
      const int li = ((base[0] - ox0 + ox) * kEdge + (base[1] - oy0 + oy)) * kEdge + (base[2] - oz0 + oz);
#pragma unroll
      for (int d = 0; d < 3; ++d) out[d] = tv[d][li];
    };
    const int32_t beg = b.offset[k], cnt = b.count[k];
    for (int32_t t = threadIdx.x; t < cnt; t += kBlock) g2p_particle<false>(a, (uint32_t)b.sorted[beg + t], none, vel);
    __syncthreads();  // the velocity tile is reloaded for the next block
  }
}

// Report totals 20..40 of the binned G2P, over every particle in particle order after the update.
// A pass of its own: in the gather kernel the float64 sums would hold registers through the whole
// particle update and halve the workgroups resident per CU.
__global__ void __launch_bounds__(kBlock) k_mpm_g2p_sums(MpmArgs a) {
  constexpr int NS = 21;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = 0.0;
  HFSI_CELL_LOOP((uint32_t)a.count) { g2p_report(a, c, acc); }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, 0ull);
}

// Radial stretch and the final report snapshot (neo_hookean_mpm.py:876-959).
__global__ void __launch_bounds__(kBlock) k_mpm_radial(MpmArgs a) {
  constexpr int NS = 3;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS] = {0.0, 0.0, 0.0};
  const double cnt = fmax(a.totals[T_CCNT], 1.0);
  const double cc[3] = {a.totals[T_CCUR] / cnt, a.totals[T_CCUR + 1] / cnt, a.totals[T_CCUR + 2] / cnt};
  const double rc[3] = {a.totals[T_CREST] / cnt, a.totals[T_CREST + 1] / cnt, a.totals[T_CREST + 2] / cnt};
  const uint32_t n = (uint32_t)a.count;
  HFSI_CELL_LOOP(n) {
    const float* xp = a.x + 3 * (size_t)c;
    float X[3];
    grid_coord(a, xp, X);
    if (stencil_oob(a, X)) continue;
    const float* rx = a.rest_x + 3 * (size_t)c;
    double rr = 0.0, cr = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      rr += ((double)rx[d] - rc[d]) * ((double)rx[d] - rc[d]);
      cr += ((double)xp[d] - cc[d]) * ((double)xp[d] - cc[d]);
    }
    rr = sqrt(rr);
    if (rr > 1.0e-12) {
      const double st = sqrt(cr) / rr;
      acc[0] += st;
      acc[1] += 1.0;
      acc[2] = fmax(acc[2], fabs(st - 1.0));
    }
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, kRadialMax);

}


// Report snapshot (neo_hookean_mpm.py:899-959) from the stage totals, run by
// the finishing workgroup of the radial-stretch reduction.
struct FinMpmReport {
  const double* totals;
  double* report;
  float dt;
  __device__ void operator()(const double*) const {
    const double* t = totals;
    double* R = report;
    double e[3], diff2 = 0.0, en = 0.0;
    for (int d = 0; d < 3; ++d) {
      e[d] = t[T_PMOM + d] + (double)dt * t[T_FEXT + d];
      en += e[d] * e[d];
      diff2 += (t[T_TRANS + d] - e[d]) * (t[T_TRANS + d] - e[d]);
    }
    const double den = fmax(fmax(sqrt(en), sqrt(t[T_PSQ])), 1.0e-20);
    R[0] = t[T_MASS];
    R[1] = t[T_VOL];
    for (int d = 0; d < 3; ++d) {
      R[2 + d] = t[T_PMOM + d];
      R[5 + d] = t[T_GMOM + d];
      R[8 + d] = t[T_FEXT + d];
      R[16 + d] = t[T_PDISP + d];
      R[19 + d] = t[T_PVEL + d];
      R[22 + d] = t[T_SDISP + d];
      R[25 + d] = t[T_SVEL + d];
    }
    R[11] = sqrt(diff2) / den;
    R[12] = t[T_MAXV];
    R[13] = t[T_MAXJ];
    R[14] = t[T_RSUM];
    R[15] = t[T_RMAX];
    R[28] = t[T_ACTIVE];
    R[29] = t[T_OOB];
    R[30] = t[T_CLAMP];
    R[31] = t[T_RCNT];
    R[32] = t[T_PCNT];
    R[33] = t[T_SCNT];
  }
};

// ---------------------------------------------------------------------------
// Particle set-up and loads (float32, the reference's operation order)
// ---------------------------------------------------------------------------

struct LayeredArgs {
  const float* centroid;  // [faces][3]
  const float* normal;    // [faces][3]
  const float* area;      // [faces]
  const int32_t* face_region;
  int32_t faces, layers, primary, secondary, fixed_region;
  float density, t_primary, t_secondary;
};

// _initialize_layered_tri_surface_kernel (neo_hookean_mpm.py:231-294): particle p = face * layers + layer
// sits at centroid + normal * (((layer + 0.5) / layers - 0.5) * thickness) with area / layers of the
// face's area and that times the thickness as volume; fixed-region faces take the primary thickness and
// fix their particles.  Region masses (slots 0, 1) reduced in float64.
__global__ void __launch_bounds__(kBlock) k_mpm_layered_init(MpmArgs a, LayeredArgs L) {
#pragma clang fp contract(off)  // separate roundings, as the reference writes the expressions
  constexpr int NS = 2;
  __shared__ double lds[NS * (kBlock / 64)];
  double acc[NS] = {0.0, 0.0};
  const int32_t n = L.faces * L.layers;
  float* mass = const_cast<float*>(a.mass);
  float* volume = const_cast<float*>(a.volume);
  float* rest_x = const_cast<float*>(a.rest_x);
  int32_t* fixed = const_cast<int32_t*>(a.fixed);
  int32_t* region_out = const_cast<int32_t*>(a.region);
  float* rest_normal = const_cast<float*>(a.rest_normal);
  float* rest_area = const_cast<float*>(a.rest_area);
  float* f_ext = const_cast<float*>(a.f_ext);
  for (int32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const int32_t face = p / L.layers, layer = p - face * L.layers;
    const int32_t region = L.face_region[face];
    const bool is_fixed = L.fixed_region >= 0 && region == L.fixed_region;
    float thickness = 0.0f;
    if (region == L.primary)
      thickness = L.t_primary;
    else if (region == L.secondary)
      thickness = L.t_secondary;
    else if (is_fixed)
      thickness = L.t_primary;
    const float frac = ((float)layer + 0.5f) / (float)L.layers - 0.5f;
    const float aw = L.area[face] / (float)L.layers;
    const float vol = aw * thickness;
    const float m = L.density * vol;
    const float off = frac * thickness;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float pos = L.centroid[3 * (size_t)face + d] + L.normal[3 * (size_t)face + d] * off;
      a.x[3 * (size_t)p + d] = pos;
      rest_x[3 * (size_t)p + d] = pos;
      a.v[3 * (size_t)p + d] = 0.0f;
      a.normal[3 * (size_t)p + d] = L.normal[3 * (size_t)face + d];
      rest_normal[3 * (size_t)p + d] = L.normal[3 * (size_t)face + d];
      f_ext[3 * (size_t)p + d] = 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 9; ++e) {
      a.C[9 * (size_t)p + e] = 0.0f;
      a.F[9 * (size_t)p + e] = (e % 4 == 0) ? 1.0f : 0.0f;
    }
    volume[p] = vol;
    a.area[p] = aw;
    rest_area[p] = aw;
    mass[p] = m;
    region_out[p] = region;
    fixed[p] = is_fixed ? 1 : 0;
    if (region == L.primary)
      acc[0] += (double)m;
    else if (region == L.secondary)
      acc[1] += (double)m;
  }
  mpm_partials<NS>(acc, a, a.prow0 + blockIdx.x, lds, 0ull);
}

struct FinRegionMass {
  float* out;  // primary, secondary (float32, as the reference's fields)
  __device__ void operator()(const double* t) const {
    out[0] = (float)t[0];
    out[1] = (float)t[1];
  }
};

struct LoadArgs {
  int32_t mode, region, primary, secondary;
  float pressure;
  float load[3];          // area load (N/m^2) of the area-load modes
  float reaction_p[3];    // layered loads: primary and secondary interface reactions (N)
  float reaction_s[3];
  const float* region_mass;  // layered loads: primary, secondary mass (device)
};

// Region loads on the external force (neo_hookean_mpm.py:357-508).
__global__ void __launch_bounds__(kBlock) k_mpm_region_load(MpmArgs a, LoadArgs L) {
#pragma clang fp contract(off)  // separate roundings, as the reference writes the expressions
  float* f = const_cast<float*>(a.f_ext);
  const float pm = L.region_mass ? fmaxf(L.region_mass[0], 1.0e-12f) : 1.0f;
  const float sm = L.region_mass ? fmaxf(L.region_mass[1], 1.0e-12f) : 1.0f;
  for (int32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < a.count; p += gridDim.x * blockDim.x) {
    const int32_t r = a.region[p];
    const float aw = a.area[p];
    float* fp = f + 3 * (size_t)p;
    if (L.mode == HFSI_MPM_LOAD_SET_PRESSURE || L.mode == HFSI_MPM_LOAD_ADD_PRESSURE) {
      const float s = -L.pressure * aw;
      if (r == L.region) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const float t = s * a.normal[3 * (size_t)p + d];
          fp[d] = L.mode == HFSI_MPM_LOAD_SET_PRESSURE ? t : fp[d] + t;
        }
      } else if (L.mode == HFSI_MPM_LOAD_SET_PRESSURE) {
        fp[0] = fp[1] = fp[2] = 0.0f;
      }
    } else if (L.mode == HFSI_MPM_LOAD_ADD_AREA) {
      if (r == L.region) {
#pragma unroll
        for (int d = 0; d < 3; ++d) fp[d] = fp[d] + L.load[d] * aw;
      }
    } else {  // HFSI_MPM_LOAD_LAYERED
      const float m = a.mass[p];
      float g[3] = {0.0f, 0.0f, 0.0f};
      if (r == L.primary) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          g[d] = g[d] + L.load[d] * aw;
          g[d] = g[d] + L.reaction_p[d] * m / pm;
        }
      } else if (r == L.secondary) {
#pragma unroll
        for (int d = 0; d < 3; ++d) g[d] = g[d] + L.reaction_s[d] * m / sm;
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) fp[d] = g[d];
    }
  }
}

// _enforce_rest_x_plane_kernel / _enforce_rest_z_plane_kernel (neo_hookean_mpm.py:540-573): the
// axis coordinate back to rest, its velocity zero, the affine and deformation couplings of the axis
// removed (F's axis row and column to the identity's), then the surface geometry from F.
__global__ void __launch_bounds__(kBlock) k_mpm_rest_plane(MpmArgs a, int axis) {
  for (int32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < a.count; p += gridDim.x * blockDim.x) {
    float* C = a.C + 9 * (size_t)p;
    float* F = a.F + 9 * (size_t)p;
    a.x[3 * (size_t)p + axis] = a.rest_x[3 * (size_t)p + axis];
    a.v[3 * (size_t)p + axis] = 0.0f;
    if (axis == 0) {
      C[0] = C[1] = C[2] = C[3] = C[6] = 0.0f;
      F[0] = 1.0f;
      F[1] = F[2] = F[3] = F[6] = 0.0f;
    } else {
      C[2] = C[5] = C[6] = C[7] = C[8] = 0.0f;
      F[2] = F[5] = F[6] = F[7] = 0.0f;
      F[8] = 1.0f;
    }
    update_surface(a, (uint32_t)p);
  }
}

}  // namespace hfsi

struct hfsi_mpm {
  int32_t capacity = 0;
  int32_t nx = 0, ny = 0, nz = 0;
  float bmin[3] = {0, 0, 0};
  float dx[3] = {0, 0, 0};
  double* partials = nullptr;
  unsigned int* counter = nullptr;
  double* totals = nullptr;
  double* report = nullptr;
  double* host_report = nullptr;
  float* region_mass = nullptr;  // primary, secondary mass of the layered surface (device)
  int32_t p2g_mode = HFSI_MPM_P2G_BINNED;
  hfsi::BinArgs bins{};
  // Grid bookkeeping of the tile path: when grid_tracked, every node of the grid arrays below lies
  // in a block of bins.prev_need or is zero, so a step zeroes only the blocks it no longer lists.
  bool grid_tracked = false;
  const float* tracked_grid[3] = {nullptr, nullptr, nullptr};
  std::vector<void*> allocs;
};

using namespace hfsi;

// At most 1024 workgroups (four per CU) per grid-stride kernel: its partial rows and the 64 of an
// out-of-bounds pass then fit one round of k_mpm_finish.
static uint32_t mpm_blocks(uint64_t n) { return grid_blocks(n, 1024); }

// Kernel arguments of the particle arrays and the grid geometry (no grid arrays, no step constants).
static MpmArgs particle_args(const hfsi_mpm* h, const hfsi_mpm_particles* P, int32_t count) {
  MpmArgs a{};
  a.x = P->x;
  a.v = P->v;
  a.C = P->C;
  a.F = P->F;
  a.mass = P->mass;
  a.volume = P->volume;
  a.rest_x = P->rest_x;
  a.fixed = P->fixed;
  a.region = P->region;
  a.f_ext = P->external_force;
  a.normal = P->normal;
  a.rest_normal = P->rest_normal;
  a.area = P->area;
  a.rest_area = P->rest_area;
  a.count = count;
  a.nx = h->nx;
  a.ny = h->ny;
  a.nz = h->nz;
  for (int d = 0; d < 3; ++d) {
    a.bmin[d] = h->bmin[d];
    a.dx[d] = h->dx[d];
  }
  a.partials = h->partials;
  a.counter = h->counter;
  a.totals = h->totals;
  a.report = h->report;
  return a;
}

static bool all_particle_arrays(const hfsi_mpm_particles* P) {
  return P && P->x && P->v && P->C && P->F && P->mass && P->volume && P->rest_x && P->fixed && P->region &&
         P->external_force && P->normal && P->rest_normal && P->area && P->rest_area;
}

extern "C" {

int hfsi_mpm_create(hfsi_mpm** out, int32_t capacity, const double* bounds_min3, const double* bounds_max3,
                    const int32_t* grid_nodes3, void* stream) {
  (void)stream;
  if (!out || capacity <= 0 || !bounds_min3 || !bounds_max3 || !grid_nodes3) {
    set_error("hfsi_mpm_create: invalid arguments");
    return HFSI_ERR_ARG;
  }
  for (int d = 0; d < 3; ++d)
    if (grid_nodes3[d] < 4 || !(bounds_max3[d] > bounds_min3[d])) {
      set_error("hfsi_mpm_create: grid must have >= 4 nodes and positive spacing per axis");
      return HFSI_ERR_ARG;
    }
  if ((uint64_t)grid_nodes3[0] * grid_nodes3[1] * grid_nodes3[2] >= (1ull << 31)) {
    set_error("hfsi_mpm_create: grid too large for 32-bit node indices");
    return HFSI_ERR_ARG;
  }
  hfsi_mpm* h = new hfsi_mpm();
  h->capacity = capacity;
  h->nx = grid_nodes3[0];
  h->ny = grid_nodes3[1];
  h->nz = grid_nodes3[2];
  for (int d = 0; d < 3; ++d) {
    h->bmin[d] = (float)bounds_min3[d];
    h->dx[d] = (float)((bounds_max3[d] - bounds_min3[d]) / grid_nodes3[d]);
  }
  {
    BinArgs& b = h->bins;
    auto blocks = [&](int edge) {
      b.edge = edge;
      b.nbx = (h->nx + edge - 1) / edge;
      b.nby = (h->ny + edge - 1) / edge;
      b.nbz = (h->nz + edge - 1) / edge;
      return (size_t)b.nbx * b.nby * b.nbz;
    };
    size_t nb = blocks(kCoarseEdge);
    if (nb > kMaxBlocks) {
      set_error("hfsi_mpm_create: grid too large for the particle binning");
      hfsi_mpm_destroy(h);
      return HFSI_ERR_ARG;
    }
    const bool with_tiles = nb <= kMaxTileBlocks;
    const bool fine = capacity <= kFineParticles;
    if (fine) nb = blocks(kFineEdge);
    auto al = [&](int32_t** p, size_t n) {
      void* q = nullptr;
      if (hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(int32_t)) != hipSuccess) return false;
      h->allocs.push_back(q);
      *p = (int32_t*)q;
      return true;
    };
    const size_t P = (size_t)capacity;
    int32_t* stage = nullptr;
    if (!(al(&b.key, P) && al(&b.rank, P) && al(&b.count, nb) && al(&b.offset, nb) && al(&b.sorted, P) &&
          al(&b.active, nb) && al(&b.nactive, 1) && al(&b.oob, P) && al(&b.noob, 1) && al(&b.svd, P) &&
          al(&b.nsvd, 1) && al(&b.slot, nb) && al(&b.nsorted, 1) &&
          al(&b.cell, P) && al(&b.scell, P) && al(&stage, 16 * P))) {
      set_error("hfsi_mpm_create: device allocation failed");
      hfsi_mpm_destroy(h);
      return HFSI_ERR_HIP;
    }
    b.stage = (float4*)stage;  // hipMalloc memory: 256-byte aligned
    if (with_tiles) {
      const size_t stride = fine ? Tile<kFineEdge>::kStride : Tile<kCoarseEdge>::kStride;
      const size_t tiles = std::min(nb, P);  // blocks that can be active together
      void* q = nullptr;
      if (!(al(&b.need_stamp, nb) && al(&b.need_list, nb) && al(&b.nneed, 1) && al(&b.prev_need, nb) &&
            al(&b.nprev, 1) && al(&b.block_force, tiles) && hipMemset(b.nprev, 0, sizeof(int32_t)) == hipSuccess &&
            hipMalloc(&q, tiles * stride * sizeof(float)) == hipSuccess &&
            hipMemset(b.need_stamp, 0, nb * sizeof(int32_t)) == hipSuccess)) {
        set_error("hfsi_mpm_create: device allocation failed");
        if (q) (void)hipFree(q);
        hfsi_mpm_destroy(h);
        return HFSI_ERR_HIP;
      }
      h->allocs.push_back(q);
      b.tiles = (float*)q;
    }
  }
  bool ok = hipMalloc((void**)&h->partials, sizeof(double) * 2048 * 32) == hipSuccess &&
            hipMalloc((void**)&h->counter, sizeof(unsigned int)) == hipSuccess &&
            hipMalloc((void**)&h->totals, sizeof(double) * (T_COUNT + 2)) == hipSuccess &&
            hipMalloc((void**)&h->report, sizeof(double) * 34) == hipSuccess &&
            hipMalloc((void**)&h->region_mass, sizeof(float) * 2) == hipSuccess &&
            hipMemset(h->region_mass, 0, sizeof(float) * 2) == hipSuccess &&
            hipHostMalloc((void**)&h->host_report, sizeof(double) * 34, hipHostMallocDefault) == hipSuccess &&
            hipMemset(h->counter, 0, sizeof(unsigned int)) == hipSuccess &&
            hipMemset(h->totals, 0, sizeof(double) * (T_COUNT + 2)) == hipSuccess &&
            hipMemset(h->report, 0, sizeof(double) * 34) == hipSuccess && hipDeviceSynchronize() == hipSuccess;
  if (!ok) {
    set_error("hfsi_mpm_create: device allocation failed");
    hfsi_mpm_destroy(h);
    return HFSI_ERR_HIP;
  }
  *out = h;
  return HFSI_OK;
}

int hfsi_mpm_set_p2g_mode(hfsi_mpm* h, int32_t mode) {
  if (!h || (mode != HFSI_MPM_P2G_BINNED && mode != HFSI_MPM_P2G_ATOMIC)) {
    set_error("hfsi_mpm_set_p2g_mode: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if (mode != h->p2g_mode) h->grid_tracked = false;
  h->p2g_mode = mode;
  return HFSI_OK;
}

int hfsi_mpm_invalidate_grid(hfsi_mpm* h) {
  if (!h) {
    set_error("hfsi_mpm_invalidate_grid: invalid arguments");
    return HFSI_ERR_ARG;
  }
  h->grid_tracked = false;
  return HFSI_OK;
}

int hfsi_mpm_destroy(hfsi_mpm* h) {
  if (!h) return HFSI_OK;
  (void)hipDeviceSynchronize();
  if (h->partials) (void)hipFree(h->partials);
  if (h->counter) (void)hipFree(h->counter);
  if (h->totals) (void)hipFree(h->totals);
  if (h->report) (void)hipFree(h->report);
  if (h->region_mass) (void)hipFree(h->region_mass);
  if (h->host_report) (void)hipHostFree(h->host_report);
  for (void* p : h->allocs) (void)hipFree(p);
  delete h;
  return HFSI_OK;
}

int hfsi_mpm_step(hfsi_mpm* h, const hfsi_mpm_particles* P, int32_t count, const hfsi_mpm_grid* G, float dt_s,
                  float mu_pa, float lambda_pa, float velocity_damping, int32_t primary_region_id,
                  int32_t secondary_region_id, double* report34, void* stream) {
  if (!h || !P || !G || count <= 0 || count > h->capacity || !P->x || !P->v || !P->C || !P->F || !P->mass ||
      !P->volume || !P->rest_x || !G->mass || !G->velocity || !G->force) {
    set_error("hfsi_mpm_step: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if ((P->rest_area != nullptr) != (P->rest_normal != nullptr) || (P->rest_area && (!P->area || !P->normal))) {
    set_error("hfsi_mpm_step: surface arrays must be given together");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  MpmArgs a = particle_args(h, P, count);
  a.gm = G->mass;
  a.gv = G->velocity;
  a.gf = G->force;
  a.dt = dt_s;
  a.mu = mu_pa;
  a.lambda = lambda_pa;
  a.damping = velocity_damping;
  a.primary = primary_region_id;
  a.secondary = secondary_region_id;
  a.partials = h->partials;
  a.counter = h->counter;
  a.totals = h->totals;
  a.report = h->report;
  const uint32_t nodes = (uint32_t)h->nx * h->ny * h->nz;
  const uint32_t pb = mpm_blocks(count), nb = mpm_blocks(nodes);
  const uint32_t pbin = grid_blocks((uint64_t)count, 2048);  // binning kernels: no partial rows
  BinArgs& b = h->bins;
  const bool binned = h->p2g_mode == HFSI_MPM_P2G_BINNED;
  const bool tile_path = binned && b.tiles != nullptr;
  const bool fine = b.edge == kFineEdge;
  const bool same_grid = h->tracked_grid[0] == G->mass && h->tracked_grid[1] == G->velocity &&
                         h->tracked_grid[2] == G->force;
  // The tile path rewrites every node of the blocks it lists and zeroes the blocks it listed last
  // step only; other paths, an untracked grid or new grid arrays clear the whole grid first.
  const bool full_clear = !tile_path || !h->grid_tracked || !same_grid;
  if (full_clear)
    hipLaunchKernelGGL(k_mpm_clear, dim3(mpm_blocks(nodes)), dim3(kBlock), 0, st, nodes, a.gm, a.gv, a.gf);
  // each reduction stage: its kernels' workgroups write rows [prow0, prow0 + grid) of a slot-major
  // table of `pstride` rows of its own, which one workgroup then combines
  double* table = h->partials;
  auto rows = [&](uint32_t row0, uint32_t stride) {
    a.partials = table;
    a.prow0 = row0;
    a.pstride = stride;
  };
  auto next_table = [&](uint32_t nrows, uint32_t slots) {
    const StageRows t{table, nrows};
    table += (size_t)nrows * slots;
    return t;
  };
  // workgroups of the per-block kernels: one per block that can be active, up to 4096 (16 per CU)
  const int64_t can_be_active = std::min<int64_t>((int64_t)b.nbx * b.nby * b.nbz, count);
  const uint32_t GP = (uint32_t)(std::min<int64_t>(can_be_active, 4096) + HFSI_NXCD - 1) / HFSI_NXCD * HFSI_NXCD;
  const uint32_t GO = 64;
  StageRows p2g_rows{}, grid_rows{}, g2p_rows{};
  if (binned) {
    b.stamp = b.stamp == INT32_MAX ? 1 : b.stamp + 1;
    b.has_force = a.f_ext != nullptr;
    const int32_t nblk = b.nbx * b.nby * b.nbz;
    b.reset_prev = full_clear ? 1 : 0;
    hipLaunchKernelGGL(k_bin_clear, dim3(std::min<int32_t>((nblk + 255) / 256, 1024)), dim3(256), 0, st, b);
    hipLaunchKernelGGL(fine ? k_bin_count<kFineEdge> : k_bin_count<kCoarseEdge>, dim3(pbin), dim3(kBlock), 0, st, a, b);
    hipLaunchKernelGGL(k_bin_lists, dim3((nblk + kListBlocks - 1) / kListBlocks), dim3(kListBlocks), 0, st, b);
    hipLaunchKernelGGL(k_bin_scatter, dim3(pbin), dim3(kBlock), 0, st, count, b);
    rows(0, pb + GO);
    hipLaunchKernelGGL(k_mpm_p2g_prepare, dim3(pb), dim3(kBlock), 0, st, a, b);
    rows(pb, pb + GO);
    hipLaunchKernelGGL(k_mpm_p2g_prepare_svd, dim3(GO), dim3(kBlock), 0, st, a, b);
    p2g_rows = next_table(pb + GO, 12);
    if (fine)
      hipLaunchKernelGGL(k_mpm_p2g_fine, dim3(GP), dim3(kFineThreads), 0, st, a, b);
    else
      hipLaunchKernelGGL(k_mpm_p2g_cells, dim3(GP), dim3(kP2gThreads), kP2gTileBytes, st, a, b);
    if (b.has_force)
      hipLaunchKernelGGL(fine ? k_mpm_p2g_force<kFineEdge> : k_mpm_p2g_force<kCoarseEdge>, dim3(GP), dim3(kBlock), 0, st,
                         a, b);
  } else {
    rows(0, pb);
    hipLaunchKernelGGL(k_mpm_p2g, dim3(pb), dim3(kBlock), 0, st, a);
    p2g_rows = next_table(pb, 12);
  }
  if (tile_path) {
    const uint32_t GG = 1024;
    rows(0, GG);
    hipLaunchKernelGGL(fine ? k_mpm_grid_gather<kFineEdge> : k_mpm_grid_gather<kCoarseEdge>, dim3(GG + kStaleGroups), dim3(kBlock), 0, st, a, b);
    grid_rows = next_table(GG, 8);
  } else {
    rows(0, nb);
    hipLaunchKernelGGL(k_mpm_grid, dim3(nb), dim3(kBlock), 0, st, a);
    grid_rows = next_table(nb, 8);
  }
  if (binned)
    hipLaunchKernelGGL(fine ? k_mpm_g2p_binned<kFineEdge> : k_mpm_g2p_binned<kCoarseEdge>, dim3(GP + kOobGroups),
                       dim3(kBlock), 0, st, a, b);
  rows(0, pb);
  if (binned)
    hipLaunchKernelGGL(k_mpm_g2p_sums, dim3(pb), dim3(kBlock), 0, st, a);
  else
    hipLaunchKernelGGL(k_mpm_g2p, dim3(pb), dim3(kBlock), 0, st, a);
  g2p_rows = next_table(pb, 21);
  hipLaunchKernelGGL(k_mpm_finish_stages, dim3(3), dim3(kMpmFinishThreads), 0, st, p2g_rows, grid_rows, g2p_rows,
                     a.totals);
  rows(0, pb);
  hipLaunchKernelGGL(k_mpm_radial, dim3(pb), dim3(kBlock), 0, st, a);
  hipLaunchKernelGGL((k_mpm_finish<3, FinMpmReport>), dim3(1), dim3(kMpmFinishThreads), 0, st,
                     (const double*)table, pb, pb, a.totals + T_RSUM, FinMpmReport{a.totals, a.report, a.dt},
                     kRadialMax);
  HFSI_LAUNCH_CHECK();
  if (tile_path) {
    // this step's need list is the next step's previous one
    std::swap(b.need_list, b.prev_need);
    std::swap(b.nneed, b.nprev);
    h->grid_tracked = true;
    h->tracked_grid[0] = G->mass;
    h->tracked_grid[1] = G->velocity;
    h->tracked_grid[2] = G->force;
  } else {
    h->grid_tracked = false;
  }
  if (report34) {
    HFSI_CHECK(hipMemcpyAsync(h->host_report, h->report, 34 * sizeof(double), hipMemcpyDeviceToHost, st));
    HFSI_CHECK(hipStreamSynchronize(st));
    std::memcpy(report34, h->host_report, 34 * sizeof(double));
  }
  return HFSI_OK;
}

int hfsi_mpm_init_layered(hfsi_mpm* h, const hfsi_mpm_particles* P, const float* centroid, const float* normal,
                          const float* area, const int32_t* face_region, int32_t face_count, int32_t layer_count,
                          int32_t primary_region_id, int32_t secondary_region_id, int32_t fixed_region_id,
                          float density, float primary_thickness, float secondary_thickness, void* stream) {
  if (!h || !all_particle_arrays(P) || !centroid || !normal || !area || !face_region || face_count <= 0 ||
      layer_count <= 0 || (int64_t)face_count * layer_count > h->capacity) {
    set_error("hfsi_mpm_init_layered: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int32_t n = face_count * layer_count;
  MpmArgs a = particle_args(h, P, n);
  LayeredArgs L{centroid, normal, area, face_region, face_count, layer_count, primary_region_id,
                secondary_region_id, fixed_region_id, density, primary_thickness, secondary_thickness};
  const uint32_t pb = mpm_blocks(n);
  a.prow0 = 0;
  a.pstride = pb;
  hipLaunchKernelGGL(k_mpm_layered_init, dim3(pb), dim3(kBlock), 0, st, a, L);
  hipLaunchKernelGGL((k_mpm_finish<2, FinRegionMass>), dim3(1), dim3(kMpmFinishThreads), 0, st,
                     (const double*)a.partials, pb, pb, a.totals + T_COUNT, FinRegionMass{h->region_mass},
                     (uint64_t)0);
  HFSI_LAUNCH_CHECK();
  h->grid_tracked = false;
  return HFSI_OK;
}

int hfsi_mpm_region_masses(hfsi_mpm* h, float* out2, void* stream) {
  if (!h || !out2) {
    set_error("hfsi_mpm_region_masses: invalid arguments");
    return HFSI_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  HFSI_CHECK(hipMemcpyAsync(out2, h->region_mass, 2 * sizeof(float), hipMemcpyDeviceToHost, st));
  HFSI_CHECK(hipStreamSynchronize(st));
  return HFSI_OK;
}

int hfsi_mpm_region_load(hfsi_mpm* h, const hfsi_mpm_particles* P, int32_t count, int32_t mode, int32_t region_id,
                         float pressure, const float* load3, void* stream) {
  const bool area_mode = mode == HFSI_MPM_LOAD_ADD_AREA;
  if (!h || !all_particle_arrays(P) || count <= 0 || count > h->capacity ||
      (mode != HFSI_MPM_LOAD_SET_PRESSURE && mode != HFSI_MPM_LOAD_ADD_PRESSURE && !area_mode) ||
      (area_mode && !load3)) {
    set_error("hfsi_mpm_region_load: invalid arguments");
    return HFSI_ERR_ARG;
  }
  LoadArgs L{};
  L.mode = mode;
  L.region = region_id;
  L.pressure = pressure;
  if (area_mode)
    for (int d = 0; d < 3; ++d) L.load[d] = load3[d];
  const MpmArgs a = particle_args(h, P, count);
  hipLaunchKernelGGL(k_mpm_region_load, dim3(mpm_blocks(count)), dim3(kBlock), 0, (hipStream_t)stream, a, L);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_mpm_layered_region_loads(hfsi_mpm* h, const hfsi_mpm_particles* P, int32_t count, int32_t primary_region_id,
                                  int32_t secondary_region_id, const float* primary_area_load3,
                                  const float* primary_reaction3, const float* secondary_reaction3, void* stream) {
  if (!h || !all_particle_arrays(P) || count <= 0 || count > h->capacity || !primary_area_load3 ||
      !primary_reaction3 || !secondary_reaction3) {
    set_error("hfsi_mpm_layered_region_loads: invalid arguments");
    return HFSI_ERR_ARG;
  }
  LoadArgs L{};
  L.mode = HFSI_MPM_LOAD_LAYERED;
  L.primary = primary_region_id;
  L.secondary = secondary_region_id;
  for (int d = 0; d < 3; ++d) {
    L.load[d] = primary_area_load3[d];
    L.reaction_p[d] = primary_reaction3[d];
    L.reaction_s[d] = secondary_reaction3[d];
  }
  L.region_mass = h->region_mass;
  const MpmArgs a = particle_args(h, P, count);
  hipLaunchKernelGGL(k_mpm_region_load, dim3(mpm_blocks(count)), dim3(kBlock), 0, (hipStream_t)stream, a, L);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

int hfsi_mpm_enforce_rest_plane(hfsi_mpm* h, const hfsi_mpm_particles* P, int32_t count, int32_t axis,
                                void* stream) {
  if (!h || !all_particle_arrays(P) || count <= 0 || count > h->capacity || (axis != 0 && axis != 2)) {
    set_error("hfsi_mpm_enforce_rest_plane: invalid arguments");
    return HFSI_ERR_ARG;
  }
  const MpmArgs a = particle_args(h, P, count);
  hipLaunchKernelGGL(k_mpm_rest_plane, dim3(mpm_blocks(count)), dim3(kBlock), 0, (hipStream_t)stream, a, (int)axis);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

}  // extern "C"
