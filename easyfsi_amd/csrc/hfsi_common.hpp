// Shared device/host helpers for libhfsi (gfx950).
//
// Work decomposition used by every full-grid kernel: the flat cell range is
// cut into chunks of blockDim.x cells.  Workgroups are dispatched round-robin
// over the 8 XCDs (workgroup b runs on XCD b % 8), so XCD x is given the
// contiguous chunk range [x*C/8, (x+1)*C/8) and its workgroups stride over it.
// Each XCD therefore streams one contiguous slab of the grid and the +-j / +-i
// stencil neighbours of a chunk are served by that XCD's own L2.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <cstdio>
#include <string>

#ifndef HFSI_NXCD
#define HFSI_NXCD 8
#endif

namespace hfsi {

constexpr int kBlock = 256;       // threads per workgroup of the full-grid kernels
constexpr int kMaxPartials = 4096;  // workgroups of a reducing launch (upper bound)
constexpr int kMaxSums = 8;       // values reduced by one launch

void set_error(const std::string& msg);

#define HFSI_CHECK(expr)                                                               \
  do {                                                                                 \
    hipError_t _e = (expr);                                                            \
    if (_e != hipSuccess) {                                                            \
      ::hfsi::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));            \
      return HFSI_ERR_HIP;                                                             \
    }                                                                                  \
  } while (0)

#define HFSI_LAUNCH_CHECK()                                                            \
  do {                                                                                 \
    hipError_t _e = hipGetLastError();                                                 \
    if (_e != hipSuccess) {                                                            \
      ::hfsi::set_error(std::string("kernel launch: ") + hipGetErrorString(_e));      \
      return HFSI_ERR_HIP;                                                             \
    }                                                                                  \
  } while (0)

// ---------------------------------------------------------------------------
// Workgroup barrier for LDS-only exchange.  __syncthreads() also waits for
// every outstanding global load and store of the wave (it is a workgroup
// memory fence), which defeats loads issued a step ahead of their use; this
// barrier waits only for the wave's LDS accesses.  Use it only where the
// threads of the workgroup exchange data through LDS alone.
// ---------------------------------------------------------------------------

__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---------------------------------------------------------------------------
// XCD-aware chunk iteration
// ---------------------------------------------------------------------------

struct ChunkRange {
  uint32_t first, end, step;
};

// The chunks of the first `groups` workgroups (a multiple of HFSI_NXCD), for one of them.
__device__ inline ChunkRange xcd_chunks(uint32_t nchunks, uint32_t groups) {
  const uint32_t b = blockIdx.x;
  const uint32_t per = groups / HFSI_NXCD;
  const uint32_t x = b % HFSI_NXCD;
  const uint32_t s = b / HFSI_NXCD;
  const uint32_t lo = (uint32_t)(((uint64_t)nchunks * x) / HFSI_NXCD);
  const uint32_t hi = (uint32_t)(((uint64_t)nchunks * (x + 1)) / HFSI_NXCD);
  return ChunkRange{lo + s, hi, per};
}

// Requires gridDim.x to be a multiple of HFSI_NXCD.
__device__ inline ChunkRange xcd_chunks(uint32_t nchunks) { return xcd_chunks(nchunks, gridDim.x); }

// Loop over the cells [0, n) owned by this thread under the XCD-aware chunk
// decomposition; `c` is the cell index; `continue` moves to the next chunk.
#define HFSI_CELL_LOOP(n)                                                           \
  const ChunkRange _cr = xcd_chunks(((n) + blockDim.x - 1) / blockDim.x);          \
  for (uint32_t _ch = _cr.first; _ch < _cr.end; _ch += _cr.step)                   \
    for (uint32_t c = _ch * blockDim.x + threadIdx.x, _once = 1; _once; _once = 0) \
      if (c < (n))

// Division by a divisor d (1 <= d < 2^31) fixed at launch, for numerators
// n < 2^31, as a multiply-high and a shift (T. Granlund and P. Montgomery,
// "Division by invariant integers using multiplication", PLDI 1994, sec. 4):
// with l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1 < 2^32,
// floor(n / d) = (mulhi(m, n) + n) >> l; the sum stays below 2^32 because
// mulhi(m, n) < n < 2^31.
struct FastDiv {
  uint32_t d, m, l;
  static inline FastDiv make(uint32_t d) {
    uint32_t l = 0;
    while (l < 32 && (1ull << l) < d) ++l;
    const uint64_t m = ((1ull << 32) * ((1ull << l) - d)) / d + 1;
    return FastDiv{d, (uint32_t)m, l};
  }
  __device__ inline uint32_t div(uint32_t n) const { return (__umulhi(m, n) + n) >> l; }
};

// Number of workgroups for a full-grid launch over n cells.
inline uint32_t grid_blocks(uint64_t n, uint32_t max_blocks) {
  uint64_t chunks = (n + kBlock - 1) / kBlock;
  uint64_t g = chunks < max_blocks ? chunks : max_blocks;
  g = (g + HFSI_NXCD - 1) / HFSI_NXCD * HFSI_NXCD;
  if (g == 0) g = HFSI_NXCD;
  return (uint32_t)g;
}

// ---------------------------------------------------------------------------
// Wavefront / workgroup reductions (64-wide wavefronts)
// ---------------------------------------------------------------------------

// Wavefront reductions on DPP row operations (VALU only; a cross-lane shuffle is an LDS
// permute with its latency, twice per double).  Within each row of 16 lanes, row_shr by 1, 2,
// 4 and 8 accumulates every lane's prefix, so lane 15 holds the row; row_bcast:15 adds row 0's
// (row 2's) lane 15 into row 1 (row 3), row_bcast:31 adds lane 31 into rows 2 and 3, and lane
// 63 holds the wavefront's result, which every lane reads back.  Lanes whose DPP source lies
// outside the row, and rows masked off, take the identity.  Requires all 64 lanes active (as
// the shuffle form did).  A fixed order: the result does not depend on timing.
namespace dpp {
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kRowBcast15 = 0x142, kRowBcast31 = 0x143;

template <int CTRL, int ROWS>
__device__ inline double mov(double x, double identity) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(identity), __double2loint(x), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(identity), __double2hiint(x), CTRL, ROWS, 0xf, false);
  return __hiloint2double(hi, lo);
}

template <int CTRL, int ROWS>
__device__ inline float mov(float x, float identity) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(identity), __float_as_int(x), CTRL, ROWS, 0xf, false));
}

__device__ inline double lane63(double x) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63),
                          __builtin_amdgcn_readlane(__double2loint(x), 63));
}
__device__ inline float lane63(float x) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63)); }

template <typename T, typename Op>
__device__ inline T reduce(T v, T id, Op op) {
  v = op(v, mov<kRowShr1, 0xf>(v, id));
  v = op(v, mov<kRowShr2, 0xf>(v, id));
  v = op(v, mov<kRowShr4, 0xf>(v, id));
  v = op(v, mov<kRowShr8, 0xf>(v, id));
  v = op(v, mov<kRowBcast15, 0xa>(v, id));
  v = op(v, mov<kRowBcast31, 0xc>(v, id));
  return lane63(v);
}
}  // namespace dpp

__device__ inline double wave_sum(double v) {
  return dpp::reduce(v, 0.0, [](double a, double b) { return a + b; });
}

__device__ inline double wave_max(double v) {
  return dpp::reduce(v, -(double)INFINITY, [](double a, double b) { return fmax(a, b); });
}

__device__ inline float wave_sum_f32(float v) {
  return dpp::reduce(v, 0.0f, [](float a, float b) { return a + b; });
}

// Workgroup reduction of NS values with `maxmask` marking max-reduced slots;
// result valid in thread 0.  `lds` must hold NS * (blockDim.x / 64) doubles.
// The wavefront results of a slot are combined in wavefront order by one thread
// per slot (the slots in parallel: one thread walking all of them would wait on
// an LDS load per slot and wavefront).
template <int NS>
__device__ inline void block_reduce(double (&v)[NS], double* lds, uint64_t maxmask) {
  static_assert(NS <= 64, "one combining thread per slot in the first wavefront");
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
#pragma unroll
  for (int s = 0; s < NS; ++s) v[s] = ((maxmask >> s) & 1) ? wave_max(v[s]) : wave_sum(v[s]);
  if (lane == 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) lds[s * nw + wave] = v[s];
  }
  __syncthreads();
  if (threadIdx.x < (unsigned)NS) {
    const int s = (int)threadIdx.x;
    const bool mx = (maxmask >> s) & 1;
    double acc = lds[s * nw];
    for (int w = 1; w < nw; ++w) acc = mx ? fmax(acc, lds[s * nw + w]) : acc + lds[s * nw + w];
    lds[s * nw] = acc;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = lds[s * nw];
  }
  __syncthreads();
}

// Grid reductions are two launches on one stream: every workgroup of the
// producing kernel stores its NS partial results (block_partials), then
// k_finish_sums (one workgroup) combines them in workgroup order and runs the
// finaliser.  The kernel boundary publishes the partials; a device-scope fence
// per workgroup would instead write back the XCD's L2 (the producing kernels
// stream their outputs through it) once per workgroup.
template <int NS>
__device__ inline void block_partials(double (&v)[NS], double* partials, double* lds, uint64_t maxmask = 0) {
  block_reduce<NS>(v, lds, maxmask);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) partials[(size_t)blockIdx.x * NS + s] = v[s];
  }
}

constexpr int kFinishThreads = 256;

template <int NS, typename Fin>
__global__ void __launch_bounds__(kFinishThreads) k_finish_sums(const double* partials, uint32_t nblocks,
                                                                 double* totals, Fin fin, uint64_t maxmask) {
  __shared__ double lds[NS * (kFinishThreads / 64)];
  double acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = ((maxmask >> s) & 1) ? -INFINITY : 0.0;
  for (uint32_t b = threadIdx.x; b < nblocks; b += blockDim.x) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const double p = partials[(size_t)b * NS + s];
      acc[s] = ((maxmask >> s) & 1) ? fmax(acc[s], p) : acc[s] + p;
    }
  }
  block_reduce<NS>(acc, lds, maxmask);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) totals[s] = acc[s];
    fin(totals);
  }
}

}  // namespace hfsi
