// Immersed-boundary node search of the HIBM coupling (gfx950):
// HibmMpmIbNodeSearch._search_and_classify_kernel and
// _search_and_classify_grid_fields_kernel (simulation_core/hibm_mpm.py:5601-6058) with
// _closest_point_on_triangle (5494-5549), _oriented_triangle_normal (5551-5559),
// _barycentric_weights_on_triangle (5561-5580) and _nearest_triangle_marker (5582-5598).
//
// Every grid node looks for the closest point of the marker surface (projection triangles,
// or the markers themselves when there are none).  Within the search radius it keeps the
// nearest candidate and the nearest candidate on the positive side of its normal; with far
// classification a node with nothing in range becomes internal when no candidate anywhere
// has it on its positive side.  The reference runs the full node x triangle double loop.
// Here one 256-lane workgroup owns a 4 x 8 x 8 tile of nodes:
//   1. near phase: the triangles are walked in index order in chunks of 256; each lane
//      builds one triangle record (corners, edges, oriented unit normal) and tests its
//      bounding box, grown by the search radius, against the tile's box; the survivors are
//      compacted into LDS in index order (wavefront ballots) and every node tests them.
//      A triangle outside the grown box is farther than the radius from every node of the
//      tile, so the nearest / external choices are those of the full loop, ties included
//      (strict comparisons in index order).
//   2. far phase (classify_far_internal_nodes): a node without a near candidate is done at the
//      first candidate that has it on its positive side (it then stays "none" whatever the
//      others are); an internal one needs the nearest of all candidates, the lowest index among
//      equal distances.  The order of the visits does not matter to either, so every node first
//      visits the tile's closest candidate (outside nodes end there) and then the one whose
//      centroid is closest to it; the walk over all triangles after that evaluates only those
//      whose plane and bounding ball leave a chance (far_bound), about one per node on a closed
//      sphere.  128^3 nodes, 6016 triangles, 200 000 internal nodes: 12.0 -> 1.19 ms (evaluating
//      every triangle for every internal node before; 0.34 ms are the near phase).  The rest is
//      the tiles at the centre of curvature, where no plane is far enough to be skipped for a
//      whole tile.
// Nodes keep only the index and distance of their best candidates; the chosen candidate's
// point, normal, weights and nearest marker are recomputed at the end with the same
// operations.  All arithmetic is float32 in the reference's operation order without
// contraction (a dot product is (x0 y0 + x1 y1) + x2 y2).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <string>

#include "../../include/hfsi.h"
#include "hfsi_common.hpp"

namespace hfsi {

namespace {

constexpr int kIbThreads = 256;
constexpr int kTileI = 4, kTileJ = 8, kTileK = 8;  // kTileI * kTileJ * kTileK == kIbThreads
constexpr int kRecFloats = 21;                      // a, b, c, ab, ac, cb, n
constexpr int kNearUnroll = 4;                      // triangles per lane in flight in the near phase
constexpr int kFarUnroll = 4;                       // candidates per node in flight in the far walk
constexpr int kSeedChunk = 1024;                    // centroids staged at a time
constexpr int kNodeNone = 0, kNodeExternalIb = 1, kNodeInternal = 2;

struct V3 {
  float x, y, z;
};

__device__ inline V3 ld3(const float* p, int64_t i) { return {p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }
__device__ inline V3 sub(V3 a, V3 b) {
#pragma clang fp contract(off)
  return {a.x - b.x, a.y - b.y, a.z - b.z};
}
__device__ inline V3 add(V3 a, V3 b) {
#pragma clang fp contract(off)
  return {a.x + b.x, a.y + b.y, a.z + b.z};
}
__device__ inline V3 mul(V3 a, float s) {
#pragma clang fp contract(off)
  return {a.x * s, a.y * s, a.z * s};
}
__device__ inline V3 divs(V3 a, float s) {
#pragma clang fp contract(off)
  return {a.x / s, a.y / s, a.z / s};
}
__device__ inline float dot(V3 a, V3 b) {
#pragma clang fp contract(off)
  return (a.x * b.x + a.y * b.y) + a.z * b.z;
}
__device__ inline V3 cross(V3 a, V3 b) {
#pragma clang fp contract(off)
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ inline float norm(V3 a) { return sqrtf(dot(a, a)); }

struct Tri {
  V3 a, b, c, ab, ac, cb, n;
  float nn;  // |ab x ac|
  bool valid;
};

struct SearchArgs {
  int32_t nx, ny, nz;
  float bmin[3], spacing[3];
  const float *cx, *cy, *cz;  // cell centres, or NULL for the uniform node grid
  const float* xm;            // marker positions [M][3]
  const float* nm;            // marker normals [M][3]
  const int32_t* tris;        // [T][3] or NULL
  int32_t markers, triangles;
  float radius, probe, tol;
  int32_t far;
  int32_t* kind;
  int32_t* nearest;
  float* signed_distance;
  float* boundary;
  float* interior;
  int32_t* proj_idx;
  float* proj_w;
  int32_t* report;
};

__device__ inline bool tri_indices(const SearchArgs& a, int t, int& ia, int& ib, int& ic) {
  ia = a.tris[3 * t];
  ib = a.tris[3 * t + 1];
  ic = a.tris[3 * t + 2];
  return ia >= 0 && ib >= 0 && ic >= 0 && ia < a.markers && ib < a.markers && ic < a.markers;
}

// Triangle record: _closest_point_on_triangle's node-independent part plus the orientation.
__device__ inline Tri make_tri(const SearchArgs& s, int ia, int ib, int ic) {
#pragma clang fp contract(off)
  Tri t;
  t.a = ld3(s.xm, ia);
  t.b = ld3(s.xm, ib);
  t.c = ld3(s.xm, ic);
  t.ab = sub(t.b, t.a);
  t.ac = sub(t.c, t.a);
  t.cb = sub(t.c, t.b);
  V3 fn = cross(t.ab, t.ac);
  const float nn = norm(fn);
  t.nn = nn;
  t.valid = nn > 1.0e-12f;
  if (t.valid) {
    fn = divs(fn, nn);
    V3 avg = add(add(ld3(s.nm, ia), ld3(s.nm, ib)), ld3(s.nm, ic));
    const float an = norm(avg);
    if (an > 1.0e-12f) {
      avg = divs(avg, an);
      if (dot(fn, avg) < 0.0f) fn = {-fn.x, -fn.y, -fn.z};
    }
  }
  t.n = fn;
  return t;
}

__device__ inline V3 closest_point(V3 p, const Tri& t) {
#pragma clang fp contract(off)
  const V3 ap = sub(p, t.a);
  const float d1 = dot(t.ab, ap), d2 = dot(t.ac, ap);
  if (d1 <= 0.0f && d2 <= 0.0f) return t.a;
  const V3 bp = sub(p, t.b);
  const float d3 = dot(t.ab, bp), d4 = dot(t.ac, bp);
  if (d3 >= 0.0f && d4 <= d3) return t.b;
  const float vc = d1 * d4 - d3 * d2;
  if (vc <= 0.0f && d1 >= 0.0f && d3 <= 0.0f) return add(t.a, mul(t.ab, d1 / fmaxf(d1 - d3, 1.0e-30f)));
  const V3 cp = sub(p, t.c);
  const float d5 = dot(t.ab, cp), d6 = dot(t.ac, cp);
  if (d6 >= 0.0f && d5 <= d6) return t.c;
  const float vb = d5 * d2 - d1 * d6;
  if (vb <= 0.0f && d2 >= 0.0f && d6 <= 0.0f) return add(t.a, mul(t.ac, d2 / fmaxf(d2 - d6, 1.0e-30f)));
  const float va = d3 * d6 - d5 * d4;
  const float e43 = d4 - d3, e56 = d5 - d6;
  if (va <= 0.0f && e43 >= 0.0f && e56 >= 0.0f) return add(t.b, mul(t.cb, e43 / fmaxf((e43 + d5) - d6, 1.0e-30f)));
  const float denom = fmaxf((va + vb) + vc, 1.0e-30f);
  const float v = vb / denom, w = vc / denom;
  return add(add(t.a, mul(t.ab, v)), mul(t.ac, w));
}

__device__ inline V3 barycentric(V3 point, const Tri& t) {
#pragma clang fp contract(off)
  const V3 ap = sub(point, t.a);
  const float d00 = dot(t.ab, t.ab), d01 = dot(t.ab, t.ac), d11 = dot(t.ac, t.ac);
  const float d20 = dot(ap, t.ab), d21 = dot(ap, t.ac);
  const float denom = d00 * d11 - d01 * d01;
  if (!(fabsf(denom) > 1.0e-30f)) return {1.0f, 0.0f, 0.0f};
  float v = (d11 * d20 - d01 * d21) / denom;
  float w = (d00 * d21 - d01 * d20) / denom;
  float u = (1.0f - v) - w;
  u = fminf(fmaxf(u, 0.0f), 1.0f);
  v = fminf(fmaxf(v, 0.0f), 1.0f);
  w = fminf(fmaxf(w, 0.0f), 1.0f);
  const float total = fmaxf((u + v) + w, 1.0e-30f);
  return {u / total, v / total, w / total};
}

__device__ inline V3 node_position(const SearchArgs& s, int i, int j, int k) {
#pragma clang fp contract(off)
  if (s.cx) return {s.cx[i], s.cy[j], s.cz[k]};
  return {s.bmin[0] + ((float)i + 0.5f) * s.spacing[0], s.bmin[1] + ((float)j + 0.5f) * s.spacing[1],
          s.bmin[2] + ((float)k + 0.5f) * s.spacing[2]};
}

// Workgroup-ordered compaction: lanes with `keep` get consecutive slots in lane order.
__device__ inline int compact_slot(bool keep, int* wave_count, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t mask = __ballot(keep);
  if (lane == 0) wave_count[wave] = __popcll(mask);
  __syncthreads();
  int base = 0;
  total = 0;
  for (int w = 0; w < kIbThreads / 64; ++w) {
    if (w < wave) base += wave_count[w];
    total += wave_count[w];
  }
  const int slot = base + __popcll(mask & ((1ull << lane) - 1ull));
  return keep ? slot : -1;
}

__global__ void k_ib_zero_report(int32_t* report) {
  if (threadIdx.x < 4) report[threadIdx.x] = 0;
}

// What a tile needs to decide, before any closest-point evaluation, that a triangle cannot change a
// node's far result.  With u = 2^-24, S the largest coordinate, D the largest distance of a tile node
// to a corner and L the longest edge:
//   - each of va, vb, vc of closest_point is off by at most 19 u (L D)^2, so with q = L D / nn
//     (nn = twice the area) and 60 u q^2 <= 1/4 the point it returns is a + v ab + w ac with
//     |v|, |w| <= 2, at most 2 L (105 u q^2) away from the triangle;
//   - the triangle's plane then bounds both tests: the signed distance the node would compute is at
//     most h + m and its distance at least |h| - m, h = (p - a) . n, with
//     m = 2 (|ab . n| + |ac . n|) + 32 u (S + D + L).
// A triangle whose q is too large (a far sliver) is never skipped.
struct Bound {
  V3 n;      // plane normal (0: never skipped)
  float d;   // a . n - m (-inf: never skipped): h + m = p . n - d
  V3 g;      // centroid
  float r;   // every point closest_point can return lies within r of g
};

__device__ inline Bound far_bound(const Tri& t, V3 tc, float rt, float s_max) {
  constexpr float u = 5.9604645e-8f;
  Bound b{{0.0f, 0.0f, 0.0f}, -INFINITY, t.a, INFINITY};
  const float L = sqrtf(fmaxf(fmaxf(dot(t.ab, t.ab), dot(t.ac, t.ac)), dot(t.cb, t.cb)));
  const V3 ca = sub(tc, t.a);
  const float D = norm(ca) + rt + L;
  const float q = L * D / t.nn;
  if (!(60.0f * u * q * q <= 0.25f)) return b;
  const float S = fmaxf(s_max, fmaxf(fabsf(t.a.x), fmaxf(fabsf(t.a.y), fabsf(t.a.z))) + L);
  const float slack = 32.0f * u * (S + D + L);
  const float m = 2.0f * (fabsf(dot(t.ab, t.n)) + fabsf(dot(t.ac, t.n))) + slack;
  b.n = t.n;
  b.d = dot(t.a, t.n) - m;
  b.g = add(t.a, mul(add(t.ab, t.ac), 0.33333334f));
  const V3 ga = sub(t.a, b.g), gb = sub(t.b, b.g), gc = sub(t.c, b.g);
  b.r = sqrtf(fmaxf(fmaxf(dot(ga, ga), dot(gb, gb)), dot(gc, gc))) + 2.0f * L * (105.0f * u * q * q) + slack;
  return b;
}

// Bounded by the latency of the triangle walk (indices, then corners, from L2) and, where a tile has
// deep internal nodes, by the plane test per node and triangle (one 16-byte LDS broadcast, four
// operations).  Four triangles per lane are in flight in the near phase, and a chunk without a
// survivor costs one barrier.
__global__ void __launch_bounds__(kIbThreads) k_ib_search(SearchArgs s) {
#pragma clang fp contract(off)
  __shared__ float rec[kIbThreads][kRecFloats];
  __shared__ int rec_id[kIbThreads];
  __shared__ float4 plane[kIbThreads + kFarUnroll], ball[kIbThreads + kFarUnroll];
  __shared__ float tile_box[6];
  __shared__ int wave_count[kIbThreads / 64];
  __shared__ unsigned long long seed_key;
  __shared__ int far_max, cent_count;

  const int tk_n = (s.nz + kTileK - 1) / kTileK, tj_n = (s.ny + kTileJ - 1) / kTileJ;
  const int tile = blockIdx.x;
  const int ti = tile / (tj_n * tk_n), tj = (tile / tk_n) % tj_n, tk = tile % tk_n;
  const int tid = threadIdx.x;
  const int i = ti * kTileI + tid / (kTileJ * kTileK);
  const int j = tj * kTileJ + (tid / kTileK) % kTileJ;
  const int k = tk * kTileK + tid % kTileK;
  const bool active = i < s.nx && j < s.ny && k < s.nz;
  const V3 p = active ? node_position(s, i, j, k) : V3{0.0f, 0.0f, 0.0f};

  // the tile's box: the nodes are a product of three axes, lane d < 3 walks axis d
  if (tid < 3) {
    const int n = tid == 0 ? s.nx : tid == 1 ? s.ny : s.nz;
    const int begin = tid == 0 ? ti * kTileI : tid == 1 ? tj * kTileJ : tk * kTileK;
    const int end = min(n, begin + (tid == 0 ? kTileI : tid == 1 ? kTileJ : kTileK));
    float mn = INFINITY, mx = -INFINITY;
    for (int q = begin; q < end; ++q) {
      const V3 c = node_position(s, tid == 0 ? q : 0, tid == 1 ? q : 0, tid == 2 ? q : 0);
      const float v = tid == 0 ? c.x : tid == 1 ? c.y : c.z;
      mn = fminf(mn, v);
      mx = fmaxf(mx, v);
    }
    tile_box[tid] = mn;
    tile_box[3 + tid] = mx;
  }
  if (tid == 3) {
    seed_key = ~0ull;
    far_max = 0;
  }
  __syncthreads();
  float lo[3], hi[3];
  const float scale = fmaxf(fmaxf(fabsf(tile_box[0]), fabsf(tile_box[3])),
                            fmaxf(fmaxf(fabsf(tile_box[1]), fabsf(tile_box[4])),
                                  fmaxf(fabsf(tile_box[2]), fabsf(tile_box[5]))));
  {
    const float grow = s.radius * 1.001f + 1.0e-6f * (1.0f + scale);  // conservative
    for (int d = 0; d < 3; ++d) {
      lo[d] = tile_box[d] - grow;
      hi[d] = tile_box[3 + d] + grow;
    }
  }
  const V3 tc = {0.5f * (tile_box[0] + tile_box[3]), 0.5f * (tile_box[1] + tile_box[4]),
                 0.5f * (tile_box[2] + tile_box[5])};
  const V3 half = {0.5001f * (tile_box[3] - tile_box[0]), 0.5001f * (tile_box[4] - tile_box[1]),
                   0.5001f * (tile_box[5] - tile_box[2])};

  const bool use_tris = s.triangles > 0;
  const int count = use_tris ? s.triangles : s.markers;
  int tn = -1, te = -1, tg = -1;
  float dn = 1.0e30f, de = 1.0e30f, dg = 1.0e30f;
  bool ext_seen = false, gext_seen = false;

  // lane `keep`'s candidate `t` into the next LDS slot in lane order; returns the slot (-1: none)
  auto store_rec = [&](bool keep, const Tri& tr, int t, int& total) {
    const int slot = compact_slot(keep, wave_count, total);
    if (slot >= 0) {
      const float v[kRecFloats] = {tr.a.x,  tr.a.y,  tr.a.z,  tr.b.x,  tr.b.y,  tr.b.z,  tr.c.x,
                                   tr.c.y,  tr.c.z,  tr.ab.x, tr.ab.y, tr.ab.z, tr.ac.x, tr.ac.y,
                                   tr.ac.z, tr.cb.x, tr.cb.y, tr.cb.z, tr.n.x,  tr.n.y,  tr.n.z};
#pragma unroll
      for (int q = 0; q < kRecFloats; ++q) rec[slot][q] = v[q];
      rec_id[slot] = t;
    }
    return slot;
  };
  auto load_rec = [&](int q) {
    const float* r = rec[q];
    Tri c;
    c.a = {r[0], r[1], r[2]};
    c.b = {r[3], r[4], r[5]};
    c.c = {r[6], r[7], r[8]};
    c.ab = {r[9], r[10], r[11]};
    c.ac = {r[12], r[13], r[14]};
    c.cb = {r[15], r[16], r[17]};
    c.n = {r[18], r[19], r[20]};
    return c;
  };
  auto load_tri = [&](int t, Tri& tr) {  // false: not a candidate
    if (use_tris) {
      int ia, ib, ic;
      if (!tri_indices(s, t, ia, ib, ic)) return false;
      tr = make_tri(s, ia, ib, ic);
      return tr.valid;
    }
    tr.a = ld3(s.xm, t);
    tr.b = tr.c = tr.a;
    tr.n = ld3(s.nm, t);
    return true;
  };

  // 1. near phase; each lane also keeps its candidate whose first corner is closest to the tile's centre
  float best = INFINITY;
  int best_t = -1;
  for (int base = 0; base < count; base += kNearUnroll * kIbThreads) {
    uint32_t in_reach = 0;
    int idx[kNearUnroll][3];
#pragma unroll
    for (int q = 0; q < kNearUnroll; ++q) {
      const int t = base + q * kIbThreads + tid;
      idx[q][0] = idx[q][1] = idx[q][2] = t < count ? t : -1;
      if (use_tris && t < count && !tri_indices(s, t, idx[q][0], idx[q][1], idx[q][2])) idx[q][0] = -1;
    }
#pragma unroll
    for (int q = 0; q < kNearUnroll; ++q) {
      if (idx[q][0] < 0) continue;
      const V3 a = ld3(s.xm, idx[q][0]);
      const V3 b = use_tris ? ld3(s.xm, idx[q][1]) : a, c = use_tris ? ld3(s.xm, idx[q][2]) : a;
      const float mn[3] = {fminf(fminf(a.x, b.x), c.x), fminf(fminf(a.y, b.y), c.y), fminf(fminf(a.z, b.z), c.z)};
      const float mx[3] = {fmaxf(fmaxf(a.x, b.x), c.x), fmaxf(fmaxf(a.y, b.y), c.y), fmaxf(fmaxf(a.z, b.z), c.z)};
      bool in = true;
      for (int d = 0; d < 3; ++d)
        if (!(mn[d] <= hi[d] && mx[d] >= lo[d])) in = false;
      if (in) in_reach |= 1u << q;
      const V3 o = sub(a, tc);
      const float o2 = dot(o, o);
      if (o2 < best) {
        best = o2;
        best_t = base + q * kIbThreads + tid;
      }
    }
    if (!__syncthreads_or(in_reach != 0)) continue;
    for (int q = 0; q < kNearUnroll; ++q) {
      const int t = base + q * kIbThreads + tid;
      Tri tr{};
      const bool keep = (in_reach >> q & 1) && load_tri(t, tr);
      if (!__syncthreads_or(keep)) continue;  // also: the records of the round before are consumed
      int total;
      store_rec(keep, tr, t, total);
      __syncthreads();
      if (active) {
        for (int e = 0; e < total; ++e) {
          const Tri c = load_rec(e);
          const V3 cl = use_tris ? closest_point(p, c) : c.a;
          const V3 off = sub(p, cl);
          const float dist = norm(off);
          if (dist < s.radius) {
            const float sd = dot(off, c.n);
            if (sd > s.tol) {
              ext_seen = true;
              if (dist < de) {
                de = dist;
                te = rec_id[e];
              }
            }
            if (dist < dn) {
              dn = dist;
              tn = rec_id[e];
            }
          }
        }
      }
    }
  }

  // 2. far phase: every candidate for the nodes left without a near one
  const bool need = active && tn < 0;
  if (s.far && __syncthreads_or(need)) {
    // the nearest over all candidates, the lowest index among equal distances; false: on the positive
    // side of this one, so the node stays "none" whatever the others are
    auto visit = [&](const Tri& c, int t) {
      const V3 cl = use_tris ? closest_point(p, c) : c.a;
      const V3 off = sub(p, cl);
      const float dist = norm(off);
      if (dot(off, c.n) > s.tol) return false;
      if (dist < dg || (dist == dg && t < tg)) {
        dg = dist;
        tg = t;
      }
      return true;
    };
    // every node starts from the tile's closest candidate: outside nodes end there, internal ones
    // have nearly their final distance for the bounds below
    if (best_t >= 0) atomicMin(&seed_key, ((unsigned long long)__float_as_uint(best) << 32) | (uint32_t)best_t);
    __syncthreads();
    if (seed_key != ~0ull) {
      const int t = (int)(uint32_t)seed_key;
      Tri tr{};
      if (load_tri(t, tr) && need) gext_seen = !visit(tr, t);
    }
    if (need && !gext_seen) atomicMax(&far_max, __float_as_int(dg));  // dg >= 0: ordered as integers
    const float rt = norm(half);
    // internal nodes then take the candidate whose centroid is closest to them: from there about one
    // closest-point evaluation per node is left (near a centre of curvature, where all candidates are
    // about equally far, the walk in index order would otherwise evaluate most of them)
    if (use_tris && __syncthreads_or(need && !gext_seen)) {
      float4* cent = reinterpret_cast<float4*>(&rec[0][0]);
      static_assert((kSeedChunk + kFarUnroll) * sizeof(float4) <= sizeof(rec), "the centroids fit the records");
      const float dmax = __int_as_float(far_max);
      float c2 = INFINITY;
      int first = -1;
      for (int base = 0; base < count; base += kSeedChunk) {
        if (tid == 0) cent_count = 0;
        __syncthreads();
        for (int t = base + tid; t < min(count, base + kSeedChunk); t += kIbThreads) {
          int ia, ib, ic;
          if (!tri_indices(s, t, ia, ib, ic)) continue;
          const V3 a = ld3(s.xm, ia), b = ld3(s.xm, ib), c = ld3(s.xm, ic);
          const V3 g = mul(add(add(a, b), c), 0.33333334f);
          const V3 ga = sub(a, g), gb = sub(b, g), gc = sub(c, g);
          const float r = sqrtf(fmaxf(fmaxf(dot(ga, ga), dot(gb, gb)), dot(gc, gc)));
          if (norm(sub(tc, g)) - rt > dmax + r) continue;
          cent[atomicAdd(&cent_count, 1)] = make_float4(g.x, g.y, g.z, __int_as_float(t));
        }
        __syncthreads();
        const int total = cent_count;
        if (tid < kFarUnroll) cent[total + tid] = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
        __syncthreads();
        if (need && !gext_seen) {
          for (int q = 0; q < total; q += kFarUnroll) {
            float4 g[kFarUnroll];
            float o2[kFarUnroll];
#pragma unroll
            for (int e = 0; e < kFarUnroll; ++e) {
              g[e] = cent[q + e];
              const V3 o = {p.x - g[e].x, p.y - g[e].y, p.z - g[e].z};
              o2[e] = dot(o, o);
            }
#pragma unroll
            for (int e = 0; e < kFarUnroll; ++e)
              if (o2[e] < c2) {
                c2 = o2[e];
                first = __float_as_int(g[e].w);
              }
          }
        }
        __syncthreads();
      }
      Tri tr{};
      if (first >= 0 && load_tri(first, tr)) gext_seen = !visit(tr, first);
      if (tid == 0) far_max = 0;
      __syncthreads();
      if (need && !gext_seen) atomicMax(&far_max, __float_as_int(dg));
    }
    for (int base = 0; base < count && __syncthreads_or(need && !gext_seen); base += kIbThreads) {
      const int t = base + tid;
      const float dmax = __int_as_float(far_max);  // no node of the tile looks farther than this
      Tri tr{};
      bool keep = t < count && load_tri(t, tr);
      Bound b{{0.0f, 0.0f, 0.0f}, -INFINITY, {0.0f, 0.0f, 0.0f}, INFINITY};
      if (keep && use_tris) {
        b = far_bound(tr, tc, rt, scale);
        const float hmax = (dot(tc, b.n) - b.d) + ((half.x * fabsf(b.n.x) + half.y * fabsf(b.n.y)) +
                                                   half.z * fabsf(b.n.z)) * 1.0001f;
        if (hmax <= -dmax) keep = false;
        if (hmax <= s.tol && norm(sub(tc, b.g)) * 0.9999f - rt >= (dmax + b.r) * 1.0001f) keep = false;
      }
      int total;
      const int slot = store_rec(keep, tr, t, total);
      if (slot >= 0) {
        plane[slot] = make_float4(b.n.x, b.n.y, b.n.z, b.d);
        ball[slot] = make_float4(b.g.x, b.g.y, b.g.z, b.r);
      }
      if (tid < kFarUnroll) {  // padding that no node visits
        plane[total + tid] = make_float4(0.0f, 0.0f, 0.0f, INFINITY);
        ball[total + tid] = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
      }
      __syncthreads();
      if (need && !gext_seen) {
        for (int q = 0; q < total && !gext_seen; q += kFarUnroll) {
          float h[kFarUnroll];
          bool any = false;
#pragma unroll
          for (int e = 0; e < kFarUnroll; ++e) {
            const float4 pl = plane[q + e];
            h[e] = ((p.x * pl.x + p.y * pl.y) + p.z * pl.z) - pl.w;
            any |= !(h[e] <= -dg);
          }
          if (!any) continue;
#pragma unroll 1
          for (int e = 0; e < kFarUnroll; ++e) {
            const float he = e == 0 ? h[0] : e == 1 ? h[1] : e == 2 ? h[2] : h[3];
            if (he <= -dg) continue;
            if (he <= s.tol) {
              const float4 g = ball[q + e];
              const V3 o = {p.x - g.x, p.y - g.y, p.z - g.z};
              const float reach = dg + g.w;
              if (dot(o, o) > reach * reach * 1.0001f) continue;
            }
            if (!visit(load_rec(q + e), rec_id[q + e])) {
              gext_seen = true;
              break;
            }
          }
        }
      }
    }
  }

  // 3. the chosen candidate, recomputed, and the node's fields
  int kind = kNodeNone;
  bool invalid = false;
  int sel = -1;
  bool far_internal = false;
  if (active) {
    if (tn >= 0) {
      sel = (ext_seen && te >= 0) ? te : tn;
      kind = ext_seen ? kNodeExternalIb : kNodeInternal;
    } else if (s.far && tg >= 0 && !gext_seen) {
      sel = tg;
      kind = kNodeInternal;
      far_internal = true;
    }
    const int64_t c = ((int64_t)i * s.ny + j) * s.nz + k;
    V3 bp{0.0f, 0.0f, 0.0f}, ip{0.0f, 0.0f, 0.0f}, w{0.0f, 0.0f, 0.0f};
    int marker = -1, idx[3] = {-1, -1, -1};
    float sd = 0.0f;
    if (sel >= 0) {
      V3 normal;
      if (use_tris) {
        int ia, ib, ic;
        tri_indices(s, sel, ia, ib, ic);
        const Tri tr = make_tri(s, ia, ib, ic);
        bp = closest_point(p, tr);
        normal = tr.n;
        w = barycentric(bp, tr);
        const V3 oa = sub(p, tr.a), ob = sub(p, tr.b), oc = sub(p, tr.c);
        float best = dot(oa, oa);
        marker = ia;
        const float db = dot(ob, ob);
        if (db < best) {
          best = db;
          marker = ib;
        }
        if (dot(oc, oc) < best) marker = ic;
        idx[0] = ia;
        idx[1] = ib;
        idx[2] = ic;
      } else {
        bp = ld3(s.xm, sel);
        normal = ld3(s.nm, sel);
        w = {1.0f, 0.0f, 0.0f};
        marker = sel;
        idx[0] = sel;
      }
      const V3 off = sub(p, bp);
      sd = dot(off, normal);
      if (far_internal) {
        ip = add(bp, mul(normal, s.probe));
      } else {
        const float nd = dot(off, normal);
        const float interior_distance = nd > s.tol ? nd + s.probe : s.probe;
        ip = add(bp, mul(normal, interior_distance));
        invalid = fabsf(sd) <= s.tol;
      }
    }
    s.kind[c] = kind;
    s.nearest[c] = marker;
    s.signed_distance[c] = sd;
    s.boundary[3 * c] = bp.x;
    s.boundary[3 * c + 1] = bp.y;
    s.boundary[3 * c + 2] = bp.z;
    s.interior[3 * c] = ip.x;
    s.interior[3 * c + 1] = ip.y;
    s.interior[3 * c + 2] = ip.z;
    s.proj_idx[3 * c] = idx[0];
    s.proj_idx[3 * c + 1] = idx[1];
    s.proj_idx[3 * c + 2] = idx[2];
    s.proj_w[3 * c] = w.x;
    s.proj_w[3 * c + 1] = w.y;
    s.proj_w[3 * c + 2] = w.z;
  }
  const int near_count = __syncthreads_count(active && tn >= 0);
  const int ext_count = __syncthreads_count(active && tn >= 0 && ext_seen);
  const int int_count = __syncthreads_count(active && kind == kNodeInternal);
  const int inv_count = __syncthreads_count(active && invalid);
  if (tid == 0) {
    if (near_count) atomicAdd(&s.report[0], near_count);
    if (ext_count) atomicAdd(&s.report[1], ext_count);
    if (int_count) atomicAdd(&s.report[2], int_count);
    if (inv_count) atomicAdd(&s.report[3], inv_count);
  }
}

}  // namespace

extern "C" {

int hfsi_ib_node_search(int32_t nx, int32_t ny, int32_t nz, const float* bounds_min3, const float* spacing3,
                        const float* center_x, const float* center_y, const float* center_z,
                        const hfsi_ib_markers* m, float search_radius, float interior_probe_distance,
                        float sign_tolerance, int32_t classify_far_internal_nodes, const hfsi_ib_nodes* out,
                        int32_t* report4, void* stream) {
  const bool centres = center_x || center_y || center_z;
  if (nx <= 0 || ny <= 0 || nz <= 0 || !m || !out || !report4 || !m->positions || !m->normals ||
      m->marker_count < 0 || m->triangle_count < 0 || (m->triangle_count > 0 && !m->triangles) ||
      (centres && !(center_x && center_y && center_z)) || (!centres && !(bounds_min3 && spacing3)) ||
      !out->kind || !out->nearest_marker || !out->signed_distance || !out->boundary_point ||
      !out->interior_point || !out->projection_indices || !out->projection_weights) {
    set_error("hfsi_ib_node_search: invalid arguments");
    return HFSI_ERR_ARG;
  }
  if (!(search_radius > 0.0f) || !std::isfinite(search_radius) || !(interior_probe_distance > 0.0f) ||
      !std::isfinite(interior_probe_distance) || !(sign_tolerance >= 0.0f) || !std::isfinite(sign_tolerance)) {
    set_error("hfsi_ib_node_search: search_radius and interior_probe_distance must be finite and positive, "
              "sign_tolerance finite and non-negative");
    return HFSI_ERR_ARG;
  }
  const int64_t tiles = (int64_t)((nx + kTileI - 1) / kTileI) * ((ny + kTileJ - 1) / kTileJ) *
                        ((nz + kTileK - 1) / kTileK);
  if (tiles > 0x7fffffff || (int64_t)nx * ny * nz > (int64_t)1 << 31) {
    set_error("hfsi_ib_node_search: node grid too large");
    return HFSI_ERR_ARG;
  }
  SearchArgs a{};
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  for (int d = 0; d < 3; ++d) {
    a.bmin[d] = centres ? 0.0f : bounds_min3[d];
    a.spacing[d] = centres ? 0.0f : spacing3[d];
  }
  a.cx = center_x;
  a.cy = center_y;
  a.cz = center_z;
  a.xm = m->positions;
  a.nm = m->normals;
  a.tris = m->triangles;
  a.markers = m->marker_count;
  a.triangles = m->triangle_count;
  a.radius = search_radius;
  a.probe = interior_probe_distance;
  a.tol = sign_tolerance;
  a.far = classify_far_internal_nodes ? 1 : 0;
  a.kind = out->kind;
  a.nearest = out->nearest_marker;
  a.signed_distance = out->signed_distance;
  a.boundary = out->boundary_point;
  a.interior = out->interior_point;
  a.proj_idx = out->projection_indices;
  a.proj_w = out->projection_weights;
  a.report = report4;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_ib_zero_report, dim3(1), dim3(64), 0, st, report4);
  hipLaunchKernelGGL(k_ib_search, dim3((uint32_t)tiles), dim3(kIbThreads), 0, st, a);
  HFSI_LAUNCH_CHECK();
  return HFSI_OK;
}

}  // extern "C"

}  // namespace hfsi
