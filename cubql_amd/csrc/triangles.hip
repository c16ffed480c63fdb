// triangles.hip -- closest point on a triangle mesh, and distance adjoints.
//
// Forward: replaces cuBQL::triangles::findClosest / closestPoint
// (queries/triangles/findClosest.h:56-152) as a batched kernel, one query
// per lane, over an indexed mesh (tris[3i..3i+2] index verts) or, when tris
// is NULL, the reference's non-indexed Triangle array (verts[9i..9i+8]).
// The per-triangle test is the reference's: N = (b-a)x(c-a); outside if
// N == 0 or q lies beyond any edge plane, then the closest of the three
// clamped edge projections; else the plane distance along
// normalize(N) = N*(1/sqrt(N.N)).  Float32 with contraction off; among equal
// distances the lowest triangle id wins.
//
// Backward (no reference counterpart): recomputes the closest feature of
// the saved triangle id -- no traversal state is stored -- and applies the
// envelope theorem: for d = |q - P|, P = sum_j w_j v_j,
//   dd/dq = (q-P)/d,  dd/dv_j = -w_j (q-P)/d,   (0 at d == 0)
// with w the barycentric weights of P (face: projection barycentrics,
// edge: (1-t, t), vertex: one-hot).  Vertex gradients are scatter-added.
#include "common.h"
#include "cubql_amd/traversal.hip.h"
#include "cubql_amd/triangle.hip.h"
#include "profile.h"
#include "query_order.h"
#include "radix_sort.h"
#include "wave_closest.h"

namespace cubql {
namespace tri {

constexpr int kBlock = 256;
constexpr int kFastStack = 64;
constexpr int kDeepStack = 1024;
// id of a query whose traversal needed more than kDeepStack entries
constexpr int32_t kIncomplete = -2;

using namespace cubql_dev;

struct Overflow { uint32_t count, deepFailed; };

template <int STACK, typename Stats = NoStats>
__device__ __forceinline__ bool fcp_tri_one(const cubql_bvh3f &bvh, const int32_t *tris, const float *verts,
                                            F3 q, float sqrMax, int32_t &best, float &bestD, F3 &bestP,
                                            Stats &&st = Stats()) {
  best = -1;
  bestD = sqrMax;
  bestP = {0.f, 0.f, 0.f};
  auto prim = [&](uint32_t t) -> float {
    st.prim();
    F3 a, b, c, P;
    tri_verts(tris, verts, t, a, b, c);
    float w[3];
    const float d = tri_closest<false>(a, b, c, q, P, w);
    if (d < bestD || (d == bestD && best >= 0 && (int32_t)t < best)) {
      bestD = d;
      best = (int32_t)t;
      bestP = P;
    }
    return bestD;
  };
  // seed the radius with the nearest-child leaf, which the traversal then
  // leaves out
  const uint32_t seed = cubql_dev::visit_nearest_leaf(bvh, q.x, q.y, q.z, prim, 0u, st);
  return cubql_dev::for_each_prim_except<STACK>(bvh, q.x, q.y, q.z, bestD, prim, seed, 0u, st);
}

// the mesh in primID-slot order: a and the triangle id's bits, b, c
__global__ __launch_bounds__(256) void k_slot_tris(const uint32_t *primIDs, uint32_t numPrims, const int32_t *tris,
                                                   const float *verts, float4 *stris) {
  for (uint32_t s = blockIdx.x * 256 + threadIdx.x; s < numPrims; s += gridDim.x * 256) {
    const uint32_t t = primIDs[s];
    F3 a, b, c;
    tri_verts(tris, verts, t, a, b, c);
    stris[3 * (size_t)s] = make_float4(a.x, a.y, a.z, __uint_as_float(t));
    stris[3 * (size_t)s + 1] = make_float4(b.x, b.y, b.z, 0.f);
    stris[3 * (size_t)s + 2] = make_float4(c.x, c.y, c.z, 0.f);
  }
}

__device__ __forceinline__ void write_result(uint32_t qi, int32_t best, float bestD, F3 P, int32_t *ids,
                                             float *d2, float *cp) {
  ids[qi] = best;
  if (d2) d2[qi] = best >= 0 ? bestD : INFINITY;
  if (cp) {
    cp[3 * (size_t)qi] = P.x;
    cp[3 * (size_t)qi + 1] = P.y;
    cp[3 * (size_t)qi + 2] = P.z;
  }
}

// Closest triangles.  A float triangle distance can be less than the distance
// of a box around the triangle, so which triangles a query meets depends on
// its visiting order: every query keeps its own traversal (the seeding descent
// and then the nearer child first, as fcp_tri_one), one query per lane.  The
// lanes share the tests: the (query, triangle) pairs of all lanes at a leaf
// are dealt out over the wave, 64 at a time, and the least key (distance bits
// << 32 | id) of a query is kept in LDS with its closest point.  One lane's
// leaf at a time a test, a hundred instructions and three 16-byte loads, ran
// with 12% of the lanes on.  The wave takes the step most lanes wait for:
// expanding a node, popping the stack or testing.  4M queries of 1.3M
// triangles: 3.94 ms with each lane testing its own leaf, 2.49 ms here, bound by
// VALU issue (99%).  Slower: 4 to 12 stack entries in LDS (fewer waves), lanes
// that take a new query when they are done (waves of several hundred queries end
// far apart), scalar loads where all lanes are at one node.
constexpr int kTriLeafMax = 8;  // triangles of a lane's leaf dealt out at once

struct WaveTris {
  unsigned long long best[kWave];
  float q[3][kWave];
  float P[3][kWave];
  uint32_t off[kWave];
  uint16_t pair[kTriLeafMax * kWave];
};

template <bool kSorted>
__global__ __launch_bounds__(kBlock) void k_fcp_tris(cubql_bvh3f bvh, const int32_t *tris, const float *verts,
                                                     const float4 *stris, const float *queries, uint32_t nq,
                                                     uint32_t qpw, float sqrMax, int32_t *ids, float *d2, float *cp,
                                                     Overflow *ovf, uint32_t *ovfList, const uint32_t *order) {
  __shared__ WaveTris share[kBlock / kWave];
  WaveTris &sh = share[threadIdx.x / kWave];
  const uint32_t lane = lane_id();
  // spatially ordered queries: contiguous runs of them per XCD
  const uint32_t blk = order ? xcd_chunk(blockIdx.x, gridDim.x) : blockIdx.x;
  const uint64_t i = (uint64_t)(blk * (kBlock / kWave) + threadIdx.x / kWave) * qpw + lane;
  const bool live = lane < qpw && i < nq;
  const uint32_t qi = live ? (order ? order[i] : (uint32_t)i) : 0u;
  F3 q = {0.f, 0.f, 0.f};
  if (live) q = ld3(queries, qi);
  const uint64_t root = bvh.nodes[0].offsetAndCountBits;
  const unsigned long long none = closest_none(sqrMax);
  sh.q[0][lane] = q.x;
  sh.q[1][lane] = q.y;
  sh.q[2][lane] = q.z;
  sh.best[lane] = none;
  sh.P[0][lane] = sh.P[1][lane] = sh.P[2][lane] = 0.f;
  sync_wave_lds();
  enum : uint32_t { kDone, kInner, kLeaf, kPop };
  PrivateStack<kFastStack> stack;
  uint32_t state = kDone, off = 0, cnt = 0, start = 0, seed = 0;
  int sp = 0;
  bool seeding = true, failed = false;
  float cull = 0.f;
  // where a node's word leads: an inner node, or a leaf, which the traversal
  // leaves out if it seeded the query
  auto enter = [&](uint64_t word) __attribute__((always_inline)) {
    off = oc_off(word);
    cnt = oc_cnt(word);
    start = off;
    state = cnt == 0 ? kInner : seeding || off != seed ? kLeaf : kPop;
  };
  if (live) enter(root);
  while (true) {
    // the step most lanes wait for (one that has a lane: without inner
    // nodes and leaves nPop is the largest)
    const uint32_t nInner = __popcll(__ballot(state == kInner)), nLeaf = __popcll(__ballot(state == kLeaf)),
                   nPop = __popcll(__ballot(state == kPop));
    if (nInner + nLeaf + nPop == 0) break;
    if (nPop > max(nInner, nLeaf)) {
      if (state == kPop) {
        if (sp == 0) {
          state = kDone;
        } else {
          const uint2 e = stack.get(--sp);
          if (__uint_as_float(e.y) <= cull) enter(bvh.nodes[e.x].offsetAndCountBits);
        }
      }
    } else if (nInner && nInner >= nLeaf) {
      if (state == kInner) {
        const QNode n0 = load_node(bvh.nodes, off), n1 = load_node(bvh.nodes, off + 1);
        const float d0 = sqr_dist_box(q.x, q.y, q.z, n0), d1 = sqr_dist_box(q.x, q.y, q.z, n1);
        const bool near0 = d0 < d1;
        const float far = fmaxf(d0, d1);
        bool go = true;
        if (!seeding) {
          go = !(fminf(d0, d1) > cull);
          if (go && far <= cull) {
            if (sp < kFastStack) {
              stack.put(sp++, make_uint2(near0 ? off + 1 : off, __float_as_uint(far)));
            } else {
              failed = true;  // deeper than the stack: the deep kernel runs it again
              go = false;
              sp = 0;
            }
          }
        }
        if (go) enter(near0 ? node_oc(n0) : node_oc(n1));
        else state = kPop;
      }
    } else {
      // deal out the tests: pair[] holds the owner's lane and the triangle's
      // number in its leaf
      const uint32_t c = state == kLeaf ? min(cnt, (uint32_t)kTriLeafMax) : 0u;
      uint32_t at = 0, total = 0;
#pragma unroll
      for (int b = 0; (1 << b) <= kTriLeafMax; b++) {
        const uint64_t m = __ballot((c >> b) & 1u);
        at += mbcnt(m) << b;
        total += (uint32_t)__popcll(m) << b;
      }
      sh.off[lane] = off;
      for (uint32_t j = 0; j < c; j++) sh.pair[at + j] = (uint16_t)(lane | j << 6);
      sync_wave_lds();
      for (uint32_t base = 0; base < total; base += kWave) {
        if (base + lane < total) {
          const uint32_t pr = sh.pair[base + lane], o = pr & 63u;
          const uint32_t slot = sh.off[o] + (pr >> 6);
          F3 a, b, cc, P;
          uint32_t t;
          if constexpr (kSorted) {
            const float4 va = stris[3 * (size_t)slot], vb = stris[3 * (size_t)slot + 1],
                         vc = stris[3 * (size_t)slot + 2];
            a = {va.x, va.y, va.z};
            b = {vb.x, vb.y, vb.z};
            cc = {vc.x, vc.y, vc.z};
            t = __float_as_uint(va.w);
          } else {
            t = bvh.primIDs[slot];
            tri_verts(tris, verts, t, a, b, cc);
          }
          float w[3];
          const float d = tri_closest<false>(a, b, cc, {sh.q[0][o], sh.q[1][o], sh.q[2][o]}, P, w);
          const unsigned long long key = closest_key(d, t);
          const unsigned long long old = atomicMin(&sh.best[o], key);
          sync_wave_lds();
          // (ids differ: only the lane that holds the least key writes)
          if (key < old && sh.best[o] == key) {
            sh.P[0][o] = P.x;
            sh.P[1][o] = P.y;
            sh.P[2][o] = P.z;
          }
        }
        sync_wave_lds();
      }
      if (state == kLeaf) {
        off += c;
        cnt -= c;
        if (cnt == 0) {
          cull = __uint_as_float((uint32_t)(sh.best[lane] >> 32));
          state = kPop;
          if (seeding) {
            seeding = false;
            seed = start;
            enter(root);
          }
        }
      }
    }
  }
  if (!live) return;
  if (failed) {
    ovfList[atomicAdd(&ovf->count, 1u)] = qi;
    return;
  }
  const unsigned long long best = sh.best[lane];
  const bool found = best != none;
  write_result(qi, found ? (int32_t)(uint32_t)best : -1, __uint_as_float((uint32_t)(best >> 32)),
               {sh.P[0][lane], sh.P[1][lane], sh.P[2][lane]}, ids, d2, cp);
}

__global__ __launch_bounds__(64) void k_fcp_tris_deep(cubql_bvh3f bvh, const int32_t *tris, const float *verts,
                                                      const float *queries, float sqrMax, int32_t *ids,
                                                      float *d2, float *cp, Overflow *ovf,
                                                      const uint32_t *ovfList) {
  const uint32_t n = ovf->count;
  for (uint32_t i = blockIdx.x * 64 + threadIdx.x; i < n; i += gridDim.x * 64) {
    const uint32_t qi = ovfList[i];
    const F3 q = ld3(queries, qi);
    int32_t best;
    float bestD;
    F3 P;
    if (!fcp_tri_one<kDeepStack>(bvh, tris, verts, q, sqrMax, best, bestD, P)) {
      // deeper than the deep stack: marked incomplete, not "none found"
      atomicAdd(&ovf->deepFailed, 1u);
      best = kIncomplete;
    }
    write_result(qi, best, bestD, P, ids, d2, cp);
  }
}

__global__ void k_tri_boxes(const int32_t *tris, const float *verts, uint32_t n, cubql_box3f *boxes) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    F3 a, b, c;
    tri_verts(tris, verts, i, a, b, c);
    cubql_box3f bx;  // Triangle::bounds() (Triangle.h:35-36)
    bx.lower[0] = fminf(fminf(a.x, b.x), c.x);
    bx.lower[1] = fminf(fminf(a.y, b.y), c.y);
    bx.lower[2] = fminf(fminf(a.z, b.z), c.z);
    bx.upper[0] = fmaxf(fmaxf(a.x, b.x), c.x);
    bx.upper[1] = fmaxf(fmaxf(a.y, b.y), c.y);
    bx.upper[2] = fmaxf(fmaxf(a.z, b.z), c.z);
    boxes[i] = bx;
  }
}

// Each query's terms for the three vertices go through LDS so that three
// neighbouring lanes add x, y and z of one vertex: the memory side takes one
// request per vertex instead of three.  Bound by those requests (4M queries,
// 1.3M triangles: 348 us with one, 1841 us with three).
__global__ __launch_bounds__(kBlock) void k_tri_backward(const int32_t *tris, const float *verts,
                                                         const float *queries, uint32_t nq,
                                                         const int32_t *ids, const float *gradDist,
                                                         float *gradQ, float *gradV) {
  __shared__ uint32_t sVert[kBlock * 3];
  __shared__ float sTerm[kBlock * 9];
  const uint32_t qi = blockIdx.x * kBlock + threadIdx.x;
  const bool act = qi < nq;
  const int32_t t = act ? ids[qi] : -1;
  F3 gq = {0.f, 0.f, 0.f};
  float w[3] = {0.f, 0.f, 0.f};
  uint32_t v[3] = {0u, 0u, 0u};
  if (t >= 0) {
    const F3 q = ld3(queries, qi);
    F3 a, b, c, P;
    for (int j = 0; j < 3; j++) v[j] = tris ? (uint32_t)tris[3 * (size_t)t + j] : 3u * (uint32_t)t + j;
    a = ld3(verts, v[0]);
    b = ld3(verts, v[1]);
    c = ld3(verts, v[2]);
    const float s = tri_closest<true>(a, b, c, q, P, w);
    const float d = sqrtf(s);
    if (d > 0.f) {
      gq = mul(gradDist[qi] / d, sub(q, P));
    } else {
      w[0] = w[1] = w[2] = 0.f;
    }
  }
  if (gradQ && act) {
    gradQ[3 * (size_t)qi] = gq.x;
    gradQ[3 * (size_t)qi + 1] = gq.y;
    gradQ[3 * (size_t)qi + 2] = gq.z;
  }
  if (!gradV) return;
  // a wave's own part of the arrays: no barrier is needed
  const uint32_t lane = lane_id(), w0 = threadIdx.x - lane;
  uint32_t *const wv = sVert + 3 * w0;
  float *const wt = sTerm + 9 * w0;
#pragma unroll
  for (int j = 0; j < 3; j++) {
    wv[3 * lane + j] = v[j];
    wt[9 * lane + 3 * j + 0] = -w[j] * gq.x;
    wt[9 * lane + 3 * j + 1] = -w[j] * gq.y;
    wt[9 * lane + 3 * j + 2] = -w[j] * gq.z;
  }
  sync_wave_lds();
#pragma unroll
  for (uint32_t i = 0; i < 9; i++) {
    const uint32_t c = i * kWave + lane;
    const float term = wt[c];
    if (term != 0.f) atomicAdd(&gradV[3 * (size_t)wv[c / 3] + c % 3], term);
  }
}

// The term of entry (query, neighbour) of a point distance: gradDist / d *
// (q - p), or false where it contributes nothing.
__device__ __forceinline__ bool point_term(F3 q, F3 p, const float *gradDist, size_t e, F3 &g) {
  const F3 diff = sub(q, p);
  const float d = sqrtf(dot(diff, diff));
  g = {0.f, 0.f, 0.f};
  if (!(d > 0.f)) return false;
  g = mul(gradDist[e] / d, diff);
  return true;
}

// points: d = |q-p| for each (query, neighbour) entry e = qi*k + j, a thread
// per entry so that ids, weights and keys are read and written in order
// (2M x 16 entries: 655 us, bound by the gather of the points; 2150 us with a
// thread per query, which strides).
// The query gradient is the sum of its terms in entry order, taken from LDS.
// The point gradient is not scattered here: when key is given, gv[e] is the
// entry's point term and key[e] its sort key (the point id, or numPoints for
// entries that contribute nothing).
constexpr uint32_t kBackEntries = 1024;  // terms of a workgroup, in LDS
__global__ __launch_bounds__(kBlock) void k_point_backward(const float *points, const float *queries,
                                                           uint32_t nq, uint32_t k, uint32_t perBlock,
                                                           const int32_t *ids, const float *gradDist, float *gradQ,
                                                           float *gv, uint32_t *key, uint32_t numPoints) {
  __shared__ float sT[3 * kBackEntries];
  const uint32_t q0 = blockIdx.x * perBlock;
  const uint32_t nHere = min(perBlock, nq - q0);
  const uint32_t kc = min(k, kBackEntries);
  float carry = 0.f;  // (k > kBackEntries: a query's sum so far, one query here)
  for (uint32_t j0 = 0; j0 < k; j0 += kc) {
    const uint32_t kn = min(kc, k - j0);  // (several queries: all k)
    for (uint32_t i = threadIdx.x; i < nHere * kn; i += kBlock) {
      const uint32_t qi = q0 + i / kn;
      const size_t e = (size_t)qi * k + j0 + i % kn;
      const int32_t p = ids[e];
      F3 g = {0.f, 0.f, 0.f};
      const bool live = p >= 0 && point_term(ld3(queries, qi), ld3(points, (size_t)p), gradDist, e, g);
      sT[3 * i] = g.x;
      sT[3 * i + 1] = g.y;
      sT[3 * i + 2] = g.z;
      if (key) {
        gv[3 * e] = -g.x;
        gv[3 * e + 1] = -g.y;
        gv[3 * e + 2] = -g.z;
        key[e] = live && (uint32_t)p < numPoints ? (uint32_t)p : numPoints;
      }
    }
    if (!gradQ) continue;
    sync_block_lds();
    for (uint32_t c = threadIdx.x; c < 3 * nHere; c += kBlock) {
      const float *t = sT + 3 * (size_t)(c / 3) * kn + c % 3;
      float sum = carry;
      for (uint32_t j = 0; j < kn; j++) sum += t[3 * j];
      if (j0 + kn < k) carry = sum;
      else gradQ[3 * (size_t)q0 + c] = sum;
    }
    sync_block_lds();
  }
}

// The point gradient from the entries sorted by point id: each wave sums
// its runs of equal ids (contiguous after the sort) with a segmented scan;
// a run inside the wave holds all of its point's entries, so it is added
// with a plain read-modify-write, and only runs that touch the wave's first
// or last lane (which may continue in the next or previous wave) use
// atomics.  No float atomic per entry, and the sum order inside a run is
// fixed.  Bound by the gather of the terms, a line each (2M x 16 entries:
// 1150 us; as much with 16-byte terms in one load, 1385 us computing the terms
// again from the query and the weight).
__global__ __launch_bounds__(kBlock) void k_point_scatter(const uint32_t *key, const uint32_t *val,
                                                          const float *gv, uint32_t n, uint32_t numPoints,
                                                          float *gradP) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t lane = lane_id();
  const bool act = i < n;
  const uint32_t p = act ? key[i] : numPoints;
  float sx = 0.f, sy = 0.f, sz = 0.f;
  if (act && p < numPoints) {
    const F3 g = ld3(gv, val[i]);
    sx = g.x;
    sy = g.y;
    sz = g.z;
  }
  const uint32_t pPrev = (uint32_t)__shfl_up((int)p, 1, kWave);
  const bool head = lane == 0 || pPrev != p;
  bool seen = head;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const float ux = __shfl_up(sx, o, kWave), uy = __shfl_up(sy, o, kWave), uz = __shfl_up(sz, o, kWave);
    const bool us = __shfl_up((int)seen, o, kWave) != 0;
    if (lane >= (uint32_t)o && !seen) {
      sx += ux; sy += uy; sz += uz;
      seen = us;
    }
  }
  const uint32_t pNext = (uint32_t)__shfl_down((int)p, 1, kWave);
  const bool runEnd = lane == kWave - 1 || pNext != p;
  // lane 0 of a run: the lane where the run starts (a ballot over heads)
  const uint64_t heads = __ballot(head);
  const uint64_t below = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1));
  const uint32_t runStart = 63u - (uint32_t)__builtin_clzll(below);
  if (runEnd && p < numPoints) {
    float *o = gradP + 3 * (size_t)p;
    if (runStart == 0 || lane == kWave - 1) {
      atomicAdd(&o[0], sx);
      atomicAdd(&o[1], sy);
      atomicAdd(&o[2], sz);
    } else {
      o[0] += sx;
      o[1] += sy;
      o[2] += sz;
    }
  }
}

__global__ void k_fill_nf(uint32_t nq, int32_t *ids, float *d2) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nq; i += gridDim.x * blockDim.x) {
    ids[i] = -1;
    if (d2) d2[i] = INFINITY;
  }
}

}  // namespace tri
}  // namespace cubql

using namespace cubql;

extern "C" int cubql_triangle_boxes_f3(const int32_t *d_tris, const float *d_verts, uint32_t numTris,
                                       cubql_box3f *d_boxes, cubql_stream_t s) {
  clear_error();
  if (numTris == 0) return CUBQL_OK;
  if (!d_verts || !d_boxes) {
    set_error("cubql_triangle_boxes_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  tri::k_tri_boxes<<<std::min<uint32_t>(div_up(numTris, 256), 8192), 256, 0, (hipStream_t)s>>>(
      d_tris, d_verts, numTris, d_boxes);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

extern "C" int cubql_fcp_triangles_f3(const cubql_bvh3f *bvh, const int32_t *d_tris, const float *d_verts,
                                      const float *d_queries, uint32_t numQueries, float sqrMax,
                                      int32_t *d_outTriIDs, float *d_outSqrDist, float *d_outClosest,
                                      cubql_stream_t stream) {
  clear_error();
  if (!bvh || (numQueries && (!d_verts || !d_queries || !d_outTriIDs))) {
    set_error("cubql_fcp_triangles_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  if (numQueries == 0) return CUBQL_OK;
  hipStream_t s = (hipStream_t)stream;
  if (bvh->numNodes == 0) {
    tri::k_fill_nf<<<256, 256, 0, s>>>(numQueries, d_outTriIDs, d_outSqrDist);
    CUBQL_LAUNCH_CHECK();
    return CUBQL_OK;
  }
  Scratch scr(nullptr, s);
  tri::Overflow *ovf = nullptr;
  uint32_t *ovfList = nullptr;
  CUBQL_CHECK(scr.alloc(&ovf, 1));
  CUBQL_CHECK(scr.alloc(&ovfList, numQueries));
  CUBQL_CHECK(fill_u32((uint32_t *)ovf, 0u, 2, s));
  const uint32_t *order = nullptr;
  if (numQueries >= kQueryOrderMin) {
    char *w = nullptr;
    CUBQL_CHECK(scr.alloc(&w, query_order_ws_bytes(numQueries)));
    CUBQL_CHECK(query_order_ws(&bvh->nodes[0].bounds, bvh, {d_queries, numQueries, false}, s, w, &order));
  }
  // the slot-ordered copy of the mesh pays when the queries test at least
  // about as many triangles as the copy moves
  float4 *stris = nullptr;
  if (bvh->numPrims && numQueries >= kQueryOrderMin && (uint64_t)numQueries * 8 >= bvh->numPrims)
    CUBQL_CHECK(scr.alloc(&stris, 3 * (size_t)bvh->numPrims));
  const uint32_t qpw = queries_per_wave(numQueries);
  const uint32_t grid = div_up(div_up(numQueries, qpw), tri::kBlock / kWave);
  int ps = prof_begin(s);
  if (stris) {
    tri::k_slot_tris<<<std::max(1u, std::min(div_up(bvh->numPrims, 256u), 2048u)), 256, 0, s>>>(
        bvh->primIDs, bvh->numPrims, d_tris, d_verts, stris);
    tri::k_fcp_tris<true><<<grid, tri::kBlock, 0, s>>>(*bvh, d_tris, d_verts, stris, d_queries, numQueries, qpw,
                                                       sqrMax, d_outTriIDs, d_outSqrDist, d_outClosest, ovf, ovfList,
                                                       order);
  } else {
    tri::k_fcp_tris<false><<<grid, tri::kBlock, 0, s>>>(*bvh, d_tris, d_verts, nullptr, d_queries, numQueries, qpw,
                                                        sqrMax, d_outTriIDs, d_outSqrDist, d_outClosest, ovf,
                                                        ovfList, order);
  }
  prof_end(ps, s, "fcp_triangles");
  prof_set(ps, 20.0 * numQueries, numQueries);
  tri::k_fcp_tris_deep<<<64, 64, 0, s>>>(*bvh, d_tris, d_verts, d_queries, sqrMax, d_outTriIDs,
                                         d_outSqrDist, d_outClosest, ovf, ovfList);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

extern "C" int cubql_fcp_triangles_backward_f3(const int32_t *d_tris, const float *d_verts,
                                               const float *d_queries, uint32_t numQueries,
                                               const int32_t *d_triIDs, const float *d_gradDist,
                                               float *d_gradQueries, float *d_gradVerts,
                                               cubql_stream_t s) {
  clear_error();
  if (numQueries == 0) return CUBQL_OK;
  if (!d_verts || !d_queries || !d_triIDs || !d_gradDist) {
    set_error("cubql_fcp_triangles_backward_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  int ps = prof_begin((hipStream_t)s);
  tri::k_tri_backward<<<div_up(numQueries, tri::kBlock), tri::kBlock, 0, (hipStream_t)s>>>(
      d_tris, d_verts, d_queries, numQueries, d_triIDs, d_gradDist, d_gradQueries, d_gradVerts);
  prof_end(ps, (hipStream_t)s, "triangles_backward");
  prof_set(ps, (12.0 + 4.0 + 4.0 + 12.0 + 3 * 12.0 + 3 * 24.0) * numQueries, numQueries);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

extern "C" int cubql_points_distance_backward_f3(const float *d_points, uint32_t numPoints, const float *d_queries,
                                                 uint32_t numQueries, int k, const int32_t *d_ids,
                                                 const float *d_gradDist, float *d_gradQueries,
                                                 float *d_gradPoints, cubql_stream_t stream,
                                                 const cubql_mem_resource *mem) {
  clear_error();
  if (numQueries == 0) return CUBQL_OK;
  if (!d_points || !d_queries || !d_ids || !d_gradDist || k < 1) {
    set_error("cubql_points_distance_backward_f3: invalid argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  const size_t ne = (size_t)numQueries * (size_t)k;
  if (ne > 0xffffffffull || numPoints > 0x7fffffffu) {
    set_error("cubql_points_distance_backward_f3: %zu entries / %u points exceed the 32-bit entry index", ne,
              numPoints);
    return CUBQL_ERR_INVALID_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  const bool scatter = d_gradPoints && numPoints;
  ScratchArena scr(mem, s);
  float *gv = nullptr;
  uint32_t *kA = nullptr, *vA = nullptr, *kB = nullptr, *vB = nullptr, *cnt = nullptr;
  char *sortWs = nullptr;
  // key bits: enough for the sentinel numPoints
  int bits = 1;
  while (bits < 32 && (numPoints >> bits) != 0) bits++;
  if (scatter) {
    CUBQL_CHECK(scr.reserve(&gv, 3 * ne));
    CUBQL_CHECK(scr.reserve(&kA, ne));
    CUBQL_CHECK(scr.reserve(&vA, ne));
    CUBQL_CHECK(scr.reserve(&kB, ne));
    CUBQL_CHECK(scr.reserve(&vB, ne));
    CUBQL_CHECK(scr.reserve(&cnt, 1));
    CUBQL_CHECK(scr.reserve(&sortWs, radix_sort_ws_bytes((uint32_t)ne, bits)));
    CUBQL_CHECK(scr.commit());
    CUBQL_CHECK(fill_u32(cnt, (uint32_t)ne, 1, s));
  }
  int ps = prof_begin(s);
  if (scatter || d_gradQueries) {
    // a query's k terms stay in one workgroup's LDS
    const uint32_t perBlock = std::max(1u, tri::kBackEntries / (uint32_t)k);
    tri::k_point_backward<<<div_up(numQueries, perBlock), tri::kBlock, 0, s>>>(
        d_points, d_queries, numQueries, (uint32_t)k, perBlock, d_ids, d_gradDist, d_gradQueries, gv, kA,
        numPoints);
    CUBQL_LAUNCH_CHECK();
  }
  if (scatter) {
    uint32_t *kRes = nullptr, *vRes = nullptr;
    CUBQL_CHECK(radix_sort_iota_ws_u32(kA, vA, kB, vB, cnt, (uint32_t)ne, bits, s, sortWs, &kRes, &vRes));
    tri::k_point_scatter<<<div_up((uint32_t)ne, tri::kBlock), tri::kBlock, 0, s>>>(
        kRes, vRes, gv, (uint32_t)ne, numPoints, d_gradPoints);
    CUBQL_LAUNCH_CHECK();
  }
  prof_end(ps, s, "points_backward");
  prof_set(ps, (12.0 + 12.0 + k * (4.0 + 4.0 + 12.0 + 24.0)) * numQueries, numQueries);
  return CUBQL_OK;
}

// ------------------------------------------------- traversal statistics
namespace cubql {
namespace tri {

// Instrumented closest-triangle queries (deep stack): per query, bytes of
// node data loaded and triangles tested, summed into out[0], out[1];
// out[2] counts the queries.
__global__ __launch_bounds__(64) void k_fcp_tris_stats(cubql_bvh3f bvh, const int32_t *tris, const float *verts,
                                                       const float *queries, uint32_t nq, float sqrMax,
                                                       unsigned long long *out) {
  const uint32_t qi = blockIdx.x * 64 + threadIdx.x;
  TraversalCounts st;
  if (qi < nq) {
    int32_t best;
    float bestD;
    F3 P;
    fcp_tri_one<kDeepStack>(bvh, tris, verts, ld3(queries, qi), sqrMax, best, bestD, P, st);
  }
  unsigned long long nb = st.nodeBytes, np = st.prims;
  for (int o = 32; o > 0; o >>= 1) {
    nb += __shfl_xor(nb, o, 64);
    np += __shfl_xor(np, o, 64);
  }
  if (threadIdx.x == 0) {
    atomicAdd(&out[0], nb);
    atomicAdd(&out[1], np);
    atomicAdd(&out[2], (unsigned long long)min(64u, nq - blockIdx.x * 64));
  }
}

}  // namespace tri
}  // namespace cubql

extern "C" int cubql_query_stats_triangles_f3(const cubql_bvh3f *bvh, const int32_t *d_tris, const float *d_verts,
                                              const float *d_queries, uint32_t numQueries, float sqrMaxSearchDist,
                                              uint64_t *d_out, cubql_stream_t stream) {
  using namespace cubql;
  clear_error();
  if (!bvh || !d_verts || !d_out || (numQueries && !d_queries)) {
    set_error("cubql_query_stats_triangles_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  CUBQL_CHECK(fill_u32((uint32_t *)d_out, 0u, 6, s));
  if (numQueries == 0 || bvh->numNodes == 0) return CUBQL_OK;
  tri::k_fcp_tris_stats<<<div_up(numQueries, 64), 64, 0, s>>>(*bvh, d_tris, d_verts, d_queries, numQueries,
                                                              sqrMaxSearchDist, (unsigned long long *)d_out);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}
