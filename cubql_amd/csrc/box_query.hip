// box_query.hip -- batched fixed-box (range) queries.
//
// Replaces user kernels that call cuBQL::fixedBoxQuery::forEachPrim once
// per thread (traversal/fixedBoxQuery.h:42-160, 215-230) with a per-prim
// test of the prim's box against the query box: for every query box, the
// prims whose boxes overlap it (closed boxes, math/box.h:208-212), in the
// traversal's order (depth first, first child / lowest slot first).  A
// query per lane; binary and wide (W = 4, 8) trees.  Queries whose stack
// would overflow rerun with a deeper one.
//
// Large batches (kWalkMin), over a binary tree, run in spatial order
// (query_order.h), a wave of queries walking together, and read leaf prims
// from a copy of the prim boxes in primID-slot order.  1M boxes against
// themselves, leaves of 4: 1305 us with one query per lane in input order, on
// a private stack and with a gather per prim; 517 us here and 88 us for the
// order and the copy.  Bound by the wave's chain of 381 scalar loads, each
// waited for before the next address is known: a wave waits for memory 52% of
// its time and to issue 23%, with all 8 waves to a SIMD.  The busiest unit is
// the scalar one (12.5K instructions a wave: 0.33 ms at one a cycle for each
// CU); the VALU issues for 0.22 ms.
#include <type_traits>

#include "common.h"
#include "cubql_amd/traversal.hip.h"
#include "profile.h"
#include "query_order.h"
#include "uniform_load.h"

namespace cubql {
namespace bq {

// batches below this size walk the tree a query per lane, in input order
constexpr uint32_t kWalkMin = 3u << 17;
static_assert(kWalkMin >= kQueryOrderMin, "the walk takes ordered queries");

// prim boxes of a leaf that are read at once
constexpr int kLeafBoxes = 4;

constexpr int kBlock = 256;
constexpr int kFastStack = 64;
constexpr int kDeepStack = 1024;

struct Overflow { uint32_t count, deepFailed; };

__device__ __forceinline__ void load_box(const cubql_box3f *b, uint32_t i, float (&lo)[3], float (&hi)[3]) {
  const float2 *f = reinterpret_cast<const float2 *>(b + i);
  const float2 x = f[0], y = f[1], z = f[2];
  lo[0] = x.x; lo[1] = x.y; lo[2] = y.x;
  hi[0] = y.y; hi[1] = z.x; hi[2] = z.y;
}

// Collects up to maxOut overlapping prims into out[]; returns false on a
// stack overflow.  *count receives the number of overlapping prims.
template <int STACK, typename BVH>
__device__ __forceinline__ bool query_one(const BVH &bvh, const cubql_box3f *primBoxes, const float (&lo)[3],
                                          const float (&hi)[3], uint32_t maxOut, uint32_t *out, uint32_t &count) {
  count = 0;
  auto leaf = [&](const uint32_t *ids, uint32_t cnt) -> int {
    for (uint32_t j = 0; j < cnt; j++) {
      const uint32_t p = ids[j];
      float bl[3], bh[3];
      load_box(primBoxes, p, bl, bh);
      const bool ov = !(bh[0] < lo[0] || bh[1] < lo[1] || bh[2] < lo[2] || hi[0] < bl[0] || hi[1] < bl[1] ||
                        hi[2] < bl[2]);
      if (ov) {
        if (count < maxOut) out[count] = p;
        count++;
      }
    }
    return 0;
  };
  return cubql_dev::for_each_leaf_in_box<STACK>(bvh, lo, hi, leaf);
}

// prim boxes in primID-slot order: lo, hi.x | hi.y, hi.z, primID; clears *ovf
__global__ __launch_bounds__(256) void k_slot_boxes(const uint32_t *primIDs, uint32_t numPrims,
                                                    const cubql_box3f *primBoxes, float4 *sboxes, Overflow *ovf) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *ovf = Overflow{0u, 0u};
  for (uint32_t t = blockIdx.x * 256 + threadIdx.x; t < numPrims; t += gridDim.x * 256) {
    const uint32_t i = primIDs[t];
    float lo[3], hi[3];
    load_box(primBoxes, i, lo, hi);
    sboxes[2 * (size_t)t] = make_float4(lo[0], lo[1], lo[2], hi[0]);
    sboxes[2 * (size_t)t + 1] = make_float4(hi[1], hi[2], __uint_as_float(i), 0.f);
  }
}


// > 0 iff the boxes are apart: the largest gap over the axes.  a > b exactly
// where a - b > 0, and where a difference is NaN the comparison is false and
// the maximum passes it over.  Six subtractions and three maxima: six
// comparisons would be joined by scalar instructions, whose unit is this
// kernel's busiest (18.3K of them a wave and 670 us that way, 12.5K and 517 so).
__device__ __forceinline__ float box_gap(const float (&lo)[3], const float (&hi)[3], float lx, float ly, float lz,
                                         float hx, float hy, float hz) {
  const float a = fmaxf(fmaxf(lo[0] - hx, lx - hi[0]), lo[1] - hy);
  const float b = fmaxf(fmaxf(a, ly - hi[1]), lo[2] - hz);
  return fmaxf(b, lz - hi[2]);
}

// whether this lane's bit of a wave-uniform mask is set (the mask becomes the
// execution mask, no shift)
__device__ __forceinline__ bool lane_in(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// A wave of queries that are close to each other walks the tree together: the
// order of a box query (depth first, first child first) is the same for every
// query, so the wave visits each node that any of its queries overlaps once,
// with the mask of those queries, and every query meets its prims in its own
// order.  Nodes and prim boxes are wave-uniform reads.  The stack (second
// children still to visit) is four registers, entry i in lane i; deeper
// trees rerun in the deep kernel.
__global__ __launch_bounds__(kBlock) void k_box_query_wave(cubql_bvh3f bvh, const float4 *sboxes,
                                                           const cubql_box3f *queries, uint32_t nq, uint32_t maxOut,
                                                           uint32_t *outIDs, uint32_t *counts, Overflow *ovf,
                                                           uint32_t *ovfList, const uint32_t *order) {
  using namespace cubql_dev;
  const uint32_t i = xcd_chunk(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const bool live = i < nq;
  const uint32_t qi = live ? order[i] : 0u;
  float lo[3] = {0.f, 0.f, 0.f}, hi[3] = {0.f, 0.f, 0.f};
  if (live) load_box(queries, qi, lo, hi);
  uint32_t *out = outIDs + (size_t)qi * maxOut;  // (written only if maxOut > 0)
  uint32_t count = 0;
  uint64_t mask = __ballot(live);
  int sOff = 0, sCnt = 0, sLo = 0, sHi = 0, sp = 0;
  bool failed = false;
  const uint64_t root = node_oc(load_node(bvh.nodes, 0));
  uint32_t off = (uint32_t)__builtin_amdgcn_readfirstlane((int)oc_off(root));
  uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)oc_cnt(root));
  while (mask) {
    if (cnt == 0) {
      QNode n0, n1;
      load_pair_uniform(bvh.nodes, off, n0, n1);
      const uint64_t m0 = mask & ~__ballot(box_gap(lo, hi, n0.a.x, n0.a.y, n0.a.z, n0.a.w, n0.b.x, n0.b.y) > 0.f);
      const uint64_t m1 = mask & ~__ballot(box_gap(lo, hi, n1.a.x, n1.a.y, n1.a.z, n1.a.w, n1.b.x, n1.b.y) > 0.f);
      const uint64_t o0 = node_oc(n0), o1 = node_oc(n1);
      if (m0 && m1) {
        if (sp >= kWave) {
          failed = true;
          break;
        }
        const bool top = lane_id() == (uint32_t)sp;
        sOff = top ? (int)oc_off(o1) : sOff;
        sCnt = top ? (int)oc_cnt(o1) : sCnt;
        sLo = top ? (int)(uint32_t)m1 : sLo;
        sHi = top ? (int)(uint32_t)(m1 >> 32) : sHi;
        sp++;
      }
      if (m0 | m1) {
        mask = m0 ? m0 : m1;
        off = m0 ? oc_off(o0) : oc_off(o1);
        cnt = m0 ? oc_cnt(o0) : oc_cnt(o1);
        continue;
      }
    } else {
      const uniform_vec4 b = uniform_ptr(sboxes + 2 * (size_t)off);
      for (uint32_t j = 0; j < cnt; j += kLeafBoxes) {
        // (the array is padded by kLeafBoxes slots)
        vec4f u[kLeafBoxes], v[kLeafBoxes];
#pragma unroll
        for (int k = 0; k < kLeafBoxes; k++) {
          u[k] = b[2 * (j + k)];
          v[k] = b[2 * (j + k) + 1];
        }
#pragma unroll
        for (int k = 0; k < kLeafBoxes; k++) {
          if (j + k >= cnt) break;
          const uint64_t m =
              mask & ~__ballot(box_gap(lo, hi, u[k].x, u[k].y, u[k].z, u[k].w, v[k].x, v[k].y) > 0.f);
          if (m && lane_in(m)) {
            if (count < maxOut) out[count] = __float_as_uint(v[k].z);
            count++;
          }
        }
      }
    }
    if (sp == 0) break;
    sp--;
    off = (uint32_t)__builtin_amdgcn_readlane(sOff, sp);
    cnt = (uint32_t)__builtin_amdgcn_readlane(sCnt, sp);
    mask = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(sLo, sp) |
           ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(sHi, sp) << 32);
  }
  if (!live) return;
  if (failed) {
    ovfList[atomicAdd(&ovf->count, 1u)] = qi;
    return;
  }
  counts[qi] = count;
}

template <typename BVH>
__global__ __launch_bounds__(kBlock) void k_box_query(BVH bvh, const cubql_box3f *primBoxes,
                                                      const cubql_box3f *queries, uint32_t nq, uint32_t maxOut,
                                                      uint32_t *outIDs, uint32_t *counts, Overflow *ovf,
                                                      uint32_t *ovfList) {
  const uint32_t qi = blockIdx.x * kBlock + threadIdx.x;
  if (qi >= nq) return;
  float lo[3], hi[3];
  load_box(queries, qi, lo, hi);
  uint32_t count;
  if (!query_one<kFastStack>(bvh, primBoxes, lo, hi, outIDs ? maxOut : 0u,
                             outIDs ? outIDs + (size_t)qi * maxOut : nullptr, count)) {
    ovfList[atomicAdd(&ovf->count, 1u)] = qi;
    return;
  }
  counts[qi] = count;
}

template <typename BVH>
__global__ __launch_bounds__(64) void k_box_query_deep(BVH bvh, const cubql_box3f *primBoxes,
                                                       const cubql_box3f *queries, uint32_t maxOut,
                                                       uint32_t *outIDs, uint32_t *counts, Overflow *ovf,
                                                       const uint32_t *ovfList) {
  const uint32_t n = ovf->count;
  for (uint32_t i = blockIdx.x * 64 + threadIdx.x; i < n; i += gridDim.x * 64) {
    const uint32_t qi = ovfList[i];
    float lo[3], hi[3];
    load_box(queries, qi, lo, hi);
    uint32_t count;
    if (!query_one<kDeepStack>(bvh, primBoxes, lo, hi, outIDs ? maxOut : 0u,
                               outIDs ? outIDs + (size_t)qi * maxOut : nullptr, count)) {
      atomicAdd(&ovf->deepFailed, 1u);
      count = 0xffffffffu;
    }
    counts[qi] = count;
  }
}

__global__ void k_zero_counts(uint32_t *counts, uint32_t nq) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nq; i += gridDim.x * blockDim.x) counts[i] = 0;
}

template <typename BVH>
int run(const BVH &bvh, const cubql_box3f *primBoxes, const cubql_box3f *queries, uint32_t nq, uint32_t maxOut,
        uint32_t *outIDs, uint32_t *counts, hipStream_t s) {
  if (bvh.numNodes == 0) {
    k_zero_counts<<<std::min<uint32_t>(div_up(nq, 256), 4096), 256, 0, s>>>(counts, nq);
    CUBQL_LAUNCH_CHECK();
    return CUBQL_OK;
  }
  Scratch scr(nullptr, s);
  Overflow *ovf = nullptr;
  uint32_t *ovfList = nullptr;
  CUBQL_CHECK(scr.alloc(&ovf, 1));
  CUBQL_CHECK(scr.alloc(&ovfList, nq));
  const uint32_t *order = nullptr;
  float4 *sboxes = nullptr;
  if constexpr (std::is_same<BVH, cubql_bvh3f>::value) {
    // The shared walk pays while a wave's queries overlap mostly the same
    // nodes, that is while the queries are about as dense as the prims, and once
    // the batch outweighs the order and the copy (60 to 70 us).  Batches against
    // themselves, us without the walk / with it:
    //              140000      262144      300000      400000      1000000
    //   uniform    275 / 291   356 / 340   407 / 340   588 / 373   1262 / 666
    //   plane      137 / 178   179 / 198   209 / 211   289 / 226    657 / 388
    //   Gaussian   159 / 200   202 / 224   226 / 231   279 / 261    591 / 435
    //   sphere     128 / 195   172 / 211   195 / 227   270 / 247    597 / 387
    //   (leaves of 4; uniform boxes three times as long: 2165 / 800 and 5414 / 1057 at
    //   140000 and 400000; boxes that overlap next to nothing, a hundredth as long:
    //   65 / 128 and 135 / 160, in a sphere 63 / 147 and 133 / 194)
    // and 1M prims with half as many queries: uniform 770 / 544, sphere 317 / 319.
    if (nq >= kWalkMin && bvh.numPrims && (uint64_t)nq * 2 >= bvh.numPrims) {
      char *w = nullptr;
      CUBQL_CHECK(scr.alloc(&w, query_order_ws_bytes(nq)));
      CUBQL_CHECK(scr.alloc(&sboxes, 2 * ((size_t)bvh.numPrims + bq::kLeafBoxes)));
      CUBQL_CHECK(query_order_ws(&bvh.nodes[0].bounds, &bvh, {(const float *)queries, nq, true}, s, w, &order));
    }
  }
  if (!order) CUBQL_CHECK(fill_u32((uint32_t *)ovf, 0u, 2, s));
  int ps = prof_begin(s);
  if (order) {
    if constexpr (std::is_same<BVH, cubql_bvh3f>::value) {
      k_slot_boxes<<<std::max(1u, std::min(div_up(bvh.numPrims, 256u), 2048u)), 256, 0, s>>>(
          bvh.primIDs, bvh.numPrims, primBoxes, sboxes, ovf);
      k_box_query_wave<<<div_up(nq, kBlock), kBlock, 0, s>>>(bvh, sboxes, queries, nq, outIDs ? maxOut : 0u,
                                                                outIDs, counts, ovf, ovfList, order);
    }
  } else {
    k_box_query<BVH><<<div_up(nq, kBlock), kBlock, 0, s>>>(bvh, primBoxes, queries, nq, maxOut, outIDs, counts, ovf,
                                                           ovfList);
  }
  prof_end(ps, s, "box_query");
  prof_set(ps, 28.0 * nq, nq);
  k_box_query_deep<BVH><<<64, 64, 0, s>>>(bvh, primBoxes, queries, maxOut, outIDs, counts, ovf, ovfList);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

}  // namespace bq
}  // namespace cubql

using namespace cubql;

extern "C" int cubql_box_query_f3(const cubql_bvh3f *bvh, const cubql_box3f *d_primBoxes,
                                  const cubql_box3f *d_queryBoxes, uint32_t numQueries, uint32_t maxPerQuery,
                                  uint32_t *d_outIDs, uint32_t *d_counts, cubql_stream_t stream) {
  clear_error();
  if (!bvh || (numQueries && (!d_queryBoxes || !d_counts || (bvh->numNodes && !d_primBoxes)))) {
    set_error("cubql_box_query_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  if (numQueries == 0) return CUBQL_OK;
  return bq::run(*bvh, d_primBoxes, d_queryBoxes, numQueries, maxPerQuery, d_outIDs, d_counts,
                 (hipStream_t)stream);
}

extern "C" int cubql_box_query_wide_f3(const cubql_wbvh3f *bvh, int width, const cubql_box3f *d_primBoxes,
                                       const cubql_box3f *d_queryBoxes, uint32_t numQueries, uint32_t maxPerQuery,
                                       uint32_t *d_outIDs, uint32_t *d_counts, cubql_stream_t stream) {
  clear_error();
  if (!bvh || (width != 4 && width != 8) ||
      (numQueries && (!d_queryBoxes || !d_counts || (bvh->numNodes && !d_primBoxes)))) {
    set_error("cubql_box_query_wide_f3: invalid argument (width %d)", width);
    return CUBQL_ERR_INVALID_ARG;
  }
  if (numQueries == 0) return CUBQL_OK;
  hipStream_t s = (hipStream_t)stream;
  if (width == 4)
    return bq::run(cubql_dev::WideBVH<4>{(const float4 *)bvh->nodes, bvh->numNodes, bvh->primIDs, bvh->numPrims},
                   d_primBoxes, d_queryBoxes, numQueries, maxPerQuery, d_outIDs, d_counts, s);
  return bq::run(cubql_dev::WideBVH<8>{(const float4 *)bvh->nodes, bvh->numNodes, bvh->primIDs, bvh->numPrims},
                 d_primBoxes, d_queryBoxes, numQueries, maxPerQuery, d_outIDs, d_counts, s);
}
