// batch.hip -- batched build + bidirectional closest point + Chamfer adjoint
// over thousands of independent point-cloud pairs (no reference counterpart:
// the reference builds one BVH per call and syncs with the host every level).
//
// Build, for each side (source / target) at once:
//   * one workgroup per cloud computes the cloud's centroid bounds and its
//     30-bit Morton keys with that cloud's own quantizer (radix.h:41-70); the
//     sort key is (cloud << 30) | morton, the value the global point index;
//   * one stable onesweep radix sort over all keys (segmented Morton sort);
//   * one hierarchy per cloud over its sorted keys, which follows
//     radix.h:446-570 (leaf if <= T, equal keys split in the middle) and is
//     exactly the tree radix30Builder builds for the cloud alone, with its
//     exact bounds: runs of small clouds and the ranges of up to 16384 points
//     that large clouds are split into are built by one workgroup each, from
//     the roots down and back up, with the keys in LDS.
// Queries run over all clouds in Morton order of the query side, each from
// its cloud's root in the other side's forest, a wave sharing its queries'
// subtrees; the adjoint of
// loss[c] = mean_i d(s_i, T_c) + mean_j d(t_j, S_c) is scatter-added.  The
// whole sequence is a fixed number of launches on one stream with no host
// synchronisation and no allocation (caller workspace), so it can be
// captured in a HIP graph and replayed.
#include "block_ops.h"
#include "build_common.h"
#include "common.h"
#include "cubql_amd/traversal.hip.h"
#include "profile.h"
#include "radix_sort.h"
#include "wave_closest.h"

#include <algorithm>
#include <vector>

namespace cubql {
namespace bt {

constexpr int kCloudShift = 30;
constexpr uint32_t kNoRoot = 0xffffffffu;
constexpr uint32_t kNoSlot = 0xffffffffu;

struct Side {
  const float *pts;
  const uint32_t *off;  // numClouds + 1 offsets (device)
  uint32_t n;
  // persistent (kept for the queries)
  uint64_t *keys;       // sorted keys
  uint32_t *ids;        // sorted global point indices = primIDs of the forest
  float4 *spts;         // points in sorted order: x, y, z, global index (bits)
  uint32_t *nnS;        // per sorted query: sorted slot of its closest point
  float *d2S;           //   on the other side (kNoSlot if none) and its distance
  Node *nodes;          // capacity 2n + 2
  uint32_t *rootOf;     // numClouds
  uint32_t *ctr;        // counters, see C_* (C_WORDS words)
};

struct Temp {
  uint64_t *keysB;
  uint32_t *valsB;
  float *acc;           // 3 floats per point of a side
  uint4 *units;         // see k_bunits
  uint4 *open;          // ranges of large clouds, level by level: node, begin, end
  void *sortWs;
  uint32_t *ovf;        // [0] count, [1] deep failures, then the list
};

// [C_LSTART0 + l] start of level l in the list of open ranges
enum { C_N = 1, C_UNITS = 2, C_TICKET = 3, C_OPEN = 4, C_LEVELS = 5, C_LSTART0 = 256, C_WORDS = 512 };

// A unit has up to kUnit points (its keys, 64 KB of LDS, two workgroups to a
// CU).  Clouds of up to kBin points share one.
constexpr uint32_t kUnit = 16384, kBin = kUnit / 2;
// levels of a tree: 30 key bits, then halvings of equal keys (18 of them reach
// kUnit from 2^32, 14 reach one point from there)
constexpr int kTopLevels = 64, kUnitLevels = 64;

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  uint32_t x = v & 0x3ffu;
  x = (x | (x << 16)) & 0x030000ffu;
  x = (x | (x << 8)) & 0x0300f00fu;
  x = (x | (x << 4)) & 0x030c30c3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

// one workgroup per cloud: centroid bounds, quantizer, keys
__global__ __launch_bounds__(256) void k_bkeys(Side sd, uint32_t numClouds) {
  __shared__ float sb[12 * 4];
  const uint32_t c = blockIdx.x;
  const uint32_t b = sd.off[c], e = sd.off[c + 1];
  float v[12];
  for (int j = 0; j < 3; j++) { v[j] = INFINITY; v[j + 3] = -INFINITY; v[j + 6] = INFINITY; v[j + 9] = -INFINITY; }
  for (uint32_t i = b + threadIdx.x; i < e; i += 256) {
    for (int d = 0; d < 3; d++) {
      const float p = sd.pts[3 * (size_t)i + d];
      const float ce = 0.5f * (p + p);  // centre of the degenerate box (p, p)
      v[d] = fminf(v[d], ce);
      v[d + 3] = fmaxf(v[d + 3], ce);
    }
  }
  block_reduce_bounds<256>(v, sb);
  if (b == e) return;
  // Quantizer::init (radix.h:46-53), 10 bits per axis
  const float ext = fmaxf(fmaxf(v[3] - v[0], v[4] - v[1]), v[5] - v[2]);
  const float scale = 1024.f * (1.f / fmaxf(ext, 1e-20f));
  for (uint32_t i = b + threadIdx.x; i < e; i += 256) {
    uint32_t cell[3];
    for (int d = 0; d < 3; d++) {
      const float p = sd.pts[3 * (size_t)i + d];
      const float f = (0.5f * (p + p) - v[d]) * scale;
      cell[d] = min((uint32_t)f, 1023u);
    }
    const uint32_t m = spread10(cell[0]) | (spread10(cell[1]) << 1) | (spread10(cell[2]) << 2);
    sd.keys[i] = ((uint64_t)c << kCloudShift) | m;
    sd.ids[i] = i;
  }
}

// points in sorted order, with their global index in w: a leaf's prims are
// then one contiguous run for the refit and the queries.  Bound by the gathered
// lines: a thread per point, an XCD at neighbouring workgroups of points (a
// grid-stride loop over 1024 workgroups: 980 us for 2 x 38M points, 810 so)
__global__ __launch_bounds__(256) void k_bgather(Side sd) {
  const uint32_t t = xcd_chunk(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  if (t >= sd.n) return;
  const uint32_t i = sd.ids[t];
  sd.spts[t] = make_float4(sd.pts[3 * (size_t)i], sd.pts[3 * (size_t)i + 1], sd.pts[3 * (size_t)i + 2],
                           __uint_as_float(i));
}

// where a range of one cloud's sorted keys is split (all high words equal)
template <class Key>
__device__ __forceinline__ uint32_t find_split(const Key *keys, uint32_t b, uint32_t e) {
  const Key fk = keys[b], lk = keys[e - 1];
  if (fk == lk) return b + (e - b) / 2;
  const Key search = lk & ~(Key)(0x7fffffffu >> __clz((uint32_t)(fk ^ lk)));
  uint32_t lo = b, hi = e;
  while (hi > lo) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (keys[mid] < search) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint32_t first_cloud_from(const uint32_t *off, uint32_t numClouds, uint64_t at) {
  uint32_t lo = 0, hi = numClouds;
  while (hi > lo) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (off[mid] < at) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// The units the trees are built in: for each kBin points, the clouds that
// start there and have up to kBin points, as one unit (begin, end, first
// cloud, end cloud), and at most one larger cloud after them, a unit of its
// own or, above `most` points, an open range.  Nodes need no counter: a tree
// over points [b, e) has at most 2 (e - b) - 1 nodes, and a unit keeps its own
// in [2b, 2e).
__global__ __launch_bounds__(256) void k_bunits(Side sd, Temp tp, uint32_t numClouds, uint32_t most) {
  const uint32_t step = gridDim.x * 256, first = blockIdx.x * 256 + threadIdx.x;
  for (uint32_t c = first; c < numClouds; c += step)
    if (sd.off[c] == sd.off[c + 1]) sd.rootOf[c] = kNoRoot;
  for (uint32_t k = first; (uint64_t)k * kBin < sd.n; k += step) {
    const uint32_t c0 = first_cloud_from(sd.off, numClouds, (uint64_t)k * kBin);
    uint32_t c1 = first_cloud_from(sd.off, numClouds, ((uint64_t)k + 1) * kBin);
    if (c1 == c0) continue;
    const uint32_t b = sd.off[c1 - 1], e = sd.off[c1];
    if (e - b > kBin) {
      c1--;
      if (e - b <= most) {
        tp.units[atomicAdd(&sd.ctr[C_UNITS], 1u)] = make_uint4(b, e, c1, c1 + 1);
      } else {
        sd.rootOf[c1] = 2 * b + 1;
        tp.open[atomicAdd(&sd.ctr[C_OPEN], 1u)] = make_uint4(2 * b + 1, b, e, 0u);
      }
    }
    if (sd.off[c1] > sd.off[c0])
      tp.units[atomicAdd(&sd.ctr[C_UNITS], 1u)] = make_uint4(sd.off[c0], sd.off[c1], c0, c1);
  }
}

// One workgroup splits the open ranges, level by level, until none has more
// than `most` points; the parts become units of one node (begin, end, node,
// kNoRoot).  The children of a range that is split at s are nodes 2s and
// 2s + 1, which no unit uses: s begins one, and its own start at 2s + 2.
__global__ __launch_bounds__(1024) void k_btop(Side sd, Temp tp, uint32_t most) {
  __shared__ uint32_t sEnd;
  uint32_t start = 0, end = sd.ctr[C_OPEN];
  int level = 0;
  if (threadIdx.x == 0) sEnd = end;
  while (start < end) {
    __syncthreads();
    if (threadIdx.x == 0) sd.ctr[C_LSTART0 + level] = start;
    for (uint32_t i = start + threadIdx.x; i < end; i += 1024) {
      const uint4 r = tp.open[i];
      const uint32_t s = find_split(sd.keys, r.y, r.z);
      sd.nodes[r.x].oc = pack_oc(2 * (uint64_t)s, 0);
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const uint32_t b = h ? s : r.y, e = h ? r.z : s;
        if (e - b > most) tp.open[atomicAdd(&sEnd, 1u)] = make_uint4(2 * s + h, b, e, 0u);
        else tp.units[atomicAdd(&sd.ctr[C_UNITS], 1u)] = make_uint4(b, e, 2 * s + h, kNoRoot);
      }
    }
    __syncthreads();
    start = end;
    end = sEnd;
    level++;
  }
  if (threadIdx.x == 0) {
    sd.ctr[C_LEVELS] = (uint32_t)level;
    sd.ctr[C_LSTART0 + level] = end;
  }
}

__device__ __forceinline__ void fit_leaf(const Side &sd, Node *nd) {
  const uint64_t oc = nd->oc;
  const uint32_t cnt = oc_count(oc), o = (uint32_t)oc_offset(oc);
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint32_t j = 0; j < cnt; j += 4) {
    float4 p[4];
#pragma unroll
    for (int u = 0; u < 4; u++) p[u] = sd.spts[o + min(j + u, cnt - 1)];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const float x[3] = {p[u].x, p[u].y, p[u].z};
      for (int d = 0; d < 3; d++) {
        lo[d] = fminf(lo[d], x[d]);
        hi[d] = fmaxf(hi[d], x[d]);
      }
    }
  }
  for (int d = 0; d < 3; d++) { nd->lo[d] = lo[d]; nd->hi[d] = hi[d]; }
}

// an inner node from its children
__device__ __forceinline__ void fit_node(const Side &sd, Node *nd) {
  const uint32_t o = (uint32_t)oc_offset(nd->oc);
  const Node l = sd.nodes[o], r = sd.nodes[o + 1];
  for (int d = 0; d < 3; d++) {
    nd->lo[d] = fminf(l.lo[d], r.lo[d]);
    nd->hi[d] = fmaxf(l.hi[d], r.hi[d]);
  }
}

// bounds of the open ranges' nodes, the deepest level first
__global__ __launch_bounds__(1024) void k_btop_fit(Side sd, Temp tp) {
  for (int l = (int)sd.ctr[C_LEVELS] - 1; l >= 0; l--) {
    const uint32_t end = sd.ctr[C_LSTART0 + l + 1];
    for (uint32_t i = sd.ctr[C_LSTART0 + l] + threadIdx.x; i < end; i += 1024) fit_node(sd, &sd.nodes[tp.open[i].x]);
    __syncthreads();
  }
}

// The trees of the units: a workgroup takes the next unit, splits its ranges
// level by level with the keys in LDS, a thread per node (a node's range stands
// in its own offset and count until it is split), and then fits the levels'
// bounds from the last one up.  2 x 38M points in 4096 clouds: 0.70 ms a side,
// and 0.12 ms for the open ranges; 1.76 ms with two launches per level.  Bound
// by the latency of the levels.  (1024 threads, two workgroups to a CU; 512:
// the same, 256: 3% of the whole call slower.)
constexpr int kUnitBlock = 1024;
__global__ __launch_bounds__(kUnitBlock) void k_bunit(Side sd, Temp tp, uint32_t T) {
  __shared__ uint32_t sKey[kUnit];
  __shared__ uint32_t ss[kUnitBlock / kWave + 1], sLo[kUnitLevels], sHi[kUnitLevels];
  __shared__ uint32_t sUnit;
  const uint32_t numUnits = sd.ctr[C_UNITS], tid = threadIdx.x;
  for (;;) {
    if (tid == 0) sUnit = atomicAdd(&sd.ctr[C_TICKET], 1u);
    __syncthreads();
    const uint32_t u = sUnit;
    if (u >= numUnits) return;
    const uint4 un = tp.units[u];
    const uint32_t b = un.x, size = un.y - un.x;
    // (a unit of more points than kUnit is one leaf)
    if (size <= kUnit)
      for (uint32_t i = tid; i < size; i += kUnitBlock) sKey[i] = (uint32_t)sd.keys[b + i] & ((1u << kCloudShift) - 1);
    uint32_t lo, hi, at;
    if (un.w == kNoRoot) {
      lo = un.z;
      hi = lo + 1;
      at = 2 * b + 2;
      if (tid == 0) sd.nodes[lo].oc = pack_oc(b, size);
    } else {
      lo = hi = 2 * b;
      for (uint32_t c0 = un.z; c0 < un.w; c0 += kUnitBlock) {
        const uint32_t c = c0 + tid;
        const uint32_t cb = c < un.w ? sd.off[c] : 0u, ce = c < un.w ? sd.off[c + 1] : 0u;
        uint32_t tot;
        const uint32_t ex = block_excl_scan<kUnitBlock>(ce > cb ? 1u : 0u, ss, &tot);
        if (ce > cb) {
          sd.nodes[hi + ex].oc = pack_oc(cb, ce - cb);
          sd.rootOf[c] = hi + ex;
        }
        hi += tot;
      }
      at = (hi + 1) & ~1u;
    }
    int level = 0;
    const uint32_t level1 = at;
    while (lo < hi) {
      __syncthreads();
      if (tid == 0) {
        sLo[level] = lo;
        sHi[level] = hi;
      }
      const uint32_t first = at;
      for (uint32_t i0 = lo; i0 < hi; i0 += kUnitBlock) {
        const uint32_t node = i0 + tid;
        const uint64_t oc = node < hi ? sd.nodes[node].oc : 0ull;
        const uint32_t cnt = oc_count(oc), p = (uint32_t)oc_offset(oc);
        const bool split = cnt > T;
        uint32_t s = 0;
        if (split) s = b + find_split(sKey, p - b, p - b + cnt);
        uint32_t tot;
        const uint32_t ex = block_excl_scan<kUnitBlock>(split ? 1u : 0u, ss, &tot);
        if (split) {
          const uint32_t child = at + 2 * ex;
          sd.nodes[node].oc = pack_oc(child, 0);
          sd.nodes[child].oc = pack_oc(p, s - p);
          sd.nodes[child + 1].oc = pack_oc(s, p + cnt - s);
        }
        at += 2 * tot;
      }
      lo = first;
      hi = at;
      level++;
    }
    __syncthreads();
    // (all leaves together: they lie on several levels)
    for (int l = 0; l < 2; l++) {
      const uint32_t end = l ? at : sHi[0];
      for (uint32_t i = (l ? level1 : sLo[0]) + tid; i < end; i += kUnitBlock)
        if (oc_count(sd.nodes[i].oc)) fit_leaf(sd, &sd.nodes[i]);
    }
    __syncthreads();
    for (int l = level - 1; l >= 0; l--) {
      const uint32_t end = sHi[l];
      for (uint32_t i = sLo[l] + tid; i < end; i += kUnitBlock)
        if (!oc_count(sd.nodes[i].oc)) fit_node(sd, &sd.nodes[i]);
      __syncthreads();
    }
  }
}

// The closest point of one query in the tree at `root` on the deep stack: its
// global index (lowest among equal distances), its sorted slot and distance.
// Leaf prims are read from the sorted points, a contiguous run per leaf.
template <int STACK>
__device__ __forceinline__ bool fcp_forest(const Side &tgt, uint32_t root, float3 q, int32_t &best,
                                           uint32_t &bestSlot, float &bestD) {
  best = -1;
  bestSlot = kNoSlot;
  bestD = INFINITY;
  cubql_bvh3f bvh;
  bvh.nodes = (cubql_node3f *)tgt.nodes;
  bvh.numNodes = 2;
  bvh.primIDs = tgt.ids;  // only for leaf slot offsets: ids are not read
  bvh.numPrims = tgt.n;
  const float4 *spts = tgt.spts;
  auto leaf = [&](const uint32_t *ids, uint32_t cnt) -> float {
    const uint32_t off = (uint32_t)(ids - tgt.ids);
    for (uint32_t j = 0; j < cnt; j++) {
      const float4 p = spts[off + j];
      const float d = cubql_dev::sqr_dist_pt(p.x, p.y, p.z, q.x, q.y, q.z);
      const int32_t pid = (int32_t)__float_as_uint(p.w);
      if (d < bestD || (d == bestD && best >= 0 && pid < best)) {
        bestD = d;
        best = pid;
        bestSlot = off + j;
      }
    }
    return bestD;
  };
  return cubql_dev::for_each_leaf<STACK>(bvh, q.x, q.y, q.z, bestD, leaf, root);
}

// Least key of a leaf's points and the sorted slot it is at, four in flight.
struct LeafSlots {
  const float4 *spts;
  __device__ __forceinline__ unsigned long long operator()(uint32_t off, uint32_t cnt, float x, float y, float z,
                                                           uint32_t &at) const {
    unsigned long long best = ~0ull;
    for (uint32_t j = 0; j < cnt; j += 4) {
      float4 p[4];
#pragma unroll
      for (int u = 0; u < 4; u++) p[u] = spts[off + min(j + u, cnt - 1)];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const unsigned long long k =
            closest_key(cubql_dev::sqr_dist_pt(p[u].x, p[u].y, p[u].z, x, y, z), __float_as_uint(p[u].w));
        if (k < best) {
          best = k;
          at = off + min(j + u, cnt - 1);
        }
      }
    }
    return best;
  }
};

// (24 and 40 lanes: within 1%)
constexpr int kBatchLeafLanes = 32;

// queries of side `qs` against the forest of side `ts`, in Morton order of
// qs: a wave per qpw queries (wave_closest.h).  2 x 38M queries over 4096
// clouds: 16.5 ms with one query per lane on a private stack, 8.2 ms here;
// bound by the address unit (16-point leaves) and VALU issue.  (Held to 64
// registers: 8 waves to a SIMD, 3.83 ms a launch, 3.92 with 7.)
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(8)))
void k_bquery(Side qs, Side ts, uint32_t qpw, int32_t *nn, float *d2, uint32_t *ovf) {
  __shared__ WaveTasksAux tasks[BLOCK / kWave];
  const uint32_t wave = threadIdx.x / kWave, lane = lane_id();
  // queries sorted by (cloud, Morton key): contiguous runs of them per XCD
  const uint64_t i = (uint64_t)(xcd_chunk(blockIdx.x, gridDim.x) * (BLOCK / kWave) + wave) * qpw + lane;
  const bool act = lane < qpw && i < qs.n;
  const uint32_t t = act ? (uint32_t)i : 0u;
  const float4 qv = qs.spts[t];
  const uint32_t root = ts.rootOf[(uint32_t)(qs.keys[t] >> kCloudShift)];
  const bool live = act && root != kNoRoot;
  const uint64_t word = live ? ts.nodes[root].oc : 0ull;
  const unsigned long long none = closest_none(INFINITY);
  unsigned long long best = none;
  uint32_t slot = kNoSlot;
  // Queries that lost a task run again, eight at a time and then alone (the
  // queue holds more of each), and last in the deep kernel.
  uint64_t lost = 0, todo = __ballot(live);
  for (uint32_t together = kWave; todo; together /= 8) {
    uint64_t again = 0;
    while (todo) {
      const bool on = ((todo >> lane) & 1u) && mbcnt(todo) < together;
      bool failed;
      uint32_t at;
      const unsigned long long k =
          wave_closest<kBatchLeafLanes>(tasks[wave], (const cubql_node3f *)ts.nodes, on, word, qv.x, qv.y, qv.z, none,
                                        LeafSlots{ts.spts}, &failed, &at);
      todo &= ~__ballot(on);
      again |= __ballot(on && failed);
      if (on && !failed) {
        best = k;
        slot = at;
      }
    }
    if (together == 1) lost = again;
    else todo = again;
  }
  if (!act) return;
  if ((lost >> lane) & 1u) {
    ovf[2 + atomicAdd(&ovf[0], 1u)] = t;
    return;
  }
  const uint32_t qi = __float_as_uint(qv.w);
  const bool found = best != none;
  const float d = found ? __uint_as_float((uint32_t)(best >> 32)) : INFINITY;
  nn[qi] = found ? (int32_t)(uint32_t)best : -1;
  d2[qi] = d;
  qs.nnS[t] = found ? slot : kNoSlot;
  qs.d2S[t] = d;
}

__global__ __launch_bounds__(64) void k_bquery_deep(Side qs, Side ts, int32_t *nn, float *d2, uint32_t *ovf) {
  const uint32_t n = ovf[0];
  for (uint32_t i = blockIdx.x * 64 + threadIdx.x; i < n; i += gridDim.x * 64) {
    const uint32_t t = ovf[2 + i];
    const float4 qv = qs.spts[t];
    const uint32_t qi = __float_as_uint(qv.w);
    const uint32_t cloud = (uint32_t)(qs.keys[t] >> kCloudShift);
    const float3 q = make_float3(qv.x, qv.y, qv.z);
    int32_t best;
    uint32_t bestSlot;
    float bestD;
    if (!fcp_forest<1024>(ts, ts.rootOf[cloud], q, best, bestSlot, bestD)) {
      // deeper than the deep stack (a cloud's Morton tree is at most 46
      // levels deep, so this does not happen): marked incomplete
      atomicAdd(&ovf[1], 1u);
      best = -2;
      bestSlot = kNoSlot;
      bestD = INFINITY;
    }
    nn[qi] = best;
    d2[qi] = bestD;
    qs.nnS[t] = bestSlot;
    qs.d2S[t] = bestD;
  }
}

// adjoint of loss[c] = mean over the query cloud of d(q, nearest).  A
// workgroup takes kBackChunk queries, and the neighbours' terms are summed by
// sorted slot: both sides run in Morton order, so nearly all neighbours of a
// chunk lie within a window of kBackWindow slots around its middle query's,
// which is held in LDS and added to accT (by sorted slot too) once per chunk,
// with whole lines of adds that follow each other; the rest is added straight
// away, three lanes to a point.  ownQ, if given, receives a query's own term
// at its slot; gradQ, given once all terms of a side are there, own term +
// accQ at its input index, three lanes to a point.  Scattered memory requests
// and atomics, which are done in memory and not in an XCD's L2, bound the
// kernel.  2 x 38M points: 7.7 ms with both kinds of terms added at the input
// indices and the loss by one atomic per wave, 4.6 ms with three lanes to a
// point and an XCD at neighbouring chunks, 2.9 ms as here.
// (512 threads, 2048 queries and 2560 slots, four workgroups to a CU, against
// 256/1024/2048 to 1024/8192/10240: within 2% of each other.  64/64/320 keep
// small batches less idle, 1 pair of 3000 points 253 us a run against 272 and of
// 20000 391 against 404, and cost large ones, 200 pairs of 5000 979 against 860.)
constexpr int kBackBlock = 512;
constexpr uint32_t kBackChunk = 2048, kBackWindow = 2560;
__global__ __launch_bounds__(kBackBlock) void k_bback(Side qs, Side ts, float *loss, float *ownQ, float *gradQ,
                                                      const float *accQ, float *accT) {
  __shared__ uint32_t sAt[kBackBlock];
  __shared__ float sTerm[3 * kBackBlock];
  __shared__ float sAcc[3 * kBackWindow];
  __shared__ float sLoss[kBackBlock / kWave];
  const uint32_t first = xcd_chunk(blockIdx.x, gridDim.x) * kBackChunk;
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  const uint32_t last = min(first + kBackChunk, qs.n);
  // (first < qs.n: the grid has a block per started chunk)
  const uint32_t cloud0 = (uint32_t)(qs.keys[first] >> kCloudShift);
  const uint32_t mid = qs.nnS[first + (last - first) / 2];
  const uint32_t base = mid == kNoSlot || mid < kBackWindow / 2 ? 0 : mid - kBackWindow / 2;
  if (accT) {
    for (uint32_t i = threadIdx.x; i < 3 * kBackWindow; i += kBackBlock) sAcc[i] = 0.f;
    __syncthreads();
  }
  uint32_t *const wAt = sAt + wave * kWave;
  float *const wTerm = sTerm + 3 * wave * kWave;
  float sum = 0.f;
  for (uint32_t tw = first + wave * kWave; tw < last; tw += kBackBlock) {
    const uint32_t t = tw + lane;
    const bool act = t < last;
    uint32_t qi = 0, cloud = cloud0, p = kNoSlot;
    float contrib = 0.f, gx = 0.f, gy = 0.f, gz = 0.f;
    if (act) {
      const float4 qv = qs.spts[t];
      qi = __float_as_uint(qv.w);
      cloud = (uint32_t)(qs.keys[t] >> kCloudShift);
      p = qs.nnS[t];
      if (p != kNoSlot) {
        const float4 pv = ts.spts[p];
        const float d = sqrtf(qs.d2S[t]);
        const float g = 1.f / (float)(qs.off[cloud + 1] - qs.off[cloud]);
        contrib = g * d;
        if (d > 0.f) {
          const float s = g / d;
          gx = s * (qv.x - pv.x);
          gy = s * (qv.y - pv.y);
          gz = s * (qv.z - pv.z);
        }
      }
    }
    if (ownQ || gradQ) {
      // (a wave's own part of the arrays: no barrier is needed)
      wAt[lane] = qi;
      wTerm[3 * lane] = gx;
      wTerm[3 * lane + 1] = gy;
      wTerm[3 * lane + 2] = gz;
      sync_wave_lds();
      const uint32_t n = 3 * min(last - tw, (uint32_t)kWave);
#pragma unroll
      for (uint32_t i = 0; i < 3; i++) {
        const uint32_t c = i * kWave + lane;
        if (c < n) {
          const size_t at = 3 * (size_t)tw + c;
          if (ownQ) ownQ[at] = wTerm[c];
          if (gradQ) gradQ[3 * (size_t)wAt[c / 3] + c % 3] = wTerm[c] + accQ[at];
        }
      }
      sync_wave_lds();
    }
    if (accT) {
      const bool add = gx != 0.f || gy != 0.f || gz != 0.f;
      const uint32_t w = p - base;  // (wraps below the window)
      if (add && w < kBackWindow) {
        atomicAdd(&sAcc[3 * w], -gx);
        atomicAdd(&sAcc[3 * w + 1], -gy);
        atomicAdd(&sAcc[3 * w + 2], -gz);
      }
      const bool out = add && w >= kBackWindow;
      const uint64_t m = __ballot(out);
      if (out) {
        const uint32_t j = mbcnt(m);
        wAt[j] = p;
        wTerm[3 * j] = -gx;
        wTerm[3 * j + 1] = -gy;
        wTerm[3 * j + 2] = -gz;
      }
      sync_wave_lds();
      const uint32_t n = 3 * (uint32_t)__popcll(m);
      for (uint32_t c = lane; c < n; c += kWave) atomicAdd(&accT[3 * (size_t)wAt[c / 3] + c % 3], wTerm[c]);
      sync_wave_lds();
    }
    if (loss) {
      // the chunk's first cloud is summed up to its end, any other one by
      // waves that lie in it or by single queries
      const bool other = act && cloud != cloud0;
      if (!other) sum += contrib;
      const uint32_t c0 = (uint32_t)__builtin_amdgcn_readfirstlane(cloud);
      if (__all(!act || (other && cloud == c0))) {
        float v = contrib;
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
        if (lane == 0) atomicAdd(&loss[c0], v);
      } else if (other && contrib != 0.f) {
        atomicAdd(&loss[cloud], contrib);
      }
    }
  }
  if (loss) {
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
    if (lane == 0) sLoss[wave] = sum;
  }
  __syncthreads();
  if (loss && threadIdx.x == 0) {
    float v = 0.f;
    for (int w = 0; w < kBackBlock / kWave; w++) v += sLoss[w];
    atomicAdd(&loss[cloud0], v);
  }
  if (accT)
    for (uint32_t i = threadIdx.x; i < 3 * kBackWindow; i += kBackBlock) {
      const float v = sAcc[i];
      if (v != 0.f) atomicAdd(&accT[3 * (size_t)base + i], v);
    }
}

// the sums by sorted slot to their input indices, three lanes to a point
__global__ __launch_bounds__(256) void k_bscatter(Side qs, const float *accQ, float *gradQ) {
  const uint32_t t0 = (xcd_chunk(blockIdx.x, gridDim.x) * 256 + threadIdx.x) / kWave * kWave;
  if (t0 >= qs.n) return;
  const uint32_t lane = lane_id();
  const uint32_t qi = t0 + lane < qs.n ? qs.ids[t0 + lane] : 0;
  const uint32_t n = 3 * min(qs.n - t0, (uint32_t)kWave);
#pragma unroll
  for (uint32_t i = 0; i < 3; i++) {
    const uint32_t c = i * kWave + lane;
    const uint32_t at = (uint32_t)__shfl((int)qi, c / 3, kWave);
    if (c < n) gradQ[3 * (size_t)at + c % 3] = accQ[3 * (size_t)t0 + c];
  }
}

__global__ void k_fill_f32(float *p, float v, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ----------------------------------------------------------- workspace
struct Layout {
  size_t bytes = 0;
  size_t take(size_t b) {
    size_t o = bytes;
    bytes += (b + 255) & ~size_t(255);
    return o;
  }
};

struct Plan {
  size_t keys[2], ids[2], spts[2], nnS[2], d2S[2], nodes[2], roots[2], ctr[2];
  size_t keysB, valsB, acc, open, units, sortWs, ovf;
  size_t total;
};

Plan make_plan(uint32_t numClouds, uint32_t nSrc, uint32_t nTgt) {
  Layout L;
  Plan p{};
  const uint32_t nMax = std::max(std::max(nSrc, nTgt), 1u);
  const uint32_t ns[2] = {nSrc, nTgt};
  for (int s = 0; s < 2; s++) {
    const size_t n = std::max(ns[s], 1u);
    p.keys[s] = L.take(8 * n);
    p.ids[s] = L.take(4 * n);
    p.spts[s] = L.take(16 * n);
    p.nnS[s] = L.take(4 * n);
    p.d2S[s] = L.take(4 * n);
    p.nodes[s] = L.take(32 * (2 * n + 2));
    p.roots[s] = L.take(4 * (size_t)std::max(numClouds, 1u));
    p.ctr[s] = L.take(4 * C_WORDS);
  }
  // (the backward keeps 12 bytes a point of one side in keysB and valsB, and
  // of the other in acc)
  p.keysB = L.take(8 * (size_t)nMax);
  p.valsB = L.take(4 * (size_t)nMax);
  p.acc = L.take(12 * (size_t)nMax);
  const size_t maxOpen = (size_t)kTopLevels * (nMax / kUnit);
  p.open = L.take(16 * std::max<size_t>(maxOpen, 1));
  p.units = L.take(16 * (2 * ((size_t)nMax / kBin + 1) + 2 * maxOpen));
  int cloudBits = 0;
  while ((1u << cloudBits) < std::max(numClouds, 1u)) cloudBits++;
  p.sortWs = L.take(radix_sort_ws_bytes(nMax, kCloudShift + cloudBits));
  p.ovf = L.take(4 * ((size_t)nMax + 2));
  p.total = L.bytes;
  return p;
}

int cloud_bits(uint32_t numClouds) {
  int b = 0;
  while ((1u << b) < std::max(numClouds, 1u)) b++;
  return b;
}

struct Args {
  const float *src;
  const uint32_t *srcOff;
  uint32_t nSrc;
  const float *tgt;
  const uint32_t *tgtOff;
  uint32_t nTgt;
  uint32_t numClouds;
  cubql_batch_params prm;
  char *ws;
  int32_t *srcNN, *tgtNN;
  float *srcD2, *tgtD2, *loss, *gradSrc, *gradTgt;
};

int build_side(Side &sd, Temp &tp, const Args &a, const Plan &pl, hipStream_t s, int numCU) {
  const int cbits = cloud_bits(a.numClouds);
  CUBQL_CHECK(fill_u32(sd.ctr, 0u, C_WORDS, s));
  CUBQL_CHECK(fill_u32(&sd.ctr[C_N], sd.n, 1, s));
  if (a.numClouds) k_bkeys<<<a.numClouds, 256, 0, s>>>(sd, a.numClouds);
  uint64_t *kr = nullptr;
  uint32_t *vr = nullptr;
  CUBQL_CHECK(radix_sort_pairs_ws_u64(sd.keys, sd.ids, tp.keysB, tp.valsB, &sd.ctr[C_N], std::max(sd.n, 1u),
                                      kCloudShift + cbits, s, tp.sortWs, &kr, &vr));
  if (kr != sd.keys) {
    CUBQL_HIP(hipMemcpyAsync(sd.keys, kr, 8 * (size_t)sd.n, hipMemcpyDeviceToDevice, s));
    CUBQL_HIP(hipMemcpyAsync(sd.ids, vr, 4 * (size_t)sd.n, hipMemcpyDeviceToDevice, s));
  }
  if (sd.n) k_bgather<<<div_up(sd.n, 256), 256, 0, s>>>(sd);
  const uint32_t T = (uint32_t)std::max(1, std::min(a.prm.leafSize, 65535)), most = std::max(kUnit, T);
  const uint32_t bins = div_up(sd.n, kBin), work = std::max(std::max(bins, a.numClouds), 1u);
  k_bunits<<<std::min(div_up(work, 256), (uint32_t)numCU * 4), 256, 0, s>>>(sd, tp, a.numClouds, most);
  if (sd.n > most) k_btop<<<1, 1024, 0, s>>>(sd, tp, most);
  if (sd.n) k_bunit<<<std::min(2 * bins, 2 * (uint32_t)numCU), kUnitBlock, 0, s>>>(sd, tp, T);
  if (sd.n > most) k_btop_fit<<<1, 1024, 0, s>>>(sd, tp);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

template <int BLOCK>
void launch_query(const Side &q, const Side &t, int32_t *nn, float *d2, uint32_t *ovf, hipStream_t s) {
  const uint32_t qpw = queries_per_wave(q.n);
  k_bquery<BLOCK><<<div_up(div_up(q.n, qpw), BLOCK / kWave), BLOCK, 0, s>>>(q, t, qpw, nn, d2, ovf);
}

int query_dir(const Side &q, const Side &t, int32_t *nn, float *d2, uint32_t *ovf, const cubql_batch_params &p,
              hipStream_t s) {
  if (q.n == 0) return CUBQL_OK;
  CUBQL_CHECK(fill_u32(ovf, 0u, 2, s));
  // (stackDepth picks nothing any more: a wave's queue has taken the place
  // of the lanes' stacks)
  if (p.blockSize == 64) launch_query<64>(q, t, nn, d2, ovf, s);
  else if (p.blockSize == 128) launch_query<128>(q, t, nn, d2, ovf, s);
  else launch_query<256>(q, t, nn, d2, ovf, s);
  k_bquery_deep<<<64, 64, 0, s>>>(q, t, nn, d2, ovf);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

int run(const Args &a, hipStream_t s) {
  const Plan pl = make_plan(a.numClouds, a.nSrc, a.nTgt);
  int dev = 0, numCU = 256;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&numCU, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    numCU = 256;
  Side side[2];
  const float *pts[2] = {a.src, a.tgt};
  const uint32_t *offs[2] = {a.srcOff, a.tgtOff};
  const uint32_t ns[2] = {a.nSrc, a.nTgt};
  for (int i = 0; i < 2; i++) {
    side[i].pts = pts[i];
    side[i].off = offs[i];
    side[i].n = ns[i];
    side[i].keys = (uint64_t *)(a.ws + pl.keys[i]);
    side[i].ids = (uint32_t *)(a.ws + pl.ids[i]);
    side[i].spts = (float4 *)(a.ws + pl.spts[i]);
    side[i].nnS = (uint32_t *)(a.ws + pl.nnS[i]);
    side[i].d2S = (float *)(a.ws + pl.d2S[i]);
    side[i].nodes = (Node *)(a.ws + pl.nodes[i]);
    side[i].rootOf = (uint32_t *)(a.ws + pl.roots[i]);
    side[i].ctr = (uint32_t *)(a.ws + pl.ctr[i]);
  }
  Temp tp;
  tp.keysB = (uint64_t *)(a.ws + pl.keysB);
  tp.valsB = (uint32_t *)(a.ws + pl.valsB);
  tp.acc = (float *)(a.ws + pl.acc);
  tp.open = (uint4 *)(a.ws + pl.open);
  tp.units = (uint4 *)(a.ws + pl.units);
  tp.sortWs = a.ws + pl.sortWs;
  tp.ovf = (uint32_t *)(a.ws + pl.ovf);

  int ps = prof_begin(s);
  CUBQL_CHECK(build_side(side[0], tp, a, pl, s, numCU));
  CUBQL_CHECK(build_side(side[1], tp, a, pl, s, numCU));
  prof_end(ps, s, "batch_build");
  prof_set(ps, (12.0 + 12.0 + 8.0 * 2 * 6 + 8.0 + 24.0 + 32.0) * (a.nSrc + a.nTgt), a.nSrc + a.nTgt);
  const uint32_t fg = 1024;
  if (a.loss) k_fill_f32<<<std::max(1u, std::min(div_up(a.numClouds, 256), fg)), 256, 0, s>>>(a.loss, 0.f, a.numClouds);
  ps = prof_begin(s);
  CUBQL_CHECK(query_dir(side[0], side[1], a.srcNN, a.srcD2, tp.ovf, a.prm, s));
  CUBQL_CHECK(query_dir(side[1], side[0], a.tgtNN, a.tgtD2, tp.ovf, a.prm, s));
  prof_end(ps, s, "batch_query");
  prof_set(ps, 20.0 * (a.nSrc + a.nTgt), a.nSrc + a.nTgt);
  ps = prof_begin(s);
  // the sides' sums by sorted slot
  float *accSrc = a.gradSrc ? tp.acc : nullptr, *accTgt = a.gradTgt ? (float *)tp.keysB : nullptr;
  if (accTgt) k_fill_f32<<<fg, 256, 0, s>>>(accTgt, 0.f, 3 * (size_t)a.nTgt);
  if (a.nSrc && (a.loss || accSrc || accTgt))
    k_bback<<<div_up(a.nSrc, kBackChunk), kBackBlock, 0, s>>>(side[0], side[1], a.loss, accSrc, nullptr, nullptr,
                                                              accTgt);
  if (a.nTgt && (a.loss || accSrc || accTgt))
    k_bback<<<div_up(a.nTgt, kBackChunk), kBackBlock, 0, s>>>(side[1], side[0], a.loss, nullptr, a.gradTgt, accTgt,
                                                              accSrc);
  if (a.nSrc && accSrc) k_bscatter<<<div_up(a.nSrc, 256), 256, 0, s>>>(side[0], accSrc, a.gradSrc);
  prof_end(ps, s, "batch_backward");
  prof_set(ps, 68.0 * (a.nSrc + a.nTgt), a.nSrc + a.nTgt);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

int check_args(const Args &a, size_t wsBytes) {
  if (a.numClouds == 0) return CUBQL_OK;
  if (!a.src || !a.srcOff || !a.tgt || !a.tgtOff || !a.ws || !a.srcNN || !a.tgtNN || !a.srcD2 || !a.tgtD2) {
    set_error("cubql_batch_chamfer_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  const Plan pl = make_plan(a.numClouds, a.nSrc, a.nTgt);
  if (wsBytes < pl.total) {
    set_error("cubql_batch_chamfer_f3: workspace of %zu bytes is below the %zu needed", wsBytes, pl.total);
    return CUBQL_ERR_INVALID_ARG;
  }
  const int b = a.prm.blockSize;
  if (!(b == 64 || b == 128 || b == 256) || !(a.prm.stackDepth == 8 || a.prm.stackDepth == 16 || a.prm.stackDepth == 32 || a.prm.stackDepth == 64) ||
      a.prm.leafSize < 1) {
    set_error("cubql_batch_chamfer_f3: params must have blockSize 64/128/256, stackDepth 8/16/32/64, leafSize >= 1");
    return CUBQL_ERR_INVALID_ARG;
  }
  return CUBQL_OK;
}

}  // namespace bt
}  // namespace cubql

using namespace cubql;

struct cubql_graph_s {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

extern "C" size_t cubql_batch_chamfer_workspace_f3(uint32_t numClouds, uint32_t numSrc, uint32_t numTgt) {
  return bt::make_plan(numClouds, numSrc, numTgt).total;
}

static bt::Args make_args(const float *src, const uint32_t *srcOff, uint32_t nSrc, const float *tgt,
                          const uint32_t *tgtOff, uint32_t nTgt, uint32_t numClouds,
                          const cubql_batch_params *prm, void *ws, int32_t *srcNN, float *srcD2,
                          int32_t *tgtNN, float *tgtD2, float *loss, float *gradSrc, float *gradTgt) {
  bt::Args a{};
  a.src = src; a.srcOff = srcOff; a.nSrc = nSrc;
  a.tgt = tgt; a.tgtOff = tgtOff; a.nTgt = nTgt;
  a.numClouds = numClouds;
  if (prm) a.prm = *prm;
  else a.prm = cubql_batch_params{8, 256, 64, 0};
  a.ws = (char *)ws;
  a.srcNN = srcNN; a.srcD2 = srcD2; a.tgtNN = tgtNN; a.tgtD2 = tgtD2;
  a.loss = loss; a.gradSrc = gradSrc; a.gradTgt = gradTgt;
  return a;
}

extern "C" int cubql_batch_chamfer_f3(const float *d_src, const uint32_t *d_srcOffsets, uint32_t numSrc,
                                      const float *d_tgt, const uint32_t *d_tgtOffsets, uint32_t numTgt,
                                      uint32_t numClouds, const cubql_batch_params *params, void *d_workspace,
                                      size_t workspaceBytes, int32_t *d_srcNN, float *d_srcSqrDist,
                                      int32_t *d_tgtNN, float *d_tgtSqrDist, float *d_loss,
                                      float *d_gradSrc, float *d_gradTgt, cubql_stream_t s) {
  clear_error();
  bt::Args a = make_args(d_src, d_srcOffsets, numSrc, d_tgt, d_tgtOffsets, numTgt, numClouds, params,
                         d_workspace, d_srcNN, d_srcSqrDist, d_tgtNN, d_tgtSqrDist, d_loss, d_gradSrc, d_gradTgt);
  CUBQL_CHECK(bt::check_args(a, workspaceBytes));
  if (numClouds == 0) return CUBQL_OK;
  return bt::run(a, (hipStream_t)s);
}

extern "C" int cubql_batch_chamfer_graph_f3(const float *d_src, const uint32_t *d_srcOffsets, uint32_t numSrc,
                                            const float *d_tgt, const uint32_t *d_tgtOffsets, uint32_t numTgt,
                                            uint32_t numClouds, const cubql_batch_params *params,
                                            void *d_workspace, size_t workspaceBytes, int32_t *d_srcNN,
                                            float *d_srcSqrDist, int32_t *d_tgtNN, float *d_tgtSqrDist,
                                            float *d_loss, float *d_gradSrc, float *d_gradTgt,
                                            cubql_graph *out) {
  clear_error();
  if (!out) {
    set_error("cubql_batch_chamfer_graph_f3: out is NULL");
    return CUBQL_ERR_INVALID_ARG;
  }
  *out = nullptr;
  bt::Args a = make_args(d_src, d_srcOffsets, numSrc, d_tgt, d_tgtOffsets, numTgt, numClouds, params,
                         d_workspace, d_srcNN, d_srcSqrDist, d_tgtNN, d_tgtSqrDist, d_loss, d_gradSrc, d_gradTgt);
  CUBQL_CHECK(bt::check_args(a, workspaceBytes));
  if (numClouds == 0) {
    set_error("cubql_batch_chamfer_graph_f3: empty batch");
    return CUBQL_ERR_INVALID_ARG;
  }
  hipStream_t cs;
  CUBQL_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
  cubql_graph g = new cubql_graph_s();
  const bool profWas = prof_on();
  if (profWas) cubql_profile_enable(0);
  hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
  int st = e == hipSuccess ? bt::run(a, cs) : CUBQL_ERR_HIP;
  hipError_t e2 = hipStreamEndCapture(cs, &g->graph);
  if (profWas) cubql_profile_enable(1);
  if (st == CUBQL_OK && (e != hipSuccess || e2 != hipSuccess)) {
    set_error("graph capture failed: %s", hipGetErrorString(e != hipSuccess ? e : e2));
    st = CUBQL_ERR_HIP;
  }
  if (st == CUBQL_OK) {
    e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
      set_error("hipGraphInstantiate failed: %s", hipGetErrorString(e));
      st = CUBQL_ERR_HIP;
    }
  }
  (void)hipStreamDestroy(cs);
  if (st != CUBQL_OK) {
    if (g->graph) (void)hipGraphDestroy(g->graph);
    delete g;
    return st;
  }
  *out = g;
  return CUBQL_OK;
}

extern "C" int cubql_graph_launch(cubql_graph g, cubql_stream_t s) {
  clear_error();
  if (!g || !g->exec) {
    set_error("cubql_graph_launch: invalid graph");
    return CUBQL_ERR_INVALID_ARG;
  }
  CUBQL_HIP(hipGraphLaunch(g->exec, (hipStream_t)s));
  return CUBQL_OK;
}

extern "C" int cubql_graph_destroy(cubql_graph g) {
  if (!g) return CUBQL_OK;
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  delete g;
  return CUBQL_OK;
}
