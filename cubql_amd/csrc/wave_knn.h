// wave_knn.h -- k-nearest-neighbour queries whose traversal is shared by a
// wave (see wave_closest.h for the queue of subtrees).
//
// A query's list of its K nearest keys (squared distance bits << 32 | id) is
// in its own lane's registers.  Whichever lane visits a leaf for a query puts
// the prims nearer than the query's k-th key into the query's buffer in LDS;
// when a buffer is full, every lane takes its own query's buffer into its
// list.  So the insertion network, which costs as much for one lane as for
// 64, runs with most lanes on (one query per lane: a fifth of them).
//
// Before the traversal a query descends to its nearest leaf and, until it has
// k prims, to the nearest leaves beside it.  The k-th of those keys bounds the
// traversal, which then collects the list from nothing: every prim at or
// under the bound is met exactly once.  (Without a bound every subtree is queued:
// 200K clustered queries, 16 neighbours, leaves of one prim 30.2 ms where nine
// leaves were too few, 0.74 ms so.)
#pragma once
#include "common.h"
#include "uniform_load.h"
#include "wave_closest.h"

namespace cubql {

// Keys a query's buffer holds (12 and 16 leave fewer waves in flight and are
// 5 to 40% slower, 4 and 6 are up to 3%).
constexpr int kKnnBuf = 8;

// Far siblings of a query's last descents that may seed it, as many as it wants
// prims.  (In LDS: a ring of registers is shifted at each step, 2M clustered
// queries with 16 neighbours 3.29 ms so and 3.15 here.)
constexpr uint32_t kKnnSibs = 16;
static_assert(kKnnSibs * sizeof(uint32_t) <= kKnnBuf * sizeof(unsigned long long), "the ring lies in the buffer");

// The queue holds what still leaves four workgroups a CU with up to 8
// neighbours (320 slots: 6% slower) and three, as many as the registers allow,
// with 16: a wave that has filled its queue expands few lanes at a time (2M
// clustered queries, 16 neighbours: a step of 11.2 ms with 320 slots, 8.0 with
// 768).
template <int K>
struct WaveKnn {
  static constexpr int kCap = K <= 8 ? 448 : 768;
  uint2 task[kCap];
  unsigned long long kth[kWave];   // keys below it are wanted
  union {
    unsigned long long buf[kKnnBuf][kWave];
    uint32_t sib[kKnnSibs][kWave];  // (before the traversal) siblings, a ring
  };
  float q[3][kWave];
  uint32_t count[kWave];           // keys put into the buffer (may pass kKnnBuf)
  uint32_t failed[2];              // queries that lost a task to a full queue
  uint16_t cnt[kCap];
};

// (sorted ascending) keeps the K smallest of list and key
template <int K>
__device__ __forceinline__ void knn_insert(unsigned long long (&list)[K], unsigned long long key) {
#pragma unroll
  for (int j = 0; j < K; j++) {
    const bool less = key < list[j];
    const unsigned long long t = list[j];
    list[j] = less ? key : t;
    key = less ? t : key;
  }
}
// list[k - 1] for k in [1, K]
template <int K>
__device__ __forceinline__ unsigned long long knn_kth(const unsigned long long (&list)[K], int k) {
  unsigned long long v = 0ull;
#pragma unroll
  for (int j = 0; j < K; j++) v |= (j == k - 1 ? ~0ull : 0ull) & list[j];
  return v;
}

// (16 lanes: 4% slower, 48: 1%)
constexpr int kKnnLeafLanes = 32;

// All 64 lanes of the wave call this; lanes with `live` hold a query of the
// tree `nodes`, whose root is node 0.  point(slot) is the prim at a primID
// slot (x, y, z, id bits).  list receives the lane's K smallest keys below
// `none`, ~0 where there are fewer (the first k of them are exact).
template <int K, typename PointFn>
__device__ __forceinline__ void wave_knn(WaveKnn<K> &sh, const cubql_node3f *nodes, bool live, float x, float y, float z,
                                         int k, unsigned long long none, PointFn &&point,
                                         unsigned long long (&list)[K], bool *failed) {
  using namespace cubql_dev;
  constexpr uint32_t CAP = WaveKnn<K>::kCap;
  const uint32_t lane = lane_id();
  const uint64_t rootWord = nodes[0].offsetAndCountBits;
#pragma unroll
  for (int j = 0; j < K; j++) list[j] = ~0ull;
  // (1) bound: the k-th key of the nearest leaf and its neighbours
  unsigned long long limit = none;
  if (live) {
    uint32_t top = 0, nsib = 0;
    int found = 0, left = k;
    bool beyond = false;
    uint32_t off = oc_off(rootWord), cnt = oc_cnt(rootWord);
    auto step = [&](const QNode &n0, const QNode &n1, bool keep) {
      const bool near0 = sqr_dist_box(x, y, z, n0) < sqr_dist_box(x, y, z, n1);
      const uint64_t oc = near0 ? node_oc(n0) : node_oc(n1);
      if (keep) {
        sh.sib[top++ % kKnnSibs][lane] = near0 ? off + 1 : off;
        nsib = min(nsib + 1, kKnnSibs);
      }
      off = oc_off(oc);
      cnt = oc_cnt(oc);
    };
    while (cnt == 0) {
      const uint32_t u = (uint32_t)__builtin_amdgcn_readfirstlane((int)off);
      if (__ballot(off == u) != __ballot(true)) break;
      QNode n0, n1;
      load_pair_uniform(nodes, u, n0, n1);
      step(n0, n1, true);
    }
    while (cnt == 0) {
      const QNode n0 = load_node(nodes, off), n1 = load_node(nodes, off + 1);
      step(n0, n1, true);
    }
    const float far = __uint_as_float((uint32_t)(none >> 32));
    // With few prims to a leaf the nearest subtrees are taken whole: the nearest
    // leaves of many siblings lie far apart and bound little (uniform points, leaves
    // of one, 200K queries, 16 neighbours: 4.50 ms by nearest leaves, 0.65 so).
    const bool whole = 4 * cnt < (uint32_t)k;
    while (true) {
      for (uint32_t j = 0; j < cnt; j++) {
        const float4 p = point(off + j);
        const unsigned long long key =
            closest_key(sqr_dist_pt(p.x, p.y, p.z, x, y, z), __float_as_uint(p.w));
        if (key < none) {
          found++;
          if (key < list[K - 1]) knn_insert<K>(list, key);
        } else {
          beyond = true;
        }
      }
      // the nearest leaf under the deepest unused sibling that is within the radius;
      // k leaves hold k prims, and a radius that leaves out prims of these leaves
      // bounds as well (200K queries, about 6 of 16 neighbours within it, leaves of
      // one: 0.50 ms seeding on, 0.36 so)
      if (found >= k || beyond || --left == 0) break;
      bool near = false;
      while (nsib && !near) {
        const QNode n = load_node(nodes, sh.sib[--top % kKnnSibs][lane]);
        nsib--;
        near = sqr_dist_box(x, y, z, n) <= far;
        off = oc_off(node_oc(n));
        cnt = oc_cnt(node_oc(n));
      }
      if (!near) break;
      while (cnt == 0) {
        const QNode n0 = load_node(nodes, off), n1 = load_node(nodes, off + 1);
        step(n0, n1, whole);
      }
    }
    const unsigned long long kth = knn_kth<K>(list, k);
    if (kth != ~0ull) limit = kth + 1;  // (a key's id is below 2^32 - 1)
  }
#pragma unroll
  for (int j = 0; j < K; j++) list[j] = ~0ull;
  sh.kth[lane] = limit;
  sh.count[lane] = 0u;
  sh.q[0][lane] = x;
  sh.q[1][lane] = y;
  sh.q[2][lane] = z;
  if (lane < 2) sh.failed[lane] = 0u;
  sync_wave_lds();
  // (2) the traversal: the path again, then the queued subtrees
  enum : uint32_t { kFree, kInner, kLeaf };
  float cull = __uint_as_float((uint32_t)(limit >> 32));
  uint32_t off = oc_off(rootWord), cnt = oc_cnt(rootWord), q = lane, steps = 0;
  uint32_t state = !live ? kFree : cnt ? kLeaf : kInner;
  uint32_t qn = 0;
  auto expand = [&](const QNode &n0, const QNode &n1, bool on, bool &push, uint2 &t, uint32_t &c) {
    const float d0 = sqr_dist_box(x, y, z, n0), d1 = sqr_dist_box(x, y, z, n1);
    const bool near0 = d0 < d1;
    const uint64_t ocN = near0 ? node_oc(n0) : node_oc(n1), ocF = near0 ? node_oc(n1) : node_oc(n0);
    const float dn = fminf(d0, d1), df = fmaxf(d0, d1);
    push = on && df <= cull;
    t = make_uint2(oc_off(ocF), (__float_as_uint(df) & ~63u) | q);
    c = oc_cnt(ocF);
    if (on) {
      off = oc_off(ocN);
      cnt = oc_cnt(ocN);
      state = dn > cull ? kFree : cnt ? kLeaf : kInner;
      if (++steps > kMaxSteps && state == kInner) {
        atomicOr(&sh.failed[q >> 5], 1u << (q & 31));
        state = kFree;
      }
    }
  };
  auto enqueue = [&](bool push, uint2 t, uint32_t c) {
    const uint64_t m = __ballot(push);
    if (!m) return;
    const uint32_t slot = qn + mbcnt(m);
    if (push) {
      if (slot < CAP) {
        sh.task[slot] = t;
        sh.cnt[slot] = (uint16_t)c;
      } else {
        atomicOr(&sh.failed[q >> 5], 1u << (q & 31));
      }
    }
    qn = min(qn + (uint32_t)__popcll(m), CAP);
    sync_wave_lds();
  };
  // What is left of a query that has lost a task is dropped: it runs again, and
  // the others have its room.  (Going on with it, one lane at a time in a full
  // queue, and losing tasks of every other query: 200K queries of 100 places with
  // 1000 points each, 8 neighbours, leaves of 2: 24.0 ms, 7.0 so.)
  auto drop = [&](uint32_t lost) {
    if (q == lost) state = kFree;
    uint32_t kept = 0;
    for (uint32_t i0 = 0; i0 < qn; i0 += kWave) {
      const uint32_t i = min(i0 + lane, qn - 1);
      const uint2 t = sh.task[i];
      const uint16_t c = sh.cnt[i];
      const bool keep = i0 + lane < qn && (t.y & 63u) != lost;
      const uint64_t m = __ballot(keep);
      if (keep) {
        sh.task[kept + mbcnt(m)] = t;
        sh.cnt[kept + mbcnt(m)] = c;
      }
      kept += (uint32_t)__popcll(m);
      sync_wave_lds();
    }
    qn = kept;
  };
  // every lane takes its query's buffer into its list
  auto merge = [&]() __attribute__((always_inline)) {
    const uint32_t n = min(sh.count[lane], (uint32_t)kKnnBuf);
    for (uint32_t j = 0; j < (uint32_t)kKnnBuf && __ballot(j < n); j++) {
      const unsigned long long key = sh.buf[j][lane];
      if (j < n && key < list[K - 1]) knn_insert<K>(list, key);
    }
    const unsigned long long kth = knn_kth<K>(list, k);
    sh.kth[lane] = kth != ~0ull ? kth : limit;
    sh.count[lane] = 0u;
    sync_wave_lds();
  };
  while (true) {
    const uint64_t m = __ballot(state == kInner);
    if (!m || qn + kWave > CAP) break;
    const uint32_t u = (uint32_t)__builtin_amdgcn_readlane((int)off, __builtin_ctzll(m));
    if (__ballot(state == kInner && off == u) != m) break;
    QNode n0, n1;
    load_pair_uniform(nodes, u, n0, n1);
    bool push;
    uint2 t;
    uint32_t c;
    expand(n0, n1, state == kInner, push, t, c);
    enqueue(push, t, c);
  }
  while (true) {
    const uint64_t freeM = __ballot(state == kFree);
    if (qn && freeM) {
      // newest tasks first
      const uint32_t r = mbcnt(freeM);
      if (state == kFree && r < qn) {
        const uint2 t = sh.task[qn - 1 - r];
        const uint32_t c = sh.cnt[qn - 1 - r];
        q = t.y & 63u;
        if (__uint_as_float(t.y & ~63u) <= __uint_as_float((uint32_t)(sh.kth[q] >> 32))) {
          x = sh.q[0][q];
          y = sh.q[1][q];
          z = sh.q[2][q];
          off = t.x;
          cnt = c;
          steps = 0;
          state = c ? kLeaf : kInner;
        }
      }
      qn -= min(qn, (uint32_t)__popcll(freeM));
      sync_wave_lds();
    }
    const uint64_t inner = __ballot(state == kInner), leafM = __ballot(state == kLeaf);
    if (!(inner | leafM)) {
      if (!qn) break;
      continue;
    }
    // a nearly full queue: only as many lanes expand as it has room for
    const uint32_t room = CAP - qn;
    if (inner && (!leafM || (room && __popcll(leafM) < kKnnLeafLanes))) {
      bool on = state == kInner;
      if (room < (uint32_t)__popcll(inner)) on = on && mbcnt(inner) < max(room, 1u);
      bool push = false;
      uint2 t = make_uint2(0u, 0u);
      uint32_t c = 0;
      if (on) {
        cull = __uint_as_float((uint32_t)(sh.kth[q] >> 32));
        const QNode n0 = load_node(nodes, off), n1 = load_node(nodes, off + 1);
        expand(n0, n1, true, push, t, c);
      }
      enqueue(push, t, c);
      if (room == 0) {
        // (one lane expands)
        const uint64_t m = __ballot(push);
        if (m) drop((uint32_t)__builtin_amdgcn_readlane((int)q, __builtin_ctzll(m)));
      }
    } else {
      // up to four prims of each leaf; a lane whose query's buffer is full
      // stops at the first prim that found no place
      bool full = false;
      if (state == kLeaf) {
        unsigned long long key[4];
        float4 p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) p[u] = point(off + min((uint32_t)u, cnt - 1));
        const unsigned long long kth = sh.kth[q];
        uint32_t want = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          key[u] = closest_key(sqr_dist_pt(p[u].x, p[u].y, p[u].z, x, y, z), __float_as_uint(p[u].w));
          if ((uint32_t)u < cnt && key[u] < kth) want |= 1u << u;
        }
        uint32_t done = min(cnt, 4u);
        if (want) {
          uint32_t slot = atomicAdd(&sh.count[q], (uint32_t)__popc(want));
#pragma unroll
          for (int u = 0; u < 4; u++) {
            if (want >> u & 1u) {
              if (slot < (uint32_t)kKnnBuf) {
                sh.buf[slot][q] = key[u];
              } else if (!full) {
                full = true;
                done = u;
              }
              slot++;
            }
          }
        }
        off += done;
        cnt -= done;
        if (cnt == 0) state = kFree;
      }
      sync_wave_lds();
      if (__ballot(full) || __ballot(sh.count[lane] >= (uint32_t)kKnnBuf)) merge();
    }
  }
  merge();
  *failed = (sh.failed[lane >> 5] >> (lane & 31)) & 1u;
}

}  // namespace cubql
