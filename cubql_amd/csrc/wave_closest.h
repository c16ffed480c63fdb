// wave_closest.h -- closest-prim queries whose traversal is shared by a wave.
//
// One query per lane leaves a wave64 mostly idle: after the two descents to
// the nearest leaf a query visits one or two more subtrees on average, but a
// wave waits for its slowest query (10M uniform points and queries: 123 of
// its 167 node-pair iterations were such side visits, with 4% of the lanes
// on, and the node loads of those few lanes kept the address unit busy 92%
// of the time).  Here a wave's queries keep their coordinates and best
// (distance, id) in LDS, and every subtree still to visit is a task in the
// wave's LDS queue that any free lane takes.
//
// The result does not depend on who visits what: it is the minimum of
// (squared distance bits << 32 | id) over the prims within the radius, and a
// task is dropped only if its box is farther than the query's best.
//
// Two descents come first.  (1) Every query descends along its nearer
// children (ties to the second) to one leaf and tests its prims.  (2) It
// walks the same path again with that radius and queues the far children
// still within it.  While all queries of the wave are at the same node --
// queries come in Morton order -- its pair of children is read once per wave
// through the scalar cache.
#pragma once
#include <type_traits>

#include "common.h"
#include "cubql_amd/traversal.hip.h"
#include "uniform_load.h"

namespace cubql {

// Queue slots of a wave: 512 leave fewer waves in flight (10M queries of 10M
// points: 2.21 ms a call against 2.04 ms), with 256 more queries of clustered
// and Gaussian clouds lose a task and run again.  A task is {offset, distance with the query's lane
// in its low 6 bits (rounded down: the test only gets weaker)} and the
// prim count (0: an inner node).
constexpr int kTaskCap = 320;
// steps of one descent after which a query has to run again, in the end in the
// deep kernel (the depth that kernel's stack holds)
constexpr uint32_t kMaxSteps = 1024;

struct WaveTasks {
  uint2 task[kTaskCap];
  unsigned long long best[kWave];
  float q[3][kWave];
  uint32_t failed[2];  // queries that lost a task to a full queue
  uint16_t cnt[kTaskCap];
};
// the same with a word kept beside each query's best key
struct WaveTasksAux : WaveTasks {
  uint32_t aux[kWave];
};

// Waves that a small batch is spread over: in a wave of few queries the other
// lanes take their subtrees.  Calls on a tree of 1M points, spread so and as
// waves of 64 queries (us):
//   queries          64    1000    4096   16000   64000
//   closest       38/47   40/54   42/56   48/69  90/103
//   k = 8        61/122  63/167  78/179  99/181 176/216
// (100000 Gaussian points: 38/51, 39/54, 43/55, 43/56, 89/95 and 63/133,
// 63/152, 76/158, 87/158, 153/191.)
constexpr uint32_t kWavesWanted = 4096;
// Queries of one wave: 64 once they fill the chip, fewer for small batches,
// whose time is one wave's chain of dependent loads.
inline uint32_t queries_per_wave(uint32_t nq) {
  uint32_t w = 1;
  while (w < (uint32_t)kWave && (uint64_t)w * kWavesWanted < nq) w *= 2;
  return w;
}

// Key of "nothing found within sqrMax": prims must be strictly nearer.
__device__ __forceinline__ unsigned long long closest_none(float sqrMax) {
  return (unsigned long long)(sqrMax > 0.f ? __float_as_uint(sqrMax) : 0u) << 32;
}
__device__ __forceinline__ unsigned long long closest_key(float d, uint32_t id) {
  return ((unsigned long long)__float_as_uint(d) << 32) | id;
}

// All 64 lanes of the wave call this; lanes with `live` hold a query and the
// offset/count word of its root.  leaf(off, cnt, x, y, z, aux) returns the
// least key of a leaf's prims (~0 if none) and sets aux, a word that is kept
// with the best key if Tasks is WaveTasksAux (*auxOut).  LEAF_LANES lanes at a
// leaf make the wave stop expanding nodes and test their prims.  Returns the
// lane's best key; *failed is set if the query lost a task to a full queue (or is
// deeper than kMaxSteps) and has to run again.
template <int LEAF_LANES, typename Tasks, typename LeafFn>
__device__ __forceinline__ unsigned long long wave_closest(Tasks &sh, const cubql_node3f *nodes, bool live,
                                                           uint64_t rootWord, float x, float y, float z,
                                                           unsigned long long none, LeafFn &&leaf, bool *failed,
                                                           uint32_t *auxOut = nullptr) {
  using namespace cubql_dev;
  constexpr bool kAux = std::is_same<Tasks, WaveTasksAux>::value;
  const uint32_t lane = lane_id();
  unsigned long long best = none;
  uint32_t aux = 0;
  // (1) nearest leaf
  if (live) {
    uint32_t off = oc_off(rootWord), cnt = oc_cnt(rootWord);
    while (cnt == 0) {
      const uint32_t u = (uint32_t)__builtin_amdgcn_readfirstlane((int)off);
      if (__ballot(off == u) != __ballot(true)) break;
      QNode n0, n1;
      load_pair_uniform(nodes, u, n0, n1);
      const bool near0 = sqr_dist_box(x, y, z, n0) < sqr_dist_box(x, y, z, n1);
      const uint64_t oc = near0 ? node_oc(n0) : node_oc(n1);
      off = oc_off(oc);
      cnt = oc_cnt(oc);
    }
    while (cnt == 0) {
      const QNode n0 = load_node(nodes, off), n1 = load_node(nodes, off + 1);
      const bool near0 = sqr_dist_box(x, y, z, n0) < sqr_dist_box(x, y, z, n1);
      const uint64_t oc = near0 ? node_oc(n0) : node_oc(n1);
      off = oc_off(oc);
      cnt = oc_cnt(oc);
    }
    const unsigned long long k = leaf(off, cnt, x, y, z, aux);
    best = k < best ? k : best;
  }
  sh.best[lane] = best;
  if constexpr (kAux) sh.aux[lane] = aux;
  sh.q[0][lane] = x;
  sh.q[1][lane] = y;
  sh.q[2][lane] = z;
  if (lane < 2) sh.failed[lane] = 0u;
  sync_wave_lds();
  // (2) the same path again, then the queued subtrees.  Every lane stays in
  // these loops; what a lane does follows from its state.
  enum : uint32_t { kFree, kInner, kLeaf };
  float cull = __uint_as_float((uint32_t)(best >> 32));
  uint32_t off = oc_off(rootWord), cnt = 0, q = lane, steps = 0;
  uint32_t state = live && oc_cnt(rootWord) == 0 ? kInner : kFree;
  bool main = true;  // on the path of (1), whose leaf is tested
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
      state = dn > cull ? kFree : cnt == 0 ? kInner : main ? kFree : kLeaf;
    }
  };
  auto enqueue = [&](bool push, uint2 t, uint32_t c) {
    const uint64_t m = __ballot(push);
    if (!m) return;
    const uint32_t slot = qn + mbcnt(m);
    if (push) {
      if (slot < (uint32_t)kTaskCap) {
        sh.task[slot] = t;
        sh.cnt[slot] = (uint16_t)c;
      } else {
        atomicOr(&sh.failed[q >> 5], 1u << (q & 31));
      }
    }
    qn = min(qn + (uint32_t)__popcll(m), (uint32_t)kTaskCap);
    sync_wave_lds();
  };
  // What is left of a query that has lost a task is dropped: it runs again, and
  // the others have its room.  (30 clouds of 3000 points against 3000 equal ones,
  // leaves of one: 10.3 ms going on with it, 4.5 so.)
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
  while (true) {
    const uint64_t m = __ballot(state == kInner);
    if (!m || qn + kWave > (uint32_t)kTaskCap) break;
    const uint32_t u = (uint32_t)__builtin_amdgcn_readlane((int)off, __builtin_ctzll(m));
    if (__ballot(state == kInner && off == u) != m) break;
    QNode n0, n1;
    load_pair_uniform(nodes, u, n0, n1);
    bool push;
    uint2 t;
    uint32_t c;
    expand(n0, n1, state == kInner, push, t, c);
    if (++steps > kMaxSteps && state == kInner) {
      atomicOr(&sh.failed[q >> 5], 1u << (q & 31));
      state = kFree;
    }
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
        cull = __uint_as_float((uint32_t)(sh.best[q] >> 32));
        if (__uint_as_float(t.y & ~63u) <= cull) {
          x = sh.q[0][q];
          y = sh.q[1][q];
          z = sh.q[2][q];
          off = t.x;
          cnt = c;
          steps = 0;
          main = false;
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
    const uint32_t room = (uint32_t)kTaskCap - qn;
    if (inner && (!leafM || (room && __popcll(leafM) < LEAF_LANES))) {
      bool on = state == kInner;
      if (room < (uint32_t)__popcll(inner)) on = on && mbcnt(inner) < max(room, 1u);
      bool push = false;
      uint2 t = make_uint2(0u, 0u);
      uint32_t c = 0;
      if (on) {
        const QNode n0 = load_node(nodes, off), n1 = load_node(nodes, off + 1);
        expand(n0, n1, true, push, t, c);
        if (++steps > kMaxSteps && state == kInner) {
          atomicOr(&sh.failed[q >> 5], 1u << (q & 31));
          state = kFree;
        }
      }
      enqueue(push, t, c);
      if (room == 0) {
        // (one lane expands)
        const uint64_t m = __ballot(push);
        if (m) drop((uint32_t)__builtin_amdgcn_readlane((int)q, __builtin_ctzll(m)));
      }
    } else {
      if (state == kLeaf) {
        const unsigned long long k = leaf(off, cnt, x, y, z, aux);
        atomicMin(&sh.best[q], k);
        state = kFree;
        if constexpr (kAux) {
          // (keys of one query differ: only the lane that holds the best writes)
          sync_wave_lds();
          if (sh.best[q] == k) sh.aux[q] = aux;
        }
      }
      sync_wave_lds();
    }
  }
  sync_wave_lds();
  *failed = (sh.failed[lane >> 5] >> (lane & 31)) & 1u;
  if constexpr (kAux) *auxOut = sh.aux[lane];
  return sh.best[lane];
}

}  // namespace cubql
