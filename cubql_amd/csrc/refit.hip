// refit.hip -- bottom-up refit of node boxes for any BinaryBVH topology.
//
// Replaces gpuBuilder_impl::refit (builder/cuda/sm_builder.h:616-693): leaf
// box = union of its prim boxes, inner box = union of its two children.
// One thread per node; leaves start, and each parent is finished by the
// second child to arrive.  A workgroup's span of nodes holds whole subtrees in
// the builders' numberings: those climb in LDS, and what is left at their tops
// through memory (an atomic counter per node).
//
// Bound: the latency of a leaf's climb (a store acknowledged, an atomic and
// a load per level, ~20 levels at 1M prims) and the prim boxes gathered by
// primID.  A climb hands its box to the other child's thread through
// agent-scope relaxed atomic stores and loads, which are coherent between
// the XCDs' L2s by themselves, with a wait for the stores between them and
// the arrival count; an agent-scope fence writes back and invalidates the
// whole L2 instead.  1M boxes, leaf 4: 3265 us with fences, 88 us without, 58
// us with the climb in LDS first (waves wait for memory 49% of their time and
// 43% to issue; 1.5M lines fetched, 3.4 TB/s; VALU issue 7 us).
#include "block_ops.h"
#include "build_common.h"
#include "common.h"
#include "refit.h"

namespace cubql {
namespace rf {

constexpr uint32_t kSpan = 512;  // nodes of a workgroup (256 to 1024: the same)
constexpr uint32_t kNoParent = 0xffffffffu;

// GPU builders leave node 1 unused (bvh.h:66-70); a tree whose root has its
// children at 1 and 2 (the CPU builder's numbering) uses it.
__device__ inline bool node1_used(const Node *nodes) {
  uint64_t oc = nodes[0].oc;
  return oc_count(oc) == 0 && oc_offset(oc) == 1;
}

__global__ void k_parents(const Node *nodes, uint32_t numNodes, uint32_t *parent, uint32_t *arrive) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < numNodes; i += gridDim.x * blockDim.x) {
    arrive[i] = 0;
    if (i == 0) parent[0] = kNoParent;
    if (i == 1 && !node1_used(nodes)) continue;
    uint64_t oc = nodes[i].oc;
    if (oc_count(oc) != 0) continue;
    uint32_t off = (uint32_t)oc_offset(oc);
    if (off + 1 < numNodes) {
      parent[off] = i;
      parent[off + 1] = i;
    }
  }
}

__device__ inline void load_box(const cubql_box3f *p, uint32_t i, float lo[3], float hi[3]) {
  const float2 *f = reinterpret_cast<const float2 *>(p + i);
  float2 a = f[0], b = f[1], c = f[2];
  lo[0] = a.x; lo[1] = a.y; lo[2] = b.x;
  hi[0] = b.y; hi[1] = c.x; hi[2] = c.y;
}

// Union of cnt prim boxes in list order, four ids and boxes in flight.
__device__ __forceinline__ void leaf_box(const cubql_box3f *boxes, const uint32_t *ids, uint32_t cnt, float (&lo)[3],
                                         float (&hi)[3]) {
  for (uint32_t j = 0; j < cnt; j += 4) {
    uint32_t id[4];
#pragma unroll
    for (int u = 0; u < 4; u++) id[u] = ids[min(j + u, cnt - 1)];
    float bl[4][3], bh[4][3];
#pragma unroll
    for (int u = 0; u < 4; u++) load_box(boxes, id[u], bl[u], bh[u]);
    // (a repeated last box changes no bound)
#pragma unroll
    for (int u = 0; u < 4; u++)
      for (int d = 0; d < 3; d++) {
        lo[d] = fminf(lo[d], bl[u][d]);
        hi[d] = fmaxf(hi[d], bh[u][d]);
      }
  }
}

// The box of `node` stored, and those of the nodes above it for as long as this
// thread is the second to arrive.
__device__ __forceinline__ void climb(Node *nodes, const uint32_t *parent, uint32_t *arrive, uint32_t node,
                                      float (&lo)[3], float (&hi)[3]) {
  while (true) {
    store_box_agent(&nodes[node], lo, hi);
    const uint32_t p = parent[node];
    if (p == kNoParent) break;
    const uint32_t left = (uint32_t)oc_offset(nodes[p].oc);
    // this node's box has reached the coherence point before its arrival counts
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (__hip_atomic_fetch_add(&arrive[p], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
      break;  // the sibling finishes the parent
    asm volatile("" ::: "memory");
    // the sibling's box, combined in child order
    const bool isLeft = node == left;
    float sl[3], sh[3];
    load_box_agent(&nodes[isLeft ? left + 1 : left], sl, sh);
    for (int d = 0; d < 3; d++) {
      lo[d] = isLeft ? fminf(lo[d], sl[d]) : fminf(sl[d], lo[d]);
      hi[d] = isLeft ? fmaxf(hi[d], sh[d]) : fmaxf(sh[d], hi[d]);
    }
    node = p;
  }
}

__global__ __launch_bounds__(kSpan) void k_refit(Node *nodes, uint32_t numNodes, const uint32_t *primIDs,
                                                 const cubql_box3f *boxes, const uint32_t *parent,
                                                 uint32_t *arrive) {
  __shared__ float sBox[6][kSpan];
  __shared__ uint32_t sUp[kSpan], sLeft[kSpan], sSeen[kSpan];
  const uint32_t n0 = blockIdx.x * kSpan, i = threadIdx.x;
  uint32_t node = n0 + i, leaf = 0;
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  sUp[i] = kNoParent;
  sSeen[i] = 0;
  if (node < numNodes && (node != 1 || node1_used(nodes))) {
    const uint64_t oc = nodes[node].oc;
    leaf = oc_count(oc);
    sUp[i] = parent[node];
    sLeft[i] = (uint32_t)oc_offset(oc);
    if (leaf) leaf_box(boxes, primIDs + (uint32_t)oc_offset(oc), leaf, lo, hi);
  }
  __syncthreads();
  bool climbing = leaf != 0, out = false;
  while (climbing) {
    // parent and sibling in the span (the root's none is far outside)
    const uint32_t q = sUp[node - n0] - n0;
    const uint32_t left = q < kSpan ? sLeft[q] - n0 : kSpan;
    out = left >= kSpan - 1;
    if (out) break;
    const uint32_t at = node - n0, side = at == left ? 0u : 1u;
    for (int d = 0; d < 3; d++) {
      nodes[node].lo[d] = lo[d];
      nodes[node].hi[d] = hi[d];
      sBox[d][at] = lo[d];
      sBox[3 + d][at] = hi[d];
    }
    // (a wave's LDS accesses run in program order)
    asm volatile("" ::: "memory");
    climbing = ((atomicOr(&sSeen[q], 1u << side) >> (side ^ 1u)) & 1u) != 0;
    asm volatile("" ::: "memory");
    if (climbing) {
      for (int d = 0; d < 3; d++) {
        const float sl = sBox[d][left + (side ^ 1u)], sh = sBox[3 + d][left + (side ^ 1u)];
        lo[d] = side == 0 ? fminf(lo[d], sl) : fminf(sl, lo[d]);
        hi[d] = side == 0 ? fmaxf(hi[d], sh) : fmaxf(sh, hi[d]);
      }
      node = n0 + q;
    }
  }
  __syncthreads();
  if (out) climb(nodes, parent, arrive, node, lo, hi);
  // a node that one child has come to in LDS, and the other has not
  const uint32_t seen = sSeen[i];
  if (seen == 1u || seen == 2u) {
    const uint32_t child = sLeft[i] + (seen >> 1);
    for (int d = 0; d < 3; d++) {
      lo[d] = sBox[d][child - n0];
      hi[d] = sBox[3 + d][child - n0];
    }
    climb(nodes, parent, arrive, child, lo, hi);
  }
}

}  // namespace rf

int refit_tree_ws(cubql_bvh3f *bvh, const cubql_box3f *boxes, hipStream_t s, uint32_t *parent, uint32_t *arrive) {
  uint32_t g = std::min<uint32_t>(div_up(bvh->numNodes, 256), 8192);
  rf::k_parents<<<g, 256, 0, s>>>((const Node *)bvh->nodes, bvh->numNodes, parent, arrive);
  rf::k_refit<<<div_up(bvh->numNodes, rf::kSpan), rf::kSpan, 0, s>>>((Node *)bvh->nodes, bvh->numNodes, bvh->primIDs,
                                                                     boxes, parent, arrive);
  CUBQL_LAUNCH_CHECK();
  return CUBQL_OK;
}

int refit_tree(cubql_bvh3f *bvh, const cubql_box3f *boxes, hipStream_t s,
               const cubql_mem_resource *mem) {
  if (bvh->numNodes == 0) return CUBQL_OK;
  Scratch scr(mem, s);
  uint32_t *parent = nullptr, *arrive = nullptr;
  CUBQL_CHECK(scr.alloc(&parent, bvh->numNodes));
  CUBQL_CHECK(scr.alloc(&arrive, bvh->numNodes));
  return refit_tree_ws(bvh, boxes, s, parent, arrive);
}

}  // namespace cubql

extern "C" int cubql_refit_f3(cubql_bvh3f *bvh, const cubql_box3f *d_boxes, cubql_stream_t s,
                              const cubql_mem_resource *mem) {
  cubql::clear_error();
  if (!bvh || !d_boxes) {
    cubql::set_error("cubql_refit_f3: null argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  return cubql::refit_tree(bvh, d_boxes, (hipStream_t)s, mem);
}
