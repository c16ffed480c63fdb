// query_order.h -- spatial ordering of a batch of queries.
//
// Lanes of a wave whose queries are close to each other walk nearly the same
// nodes, so a large batch is sorted by place before it is traversed, which
// makes node loads coherent and cuts divergence.  Results are written back to
// each query's own slot, so the output is independent of the order.
//
// The place is the Morton code of the query in cells of the tree's root box,
// or, where a few far-off prims leave most queries in a few cells, the primID
// slot of the leaf the query descends to (binary trees).  A sample of the
// queries decides on the device.
#pragma once
#include "common.h"

namespace cubql {

// Batches below this size run in input order.
constexpr uint32_t kQueryOrderMin = 32768;

// The places of a batch: points (stride 3 floats) or the centres of boxes
// (stride 6: lower xyz, upper xyz).
struct QueryPlaces {
  const float *p;
  uint32_t n;
  bool boxes;
};

// Orders `q` on a caller's workspace of query_order_ws_bytes(q.n) bytes
// (256-byte aligned): *order points into it, a device permutation (sorted
// position -> query index), or is nullptr for small batches.  rootBox: the
// box the cells are taken over (device).  bvh: the tree for the slot keys, or
// nullptr.  Allocates nothing.
size_t query_order_ws_bytes(uint32_t nq);
int query_order_ws(const cubql_box3f *rootBox, const cubql_bvh3f *bvh, const QueryPlaces &q, hipStream_t s, void *ws,
                   const uint32_t **order);

}  // namespace cubql
