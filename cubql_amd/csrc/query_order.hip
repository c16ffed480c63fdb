// query_order.hip -- spatial ordering of query batches (see query_order.h).
#include "query_order.h"

#include "cubql_amd/traversal.hip.h"
#include "radix_sort.h"

namespace cubql {
namespace qo {

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  uint32_t x = v & 0x3ffu;
  x = (x | (x << 16)) & 0x030000ffu;
  x = (x | (x << 8)) & 0x0300f00fu;
  x = (x | (x << 4)) & 0x030c30c3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

// Key bits sorted by, a sort pass per eight: up to 2^20 queries 16 bits
// leave at most 16 queries in a cell on average, a quarter of a wave (1M
// kNN queries of 10M points: the same traversal time as with 24 bits, a sort
// pass less); above, 24 bits (10M queries: less than one a cell).
constexpr uint32_t kFewQueries = 1u << 20;
inline int order_bits(uint32_t nq) { return nq <= kFewQueries ? 16 : 24; }

__device__ __forceinline__ float3 place(const QueryPlaces &q, uint32_t i) {
  if (q.boxes) {
    const float *b = q.p + 6 * (size_t)i;
    return make_float3(0.5f * (b[0] + b[3]), 0.5f * (b[1] + b[4]), 0.5f * (b[2] + b[5]));
  }
  const float *p = q.p + 3 * (size_t)i;
  return make_float3(p[0], p[1], p[2]);
}

// The 30-bit Morton key of a place in the cells of the root box (places
// outside it clamp to the border cells).
__device__ __forceinline__ uint32_t morton_key(const cubql_box3f &bounds, float3 p) {
  const float ext = fmaxf(fmaxf(bounds.upper[0] - bounds.lower[0], bounds.upper[1] - bounds.lower[1]),
                          bounds.upper[2] - bounds.lower[2]);
  const float scale = 1024.f / fmaxf(ext, 1e-20f);
  const float v[3] = {p.x, p.y, p.z};
  uint32_t cell[3];
  for (int d = 0; d < 3; d++) {
    const float f = fmaxf((v[d] - bounds.lower[d]) * scale, 0.f);
    cell[d] = f < 1023.f ? (uint32_t)f : 1023u;
  }
  return spread10(cell[0]) | (spread10(cell[1]) << 1) | (spread10(cell[2]) << 2);
}

// Counts the different 24-bit Morton cells of kSample queries spread over
// the batch: crowded[0] = 1 if they are fewer than half the queries looked
// at.  A few far-off prims stretch the root box, and then Morton cells order
// nothing (2M points of 64 tight clusters with 1% of them 1e6 away: 18 of
// 1024).
constexpr uint32_t kSample = 1024;
__global__ __launch_bounds__(kSample) void k_sample(const cubql_box3f *rootBox, QueryPlaces q, uint32_t *count,
                                                    uint32_t *crowded, bool tree) {
  __shared__ uint32_t table[2 * kSample];
  __shared__ uint32_t distinct;
  const uint32_t t = threadIdx.x;
  if (t == 0) {
    *count = q.n;
    distinct = 0;
  }
  table[t] = table[t + kSample] = 0xffffffffu;
  __syncthreads();
  if (tree) {
    const uint32_t key = morton_key(*rootBox, place(q, (uint32_t)((uint64_t)t * q.n / kSample))) >> 6;
    uint32_t slot = (key * 2654435761u) >> 21;
    // (at most kSample keys in 2 kSample slots: the probe ends)
    for (uint32_t i = 0; i < 2 * kSample; i++) {
      const uint32_t old = atomicCAS(&table[slot], 0xffffffffu, key);
      if (old == 0xffffffffu) atomicAdd(&distinct, 1u);
      if (old == 0xffffffffu || old == key) break;
      slot = (slot + 1) & (2 * kSample - 1);
    }
  }
  __syncthreads();
  if (t == 0) *crowded = tree && distinct < kSample / 2 ? 1u : 0u;
}

__global__ __launch_bounds__(256) void k_query_keys(const cubql_box3f *rootBox, cubql_bvh3f bvh, QueryPlaces q,
                                                    const uint32_t *crowded, int bits, int slotShift, uint32_t *keys) {
  const bool slots = *crowded != 0;
  const cubql_box3f bounds = *rootBox;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < q.n; i += gridDim.x * blockDim.x) {
    const float3 p = place(q, i);
    if (slots) {
      cubql_dev::NoStats st;
      keys[i] = cubql_dev::oc_off(cubql_dev::nearest_leaf(bvh, p.x, p.y, p.z, 0u, st)) >> slotShift;
    } else {
      keys[i] = morton_key(bounds, p) >> (30 - bits);
    }
  }
}

}  // namespace qo

size_t query_order_ws_bytes(uint32_t nq) {
  if (nq < kQueryOrderMin) return 0;
  const size_t arr = ((size_t)nq * 4 + 255) & ~(size_t)255;
  return 4 * arr + 256 + radix_sort_ws_bytes(nq, qo::order_bits(nq));
}

int query_order_ws(const cubql_box3f *rootBox, const cubql_bvh3f *bvh, const QueryPlaces &q, hipStream_t s, void *ws,
                   const uint32_t **order) {
  *order = nullptr;
  if (q.n < kQueryOrderMin) return CUBQL_OK;
  const size_t arr = ((size_t)q.n * 4 + 255) & ~(size_t)255;
  char *p = (char *)ws;
  uint32_t *kA = (uint32_t *)p, *vA = (uint32_t *)(p + arr), *kB = (uint32_t *)(p + 2 * arr),
           *vB = (uint32_t *)(p + 3 * arr), *cnt = (uint32_t *)(p + 4 * arr);
  void *sortWs = p + 4 * arr + 256;
  const int bits = qo::order_bits(q.n);
  int slotShift = 0;
  const cubql_bvh3f none{};
  if (bvh)
    while ((bvh->numPrims >> slotShift) >> bits) slotShift++;
  qo::k_sample<<<1, qo::kSample, 0, s>>>(rootBox, q, cnt, cnt + 1, bvh != nullptr);
  qo::k_query_keys<<<std::min<uint32_t>(div_up(q.n, 256), 4096), 256, 0, s>>>(rootBox, bvh ? *bvh : none, q, cnt + 1,
                                                                             bits, slotShift, kA);
  CUBQL_LAUNCH_CHECK();
  uint32_t *kRes = nullptr, *vRes = nullptr;
  CUBQL_CHECK(radix_sort_iota_ws_u32(kA, vA, kB, vB, cnt, q.n, bits, s, sortWs, &kRes, &vRes));
  *order = vRes;
  return CUBQL_OK;
}

}  // namespace cubql
