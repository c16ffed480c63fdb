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
// Boxes that share a wave's walk are sorted by 24 bits where the 16-bit cells are
// crowded (k_sample): flat and peaked scenes fill few of them (of 1M boxes on a
// plane, 634 of 1024 sampled ones differ), and the wave then walks the tree for
// boxes far apart: 879 us a call with 16 bits, 386 with 24; uniform boxes 717
// with 24, 705 with 16.
constexpr uint32_t kFewQueries = 1u << 20;
inline int order_bits(uint32_t nq, bool boxes) { return nq <= kFewQueries && !boxes ? 16 : 24; }

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

// What a sample of the queries decides, in device memory.
struct Decision {
  uint32_t count;    // queries (the sort reads it)
  uint32_t crowded;  // keys are leaf slots, not Morton cells
  uint32_t coarse;   // the low key byte is not sorted by
};

// Adds a key to a table of the different ones; true if it is a new one.
constexpr uint32_t kSample = 1024;
__device__ __forceinline__ bool table_add(uint32_t (&table)[2 * kSample], uint32_t key) {
  uint32_t slot = (key * 2654435761u) >> 21;
  // (at most kSample keys in 2 kSample slots: the probe ends)
  for (uint32_t i = 0; i < 2 * kSample; i++) {
    const uint32_t old = atomicCAS(&table[slot], 0xffffffffu, key);
    if (old == 0xffffffffu) return true;
    if (old == key) return false;
    slot = (slot + 1) & (2 * kSample - 1);
  }
  return false;
}

// Counts the different Morton cells of kSample queries spread over the batch.
// crowded: of 24 bits, fewer than half the queries looked at.  A few far-off prims
// stretch the root box, and then Morton cells order nothing (2M points of 64
// tight clusters with 1% of them 1e6 away: 18 of 1024).
// coarse (boxes up to kFewQueries): E cells that are equally full leave kSample^2 /
// 2E of the sample in a cell with an earlier one, so that up to 16 kSample^2 / n of
// them mean no more than 32 queries to a cell, half a wave, and 16 bits do.
__global__ __launch_bounds__(kSample) void k_sample(const cubql_box3f *rootBox, QueryPlaces q, Decision *dec,
                                                    bool tree) {
  __shared__ uint32_t fine[2 * kSample], coarse[2 * kSample];
  __shared__ uint32_t distinct[2];
  const uint32_t t = threadIdx.x;
  const bool few = q.boxes && q.n <= kFewQueries;
  if (t < 2) distinct[t] = 0;
  fine[t] = fine[t + kSample] = coarse[t] = coarse[t + kSample] = 0xffffffffu;
  __syncthreads();
  if (tree || few) {
    const uint32_t key = morton_key(*rootBox, place(q, (uint32_t)((uint64_t)t * q.n / kSample))) >> 6;
    if (tree && table_add(fine, key)) atomicAdd(&distinct[0], 1u);
    if (few && table_add(coarse, key >> 8)) atomicAdd(&distinct[1], 1u);
  }
  __syncthreads();
  if (t == 0) {
    const bool crowded = tree && distinct[0] < kSample / 2;
    dec->count = q.n;
    dec->crowded = crowded ? 1u : 0u;
    dec->coarse =
        few && (crowded || (uint64_t)(kSample - distinct[1]) * q.n <= 16ull * kSample * kSample) ? 1u : 0u;
  }
}

// One key per query, in keysB (where the pass over the low byte would have left it)
// where that byte is not sorted by.
__global__ __launch_bounds__(256) void k_query_keys(const cubql_box3f *rootBox, cubql_bvh3f bvh, QueryPlaces q,
                                                    const Decision *dec, int bits, int slotShift, int slotUp,
                                                    uint32_t *keys, uint32_t *keysB) {
  const bool slots = dec->crowded != 0;
  uint32_t *const out = dec->coarse ? keysB : keys;
  const cubql_box3f bounds = *rootBox;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < q.n; i += gridDim.x * blockDim.x) {
    const float3 p = place(q, i);
    if (slots) {
      cubql_dev::NoStats st;
      out[i] = cubql_dev::oc_off(cubql_dev::nearest_leaf(bvh, p.x, p.y, p.z, 0u, st)) >> slotShift << slotUp;
    } else {
      out[i] = morton_key(bounds, p) >> (30 - bits);
    }
  }
}

}  // namespace qo

size_t query_order_ws_bytes(uint32_t nq) {
  if (nq < kQueryOrderMin) return 0;
  const size_t arr = ((size_t)nq * 4 + 255) & ~(size_t)255;
  return 4 * arr + 256 + radix_sort_ws_bytes(nq, 24);
}

int query_order_ws(const cubql_box3f *rootBox, const cubql_bvh3f *bvh, const QueryPlaces &q, hipStream_t s, void *ws,
                   const uint32_t **order) {
  *order = nullptr;
  if (q.n < kQueryOrderMin) return CUBQL_OK;
  const size_t arr = ((size_t)q.n * 4 + 255) & ~(size_t)255;
  char *p = (char *)ws;
  uint32_t *kA = (uint32_t *)p, *vA = (uint32_t *)(p + arr), *kB = (uint32_t *)(p + 2 * arr),
           *vB = (uint32_t *)(p + 3 * arr);
  qo::Decision *dec = (qo::Decision *)(p + 4 * arr);
  void *sortWs = p + 4 * arr + 256;
  const int bits = qo::order_bits(q.n, q.boxes);
  int slotShift = 0;
  const cubql_bvh3f none{};
  // (crowded boxes are sorted by the top 16 bits)
  const int slotBits = q.boxes && q.n <= qo::kFewQueries ? 16 : bits;
  if (bvh)
    while ((bvh->numPrims >> slotShift) >> slotBits) slotShift++;
  qo::k_sample<<<1, qo::kSample, 0, s>>>(rootBox, q, dec, bvh != nullptr);
  qo::k_query_keys<<<std::min<uint32_t>(div_up(q.n, 256), 4096), 256, 0, s>>>(rootBox, bvh ? *bvh : none, q, dec, bits,
                                                                             slotShift, bits - slotBits, kA, kB);
  CUBQL_LAUNCH_CHECK();
  uint32_t *kRes = nullptr, *vRes = nullptr;
  CUBQL_CHECK(radix_sort_iota_ws_u32(kA, vA, kB, vB, &dec->count, q.n, bits, s, sortWs, &kRes, &vRes,
                                     q.boxes ? &dec->coarse : nullptr));
  *order = vRes;
  return CUBQL_OK;
}

}  // namespace cubql
