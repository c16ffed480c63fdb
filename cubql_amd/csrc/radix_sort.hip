// radix_sort.hip -- stable onesweep LSD key/value radix sort (see radix_sort.h).
#include "block_ops.h"
#include "common.h"
#include "profile.h"
#include "radix_sort.h"

#include "build_common.h"

namespace cubql {
namespace rs {

// A tile is 512 threads x ITEMS keys, staged in LDS once for the keys and
// once for the values.  Large sorts take large tiles (longer runs per digit:
// 32M random 24-bit pairs 0.75 ms with 20 keys a thread, 0.84 with 12; 32M
// 64-bit pairs 1.95 ms with 16, 2.35 with 8), small ones take 8 keys a thread,
// so that more CUs have a tile (100K 64-bit pairs 117 us with 8, 152 with 16;
// 1M 192 and 210).
constexpr int kBlock = 512;
constexpr int kSmallItems = 8;
constexpr uint32_t kSmallSort = 1u << 21;
template <typename K>
constexpr int kLargeItems = sizeof(K) == 4 ? 20 : 16;
constexpr uint32_t kDigits = 256;

// status word of (tile, digit): tag(22) | flag(2) | value(32)
__device__ __forceinline__ uint64_t st_word(uint32_t tag, uint32_t flag, uint32_t v) {
  return ((uint64_t)tag << 34) | ((uint64_t)flag << 32) | v;
}

// Digit counts of every pass: a sub-histogram per wave in LDS, then one
// global atomic per digit, pass and workgroup.  skipLow: as in radix_sort.h;
// kSkip: some of the sorts have it (tested at run time in all of them, 30916
// 63-bit keys: 9.9 us against 7.6, and 10.7 a pass against 10.4).
constexpr int kHistBlock = 256;
constexpr int kHistWaves = kHistBlock / kWave;
template <typename K, bool kSkip>
__global__ __launch_bounds__(kHistBlock) void k_hist(const K *keys, const K *keysB, const uint32_t *skipLow,
                                                     const uint32_t *nPtr, int passes, uint32_t *digitCount) {
  extern __shared__ uint32_t h[];  // [kHistWaves][passes][kDigits]
  const bool skip = kSkip && *skipLow;
  if (skip) keys = keysB;
  const uint32_t n = *nPtr;
  const int words = passes * (int)kDigits;
  for (int i = threadIdx.x; i < kHistWaves * words; i += kHistBlock) h[i] = 0;
  __syncthreads();
  uint32_t *hw = h + (threadIdx.x / kWave) * words;
  constexpr int U = 4;
  const uint64_t stride = (uint64_t)gridDim.x * kHistBlock * U;
  for (uint64_t i0 = (uint64_t)blockIdx.x * kHistBlock * U + threadIdx.x; i0 < n; i0 += stride) {
    K key[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint64_t i = i0 + u * kHistBlock;
      key[u] = i < n ? keys[i] : (K)0;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (i0 + u * kHistBlock < n)
        for (int p = skip ? 1 : 0; p < passes; p++)
          atomicAdd(&hw[p * kDigits + ((uint32_t)(key[u] >> (8 * p)) & 255u)], 1u);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < words; i += kHistBlock) {
    uint32_t v = 0;
    for (int w = 0; w < kHistWaves; w++) v += h[w * words + i];
    if (v) atomicAdd(&digitCount[i], v);
  }
}

// One pass over 8 key bits, a tile per workgroup.  Tiles are claimed in
// ticket order, so every tile a look-back waits on is held by a running
// workgroup.  What bounds it: the latency of a tile's chain (loads, ranking,
// look-back, two copies out) against the tiles in flight; all of a thread's
// loads are issued before the ranking, and keys and values share one LDS
// buffer so that more tiles fit a CU.
template <typename K, int ITEMS, bool kSkip>
__global__ __launch_bounds__(kBlock) void k_onesweep(const K *__restrict__ kin,
                                                              const uint32_t *__restrict__ vin,
                                                              K *__restrict__ kout, uint32_t *__restrict__ vout,
                                                              const uint32_t *nPtr, int shift, uint32_t tag,
                                                              const uint32_t *digitCount, uint64_t *status,
                                                              uint32_t *ticket, uint32_t *err,
                                                              const uint32_t *skipLow) {
  constexpr int BLOCK = kBlock, NW = BLOCK / kWave;
  constexpr uint32_t TILE = BLOCK * ITEMS;
  static_assert(BLOCK >= (int)kDigits, "one thread per digit");
  __shared__ uint32_t sHist[NW][kDigits];
  __shared__ uint32_t sGlob[kDigits];  // global slot of a digit's first key less its slot in the tile
  __shared__ uint32_t ss[2][BLOCK / kWave + 1];
  __shared__ __align__(16) unsigned char sBuf[TILE * sizeof(K)];
  __shared__ uint32_t sTile;
  K *const sK = reinterpret_cast<K *>(sBuf);
  uint32_t *const sV = reinterpret_cast<uint32_t *>(sBuf);
  const bool skip = kSkip && *skipLow;
  if (skip && shift == 0) return;
  const uint32_t n = *nPtr;
  const uint32_t lane = lane_id(), w = threadIdx.x / kWave;
  if (threadIdx.x == 0) sTile = atomicAdd(ticket, 1u);
  for (int i = threadIdx.x; i < NW * (int)kDigits; i += BLOCK) (&sHist[0][0])[i] = 0;
  const uint32_t dgt = threadIdx.x;
  const uint32_t dcount = dgt < kDigits ? digitCount[dgt] : 0u;
  __syncthreads();
  const uint32_t t = sTile;
  if (t >= div_up(n, TILE)) return;
  const uint32_t tileBase = t * TILE;
  const uint32_t tileN = min(TILE, n - tileBase);
  const uint32_t li0 = w * (ITEMS * kWave) + lane;
  K key[ITEMS];
  uint32_t val[ITEMS], rank[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) key[k] = li0 + k * kWave < tileN ? kin[tileBase + li0 + k * kWave] : (K)0;
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = tileBase + li0 + k * kWave;
    val[k] = li0 + k * kWave < tileN ? (vin && !skip ? vin[i] : i) : 0u;
  }
  uint32_t tot;
  const uint32_t digitBase = block_excl_scan<BLOCK, true>(dcount, ss[0], &tot);
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const bool valid = li0 + k * kWave < tileN;
    const uint32_t d = (uint32_t)(key[k] >> shift) & 255u;
    // lanes with the same digit
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const bool bit = (d >> b) & 1u;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const uint32_t pre = mbcnt(peers);
    const uint32_t base = valid ? sHist[w][d] : 0u;
    rank[k] = base + pre;
    __builtin_amdgcn_wave_barrier();
    if (valid && pre == 0) sHist[w][d] = base + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
  sync_block_lds();
  // per digit: exclusive offsets across waves, tile total
  uint32_t dtot = 0;
  uint64_t *const my = status + (size_t)t * kDigits + dgt;
  if (dgt < kDigits) {
#pragma unroll
    for (int ww = 0; ww < NW; ww++) {
      const uint32_t c = sHist[ww][dgt];
      sHist[ww][dgt] = dtot;
      dtot += c;
    }
    __hip_atomic_store(my, st_word(tag, t == 0 ? 2 : 1, dtot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const uint32_t tileEx = block_excl_scan<BLOCK, true>(dtot, ss[1], &tot);
  // slot of each key in the tile's digit order
  if (dgt < kDigits)
#pragma unroll
    for (int ww = 0; ww < NW; ww++) sHist[ww][dgt] += tileEx;
  sync_block_lds();
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t d = (uint32_t)(key[k] >> shift) & 255u;
    rank[k] += sHist[w][d];
    if (li0 + k * kWave < tileN) sK[rank[k]] = key[k];
  }
  // decoupled look-back for this digit across earlier tiles
  if (dgt < kDigits) {
    uint32_t prefix = 0;
    if (t) {
      uint32_t j = t - 1;
      uint32_t spins = 0;
      while (true) {
        const uint64_t wv = __hip_atomic_load(status + (size_t)j * kDigits + dgt, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t wt = (uint32_t)(wv >> 34), wf = (uint32_t)(wv >> 32) & 3u;
        if (wt != tag || wf == 0) {
          // bounded when the caller checks err (build_common.h, kSpinLimit):
          // the prefix so far is at most the true one, so writes stay in range
          if (err && ++spins > kSpinLimit) {
            atomicOr(err, 1u);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
          continue;
        }
        prefix += (uint32_t)wv;
        if (wf == 2) break;
        j--;
      }
      __hip_atomic_store(my, st_word(tag, 2, prefix + dtot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    sGlob[dgt] = digitBase + prefix - tileEx;
  }
  sync_block_lds();
  // keys, then values, in digit order: runs of consecutive addresses
  uint32_t dst[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = k * BLOCK + threadIdx.x;
    if (i < tileN) {
      const K kk = sK[i];
      dst[k] = sGlob[(uint32_t)(kk >> shift) & 255u] + i;
      kout[dst[k]] = kk;
    }
  }
  sync_block_lds();
#pragma unroll
  for (int k = 0; k < ITEMS; k++)
    if (li0 + k * kWave < tileN) sV[rank[k]] = val[k];
  sync_block_lds();
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const uint32_t i = k * BLOCK + threadIdx.x;
    if (i < tileN) vout[dst[k]] = sV[i];
  }
}

// Scratch layout (bytes): status | digitCount | tickets, cleared by one fill.
size_t sort_ws_bytes(uint32_t nMax, int keyBits) {
  const int passes = (keyBits + 7) / 8;
  const size_t maxTiles = std::max<uint32_t>(1u, div_up(nMax, kBlock * kSmallItems));
  return maxTiles * kDigits * 8 + (size_t)passes * kDigits * 4 + 64 + 256;
}

template <typename K>
int sort_pairs_ws(K *kA, uint32_t *vA, K *kB, uint32_t *vB, const uint32_t *nDev, uint32_t nMax,
                  int keyBits, hipStream_t s, void *ws, K **kRes, uint32_t **vRes, uint32_t *err = nullptr,
                  bool iota = false, const uint32_t *skipLow = nullptr) {
  const int passes = (keyBits + 7) / 8;
  const bool small = nMax < kSmallSort;
  const uint32_t maxTiles = std::max<uint32_t>(1u, div_up(nMax, kBlock * (small ? kSmallItems : kLargeItems<K>)));
  uint64_t *status = (uint64_t *)ws;
  uint32_t *digitCount = (uint32_t *)(status + (size_t)maxTiles * kDigits);
  uint32_t *tickets = digitCount + (size_t)passes * kDigits;
  CUBQL_CHECK(fill_u32((uint32_t *)status, 0u, (size_t)maxTiles * kDigits * 2 + (size_t)passes * kDigits + 16, s));
  // (two workgroups a CU: the global atomics of more would queue up)
  const uint32_t histBlocks = std::max(1u, std::min(div_up(nMax, 4096), 512u));
  auto hist = k_hist<K, false>;
  auto pass = small ? k_onesweep<K, kSmallItems, false> : k_onesweep<K, kLargeItems<K>, false>, low = pass;
  if constexpr (sizeof(K) == 4) {
    if (skipLow) {
      hist = k_hist<K, true>;
      low = small ? k_onesweep<K, kSmallItems, true> : k_onesweep<K, kLargeItems<K>, true>;
    }
  }
  hist<<<histBlocks, kHistBlock, (size_t)kHistWaves * passes * kDigits * 4, s>>>(kA, kB, skipLow, nDev, passes,
                                                                                 digitCount);
  K *ki = kA, *ko = kB;
  uint32_t *vi = vA, *vo = vB;
  for (int p = 0; p < passes; p++) {
    int ps = prof_begin(s);
    // (the second pass takes the values 0, 1, 2, ... where the first does nothing)
    (p < 2 ? low : pass)<<<maxTiles, kBlock, 0, s>>>(ki, iota && p == 0 ? nullptr : vi, ko, vo, nDev, 8 * p,
                                                     (uint32_t)(p + 1), digitCount + p * kDigits, status,
                                                     tickets + p, err, skipLow);
    prof_end(ps, s, "radix_onesweep");
    prof_set(ps, (double)nMax * 2.0 * (sizeof(K) + 4), nMax);
    std::swap(ki, ko);
    std::swap(vi, vo);
  }
  CUBQL_LAUNCH_CHECK();
  *kRes = ki;
  *vRes = vi;
  return CUBQL_OK;
}

template <typename K>
int sort_pairs(K *kA, uint32_t *vA, K *kB, uint32_t *vB, const uint32_t *nDev, uint32_t nMax,
               int keyBits, hipStream_t s, const cubql_mem_resource *mem, K **kRes, uint32_t **vRes,
               uint32_t *err) {
  Scratch scr(mem, s);
  char *ws = nullptr;
  CUBQL_CHECK(scr.alloc(&ws, sort_ws_bytes(nMax, keyBits)));
  return sort_pairs_ws<K>(kA, vA, kB, vB, nDev, nMax, keyBits, s, ws, kRes, vRes, err);
}

}  // namespace rs

size_t radix_sort_ws_bytes(uint32_t nMax, int keyBits) { return rs::sort_ws_bytes(nMax, keyBits); }
int radix_sort_pairs_ws_u32(uint32_t *kA, uint32_t *vA, uint32_t *kB, uint32_t *vB, const uint32_t *nDev,
                            uint32_t nMax, int keyBits, hipStream_t s, void *ws, uint32_t **kRes,
                            uint32_t **vRes) {
  return rs::sort_pairs_ws<uint32_t>(kA, vA, kB, vB, nDev, nMax, keyBits, s, ws, kRes, vRes);
}
int radix_sort_iota_ws_u32(uint32_t *kA, uint32_t *vA, uint32_t *kB, uint32_t *vB, const uint32_t *nDev,
                           uint32_t nMax, int keyBits, hipStream_t s, void *ws, uint32_t **kRes, uint32_t **vRes,
                           const uint32_t *skipLow) {
  return rs::sort_pairs_ws<uint32_t>(kA, vA, kB, vB, nDev, nMax, keyBits, s, ws, kRes, vRes, nullptr, true, skipLow);
}
int radix_sort_pairs_ws_u64(uint64_t *kA, uint32_t *vA, uint64_t *kB, uint32_t *vB, const uint32_t *nDev,
                            uint32_t nMax, int keyBits, hipStream_t s, void *ws, uint64_t **kRes,
                            uint32_t **vRes) {
  return rs::sort_pairs_ws<uint64_t>(kA, vA, kB, vB, nDev, nMax, keyBits, s, ws, kRes, vRes);
}

int radix_sort_pairs_dev_u32(uint32_t *kA, uint32_t *vA, uint32_t *kB, uint32_t *vB, const uint32_t *nDev,
                             uint32_t nMax, int keyBits, hipStream_t s, const cubql_mem_resource *mem,
                             uint32_t **kRes, uint32_t **vRes, uint32_t *err) {
  return rs::sort_pairs<uint32_t>(kA, vA, kB, vB, nDev, nMax, keyBits, s, mem, kRes, vRes, err);
}
int radix_sort_pairs_dev_u64(uint64_t *kA, uint32_t *vA, uint64_t *kB, uint32_t *vB, const uint32_t *nDev,
                             uint32_t nMax, int keyBits, hipStream_t s, const cubql_mem_resource *mem,
                             uint64_t **kRes, uint32_t **vRes, uint32_t *err) {
  return rs::sort_pairs<uint64_t>(kA, vA, kB, vB, nDev, nMax, keyBits, s, mem, kRes, vRes, err);
}

}  // namespace cubql

namespace {
template <typename K>
int sort_entry(K *keys, uint32_t *vals, K *keysTmp, uint32_t *valsTmp, uint32_t n, int keyBits,
               cubql_stream_t stream) {
  using namespace cubql;
  clear_error();
  if (n == 0) return CUBQL_OK;
  if (!keys || !vals || !keysTmp || !valsTmp || keyBits < 1 || keyBits > 8 * (int)sizeof(K)) {
    set_error("radix sort: invalid argument");
    return CUBQL_ERR_INVALID_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  Scratch scr(nullptr, s);
  uint32_t *nDev = nullptr;
  CUBQL_CHECK(scr.alloc(&nDev, 1));
  CUBQL_CHECK(fill_u32(nDev, n, 1, s));
  K *kr = nullptr;
  uint32_t *vr = nullptr;
  CUBQL_CHECK(rs::sort_pairs<K>(keys, vals, keysTmp, valsTmp, nDev, n, keyBits, s, nullptr, &kr, &vr, nullptr));
  if (kr != keys) {
    CUBQL_HIP(hipMemcpyAsync(keys, kr, sizeof(K) * (size_t)n, hipMemcpyDeviceToDevice, s));
    CUBQL_HIP(hipMemcpyAsync(vals, vr, sizeof(uint32_t) * (size_t)n, hipMemcpyDeviceToDevice, s));
  }
  return CUBQL_OK;
}
}  // namespace

extern "C" int cubql_radix_sort_pairs_u32(uint32_t *d_keys, uint32_t *d_vals, uint32_t *d_keysTmp,
                                          uint32_t *d_valsTmp, uint32_t n, int keyBits,
                                          cubql_stream_t s) {
  return sort_entry<uint32_t>(d_keys, d_vals, d_keysTmp, d_valsTmp, n, keyBits, s);
}

extern "C" int cubql_radix_sort_pairs_u64(uint64_t *d_keys, uint32_t *d_vals, uint64_t *d_keysTmp,
                                          uint32_t *d_valsTmp, uint32_t n, int keyBits,
                                          cubql_stream_t s) {
  return sort_entry<uint64_t>(d_keys, d_vals, d_keysTmp, d_valsTmp, n, keyBits, s);
}
