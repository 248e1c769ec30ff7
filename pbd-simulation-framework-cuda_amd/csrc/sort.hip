// sort.hip - stable LSD radix sort of (cell id, particle index) for gfx950.
//
// Replaces the reference's CUB DeviceRadixSort::SortPairs over all 32 key bits
// (kernel/SortReorder.h:39-47; 7 digit passes x {upsweep, scan, downsweep}).
// Only the significant bits of the Morton cell id are sorted (ceil(bits/8)
// 8-bit passes), and each pass is one "onesweep" kernel:
//   - a tile of 256 x ITEMS keys per 256-thread workgroup (ITEMS = 4, 8 or 16,
//     chosen per particle count: enough tiles to fill the CUs, else long digit
//     runs for the scattered writes), tile index from an atomic ticket so a
//     tile only ever waits on tiles that already started;
//   - stable in-tile ranking by wave64 multisplit (8 ballots per key give the
//     lanes with the same digit; rank = popcount below the lane);
//   - decoupled look-back over per-tile digit counts for the global offset;
//   - the tile is reordered by digit in LDS and written out in runs.
// The digit counts of all passes are added up by the kernel that makes the
// keys (k_predict_keys), so the keys are not read an extra time for them.  The
// first pass takes the particle index as the value (iota), so the value array
// is never read before it exists.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace pbd {

namespace {
constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagPre = 2u << 30;
constexpr uint32_t kValMask = (1u << 30) - 1u;
constexpr uint32_t kSpinLimit = 1u << 24;
constexpr uint32_t kWaves = kSortThreads / 64;
#ifndef PBD_SORT_LOOKBACK
#define PBD_SORT_LOOKBACK 4
#endif
constexpr uint32_t kLookBack = PBD_SORT_LOOKBACK;  // predecessor words read per look-back round trip
}  // namespace

// The largest tile that still gives a tile per CU (2^20 keys: 256 tiles of
// 4096, 38 against 43 us per pass with 512 of 2048).
uint32_t sort_items_for(uint32_t n) {
  for (uint32_t items = 16; items > kSortItemsMin; items >>= 1)
    if ((n + kSortThreads * items - 1) / (kSortThreads * items) >= 256u) return items;
  return kSortItemsMin;
}

uint32_t sort_hist_copies(uint32_t n, uint32_t tpb) {
  const uint32_t blocks = (n + tpb - 1) / tpb;
  return blocks < kSortHistCopies ? (blocks ? blocks : 1u) : kSortHistCopies;
}

uint32_t sort_passes_for(uint32_t key_bound) {
  uint32_t maxk = key_bound ? key_bound - 1u : 0u;
  uint32_t bits = 0;
  while (maxk) {
    ++bits;
    maxk >>= 1;
  }
  uint32_t p = (bits + 7u) / 8u;
  return p ? p : 1u;
}

__global__ void k_sort_prepare(uint32_t* __restrict__ hist, uint32_t* __restrict__ tile_ctr,
                               uint32_t* __restrict__ status, uint32_t status_words) {
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = gid; i < kSortHistWords; i += stride) hist[i] = 0u;
  if (gid < 4u) tile_ctr[gid] = 0u;
  for (uint32_t i = gid; i < status_words; i += stride) status[i] = 0u;
}

// Exclusive scan of each pass's 256 digit counts, summed over the histogram's
// copies: one workgroup, a thread per (pass, digit), every copy's load in
// flight at once.
__global__ __launch_bounds__(1024) void k_sort_scan(uint32_t* __restrict__ hist, uint32_t passes, uint32_t copies) {
  __shared__ uint32_t s[4][256];
  const uint32_t t = threadIdx.x & 255u, p = threadIdx.x >> 8;
  uint32_t v = 0;
  if (p < passes) {
    uint32_t a[kSortHistCopies];
#pragma unroll
    for (uint32_t c = 0; c < kSortHistCopies; ++c) a[c] = c < copies ? hist[1024u * (1u + c) + p * 256u + t] : 0u;
#pragma unroll
    for (uint32_t c = 0; c < kSortHistCopies; ++c) v += a[c];
  }
  s[p][t] = v;
  __syncthreads();
  for (uint32_t o = 1; o < 256u; o <<= 1) {
    const uint32_t add = t >= o ? s[p][t - o] : 0u;
    __syncthreads();
    s[p][t] += add;
    __syncthreads();
  }
  if (p < passes) hist[p * 256u + t] = s[p][t] - v;
}

template <uint32_t ITEMS>
__global__ __launch_bounds__(kSortThreads) void k_onesweep(const uint32_t* __restrict__ kin,
                                                          const uint32_t* __restrict__ vin,
                                                          uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                          uint32_t n, uint32_t shift,
                                                          const uint32_t* __restrict__ offs,
                                                          uint32_t* __restrict__ tile_ctr,
                                                          uint32_t* __restrict__ status, uint32_t* __restrict__ err,
                                                          int iota_vals) {
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_wcnt[kWaves][256];
  __shared__ uint32_t s_tdig[256];
  __shared__ uint32_t s_gbase[256];
  __shared__ uint32_t s_wsum[kWaves];
  constexpr uint32_t kTile = kSortThreads * ITEMS;
  __shared__ uint32_t s_keys[kTile];
  __shared__ uint32_t s_vals[kTile];

  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u;
  const uint32_t wave = tid >> 6;
  if (tid == 0) s_tile = atomicAdd(tile_ctr, 1u);
  for (uint32_t i = tid; i < kWaves * 256u; i += kSortThreads) (&s_wcnt[0][0])[i] = 0u;
  __syncthreads();
  const uint32_t tile = s_tile;
  const uint32_t base = tile * kTile;

  uint32_t keys[ITEMS], vals[ITEMS], rank[ITEMS];
#pragma unroll
  for (uint32_t r = 0; r < ITEMS; ++r) {
    const uint32_t idx = base + wave * (64u * ITEMS) + r * 64u + lane;
    const bool valid = idx < n;
    keys[r] = valid ? kin[idx] : 0xFFFFFFFFu;
    vals[r] = valid ? (iota_vals ? idx : vin[idx]) : 0u;
  }

  // Stable in-wave ranking: wave w covers a contiguous range, rounds in order,
  // lanes in order, so (wave, round, lane) is the index order.
  const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
  for (uint32_t r = 0; r < ITEMS; ++r) {
    const uint32_t idx = base + wave * (64u * ITEMS) + r * 64u + lane;
    const bool valid = idx < n;
    const uint32_t d = (keys[r] >> shift) & 255u;
    uint64_t m = __ballot(valid);
#pragma unroll
    for (uint32_t b = 0; b < 8u; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      m &= bit ? bb : ~bb;
    }
    uint32_t rk = 0;
    if (valid) {
      const uint32_t pre = s_wcnt[wave][d];
      rk = pre + (uint32_t)__popcll(m & lt);
      if ((m & lt) == 0ull) s_wcnt[wave][d] = pre + (uint32_t)__popcll(m);
    }
    rank[r] = rk;
  }
  __syncthreads();

  // Per digit (thread = digit): tile count, wave-exclusive offsets.
  const uint32_t dg = tid;
  uint32_t cnt = 0;
#pragma unroll
  for (uint32_t w = 0; w < kWaves; ++w) {
    const uint32_t c = s_wcnt[w][dg];
    s_wcnt[w][dg] = cnt;
    cnt += c;
  }
  uint32_t* my_status = status + (size_t)tile * 256u + dg;
  __hip_atomic_store(my_status, (tile == 0 ? kFlagPre : kFlagAgg) | cnt, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);

  // Exclusive scan of the tile's digit counts.
  uint32_t x = cnt;
#pragma unroll
  for (uint32_t o = 1; o < 64u; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63u) s_wsum[wave] = x;

  // Decoupled look-back for this digit, kLookBack predecessors per round trip:
  // their words are taken in order up to the first one not yet published (read
  // again in the next round) or the first inclusive prefix (the end).
  uint32_t excl = 0;
  if (tile > 0) {
    int t = (int)tile - 1;
    uint32_t spins = 0;
    bool found = false;
    while (!found) {
      uint32_t v[kLookBack];
#pragma unroll
      for (uint32_t k = 0; k < kLookBack; ++k)
        v[k] = t >= (int)k ? __hip_atomic_load(status + (size_t)(t - (int)k) * 256u + dg, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)
                           : 0u;
      int taken = 0;
#pragma unroll
      for (uint32_t k = 0; k < kLookBack; ++k) {
        const uint32_t fl = v[k] >> 30;
        if (fl == 0u) break;  // tile 0 always publishes a prefix, so t - k >= 0 here
        excl += v[k] & kValMask;
        ++taken;
        if (fl == 2u) {
          found = true;
          break;
        }
      }
      if (found) break;
      t -= taken;
      if (taken == 0) {
        if (++spins > kSpinLimit) {
          // may be host memory: a plain store, the same from every wave
          __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __hip_atomic_store(my_status, kFlagPre | ((excl + cnt) & kValMask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  s_gbase[dg] = offs[dg] + excl;
  __syncthreads();
  uint32_t wpre = 0;
  for (uint32_t w = 0; w < wave; ++w) wpre += s_wsum[w];
  s_tdig[dg] = x - cnt + wpre;
  __syncthreads();

  // Stage the tile in digit order.
#pragma unroll
  for (uint32_t r = 0; r < ITEMS; ++r) {
    const uint32_t idx = base + wave * (64u * ITEMS) + r * 64u + lane;
    if (idx < n) {
      const uint32_t d = (keys[r] >> shift) & 255u;
      const uint32_t pos = s_tdig[d] + s_wcnt[wave][d] + rank[r];
      s_keys[pos] = keys[r];
      s_vals[pos] = vals[r];
    }
  }
  __syncthreads();
  const uint32_t tile_n = (n - base) < kTile ? (n - base) : kTile;
  for (uint32_t i = tid; i < tile_n; i += kSortThreads) {
    const uint32_t k = s_keys[i];
    const uint32_t d = (k >> shift) & 255u;
    const uint32_t dst = s_gbase[d] + (i - s_tdig[d]);
    if (dst < n) {  // always true unless a look-back hit its spin limit (reported through err)
      kout[dst] = k;
      vout[dst] = s_vals[i];
    }
  }
}

hipError_t launch_sort_prepare(hipStream_t st, const SortPlan& plan, uint32_t n) {
  if (n == 0) return hipSuccess;
  if (n > plan.n_max) return hipErrorInvalidValue;
  const uint32_t items = plan.items ? plan.items : sort_items_for(n);
  const uint32_t tiles = (n + kSortThreads * items - 1) / (kSortThreads * items);
  const uint32_t status_words = plan.passes * tiles * 256u;
  uint32_t b = (status_words + 255u) / 256u;
  if (b < 4u) b = 4u;
  if (b > 2048u) b = 2048u;
  hipLaunchKernelGGL(k_sort_prepare, dim3(b), dim3(256), 0, st, plan.hist, plan.tile_ctr, plan.status, status_words);
  return hipGetLastError();
}

template <uint32_t ITEMS>
static void onesweep_passes(hipStream_t st, const SortPlan& plan, uint32_t n, const uint32_t* keys_in) {
  const uint32_t tiles = (n + kSortThreads * ITEMS - 1) / (kSortThreads * ITEMS);
  const uint32_t passes = plan.passes;
  const uint32_t* kin = keys_in;
  const uint32_t* vin = nullptr;
  for (uint32_t p = 0; p < passes; ++p) {
    const bool to_out = ((passes - 1u - p) % 2u) == 0u;
    uint32_t* ko = to_out ? plan.keys_out : plan.keys_alt;
    uint32_t* vo = to_out ? plan.vals_out : plan.vals_alt;
    hipLaunchKernelGGL(k_onesweep<ITEMS>, dim3(tiles), dim3(kSortThreads), 0, st, kin, vin, ko, vo, n, 8u * p,
                       plan.hist + 256u * p, plan.tile_ctr + p, plan.status + (size_t)p * tiles * 256u, plan.err,
                       p == 0 ? 1 : 0);
    kin = ko;
    vin = vo;
  }
}

hipError_t launch_sort_ranks(hipStream_t st, const SortPlan& plan, uint32_t n, const uint32_t* keys_in,
                             const uint32_t** keys_res, const uint32_t** vals_res) {
  *keys_res = plan.keys_out;
  *vals_res = plan.vals_out;
  if (n == 0) return hipSuccess;
  if (n > plan.n_max) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(1024), 0, st, plan.hist, plan.passes, kSortHistCopies);
  switch (plan.items ? plan.items : sort_items_for(n)) {
    case 4: onesweep_passes<4>(st, plan, n, keys_in); break;
    case 8: onesweep_passes<8>(st, plan, n, keys_in); break;
    case 16: onesweep_passes<16>(st, plan, n, keys_in); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace pbd
