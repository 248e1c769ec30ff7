// tiles.hip - LDS cell-block tile versions of the neighbour passes (gfx950).
//
// Particles are sorted by Morton cell id, so an aligned Morton block of 2^BITS
// cells (2x4x4 cells for BITS = 5, 4x4x4 for BITS = 6) is one contiguous range
// of the sorted arrays.  One 256-thread workgroup takes one occupied block:
//   1. it looks up the (EX+2)(EY+2)(EZ+2) halo cells in the cell table and
//      scans their counts into LDS offsets;
//   2. it copies the halo particles from HBM/L2 into LDS in block-local
//      coordinates (one float4 each, the pass's per-neighbour payload in .w:
//      lambda for the delta-p pass, |omega| for the vorticity pass);
//   3. every thread walks the 27-cell stencil of its own particles out of LDS.
// The per-pair arithmetic and the per-particle epilogues are the ones of the
// per-particle kernels (particle_ops.hpp).  A block whose halo does not fit in
// LDS, and a particle whose 27-cell count exceeds maxNeighboursPerParticle
// (where the reference's truncation order matters), take the per-particle
// global-memory path.  Only the 27-cell stencil (kernelWidthNeighbours = 1,
// findContacts on) is tiled; wider stencils use the per-particle kernels.
#include <hip/hip_runtime.h>

#include "adjoint_list.hpp"
#include "device.hpp"
#include "kernels.hpp"
#include "particle_ops.hpp"

namespace pbd {

template <int BITS>
struct TileGeom {
  static constexpr int EZ = 1 << ((BITS + 2) / 3);  // Morton bit order from the LSB is z, y, x, z, ...
  static constexpr int EY = 1 << ((BITS + 1) / 3);
  static constexpr int EX = 1 << (BITS / 3);
  static constexpr int HX = EX + 2, HY = EY + 2, HZ = EZ + 2;
  static constexpr int NH = HX * HY * HZ;  // halo cells
  static constexpr int SX = HY * HZ, SY = HZ;
};

constexpr uint32_t kTileThreads = 256;

// The thread's index.  LOOP, for a kernel whose workgroups take tile after tile: as a value
// that the compiler cannot trace to the hardware's.  What a tile derives from the index
// (halo cells, cell groups, addresses) is otherwise kept in registers over the whole loop:
// 143 to 172 VGPRs in the 2^5-cell passes of a capped grid, 110 to 127 so (with a bound of
// four waves for omega and final).  us, before / now: four steps of 256 scenes of 2K to 64K
// 54940 / 45790, a step of 1.2M particles in a 300-cell box 1818 / 1360, its splash 2650 / 2018.
template <bool LOOP>
__device__ __forceinline__ uint32_t thread_index() {
  uint32_t t = threadIdx.x;
  if (LOOP) asm volatile("" : "+v"(t));
  return t;
}

// A team walks one tile: the whole workgroup for a large tile, one wave for a
// small one.  A wave's LDS accesses complete in order, so a wave team needs no
// hardware barrier, only one the compiler does not move memory accesses across.
template <uint32_t N, bool LOOP = false>
struct TeamBlockN {
  static constexpr uint32_t kSize = N;
  static __device__ __forceinline__ uint32_t tid() { return thread_index<LOOP>(); }
  static __device__ __forceinline__ void sync() { __syncthreads(); }
};
using TeamBlock = TeamBlockN<kTileThreads>;
// The reverse-mode list builder for small scenes: four threads per particle.
constexpr uint32_t kWideThreads = 1024;
using TeamWide = TeamBlockN<kWideThreads>;
template <bool LOOP = false>
struct TeamWaveT {
  static constexpr uint32_t kSize = 64;
  static constexpr uint32_t kLoadUnroll = 4;  // halo loads in flight per lane
  static __device__ __forceinline__ uint32_t tid() { return thread_index<LOOP>() & 63u; }
  static __device__ __forceinline__ void sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
};
using TeamWave = TeamWaveT<>;

template <int BITS>
struct TileShared {
  uint32_t lstart[TileGeom<BITS>::NH + 1];  // LDS start of each halo cell; lstart[NH] = total
  uint32_t gstart[TileGeom<BITS>::NH];      // sorted index of the cell's first particle
  uint32_t wsum[kTileThreads / 64];
  float off[3][6];                          // per axis: halo cell's corner minus the block's first cell's corner
  uint32_t g0, g1;                          // the block's own particle range
  uint32_t dmax;                            // largest displacement bound in the halo (float bits)
};
static_assert(TileGeom<6>::HX <= 6 && TileGeom<6>::HY <= 6 && TileGeom<6>::HZ <= 6, "offset table");

// First sorted index of a block (its mark without kTileCrowded).
__device__ __forceinline__ uint32_t tile_begin(uint32_t start) { return (start & ~(kTileCrowded | kTileSplit)) - 1u; }

// A work item of the lists: a block, or one half of a block whose halo exceeds the tile
// capacity (half 1: its cells of y 0 and 1, half 2: of y 2 and 3; the halves of a 2^5-cell
// block are consecutive key ranges), and its own particles.
struct TileOwn {
  uint32_t blk, half, g0, g1;
  // its place in StepBuffers::BUILT and MODE
  __device__ __forceinline__ uint32_t carried() const { return 2u * blk + (half == 2u ? 1u : 0u); }
};
template <int BITS>
__device__ __forceinline__ TileOwn tile_own(const DevParams& P, const TileList& T, uint32_t item,
                                            const uint32_t* __restrict__ cs) {
  TileOwn o;
  o.half = BITS == 5 ? item >> 30 : 0u;
  o.blk = item & (kTileSplit - 1u);
  o.g0 = tile_begin(T.start[o.blk]);
  o.g1 = T.end[o.blk];
  if (o.half) {
    uint32_t mid = o.g1;  // the first particle of the second half (an empty cell starts at 2^32 - 1)
    for (uint32_t c = 16u; c < 32u; ++c) {
      const uint32_t k = (o.blk << 5) + c;
      if (compact10(k >> 2) < P.dims[0] && compact10(k >> 1) < P.dims[1] && compact10(k) < P.dims[2])
        mid = min(mid, cs[k]);
    }
    if (o.half == 1u) o.g1 = mid;
    else o.g0 = mid;
  }
  return o;
}

// Steps 1 of the tile: halo cell table, LDS offsets and, with OWN, the own range.
// Returns the halo particle count.  Every thread of the team takes R halo cells; all
// their cell-table loads are issued, then those of `pre` (what the thread reads whatever
// the halo holds), before the first is waited for: a pass over a small scene is a chain
// of loads that miss the L2, about 0.8 us each.  With the block's own range from the
// tile marks, the key, list length and first chunk read here and the tile's number read
// beside the counts (us a step, before / now): 2K 230 / 220, 32K column 250 / 235, 1M
// column 1096 / 1080, 1M splash 1725 / 1631.
struct NoLoads {
  __device__ __forceinline__ void operator()() const {}
};
template <int BITS, class Team, bool OWN = true, class Pre = NoLoads>
__device__ __forceinline__ uint32_t tile_setup(const DevParams& P, uint32_t blk, const uint32_t* __restrict__ cs,
                                               const uint32_t* __restrict__ ce, TileShared<BITS>& sh,
                                               Pre pre = Pre(), uint32_t half = 0u) {
  using G = TileGeom<BITS>;
  constexpr uint32_t R = (G::NH + Team::kSize - 1u) / Team::kSize;
  static_assert(Team::kSize == 64u || R == 1u, "a workgroup team takes one halo cell per thread");
  const uint32_t tid = Team::tid(), lane = threadIdx.x & 63u;
  const uint32_t first = blk << BITS;
  const int ix0 = (int)compact10(first >> 2), iy0 = (int)compact10(first >> 1), iz0 = (int)compact10(first);
  // a half's halo: the layers around its own y (the other cells count as empty)
  const int y0 = half == 2u ? 2 : 0, y1 = half == 1u ? 4 : G::HY;
  uint32_t s0[R], e0[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t c = r * Team::kSize + tid;
    s0[r] = 0xFFFFFFFFu;
    e0[r] = 0u;
    if (c < (uint32_t)G::NH) {
      const int hx = (int)c / G::SX, hy = ((int)c / G::SY) % G::HY, hz = (int)c % G::HZ;
      const int cx = ix0 - 1 + hx, cy = iy0 - 1 + hy, cz = iz0 - 1 + hz;
      if (cx >= 0 && cy >= 0 && cz >= 0 && cx < (int)P.dims[0] && cy < (int)P.dims[1] && cz < (int)P.dims[2] &&
          hy >= y0 && hy < y1) {
        const uint32_t k = morton3((uint32_t)cx, (uint32_t)cy, (uint32_t)cz);
        s0[r] = cs[k];
        e0[r] = ce[k];
      }
    }
  }
  pre();
  if (tid == 0) {
    if (OWN) {
      sh.g0 = 0xFFFFFFFFu;
      sh.g1 = 0u;
    }
    sh.dmax = 0u;
  }
  // Offsets of the halo cells' corners from the block's first cell's.  In a batched
  // context both cells lie in the block's scene: the occupied cells of a scene keep
  // kernelWidthNeighbours + 1 empty cells from its slot's faces, so a halo cell
  // outside the slot is empty and its offset is never used.
  if (tid < 18u) {
    const uint32_t a = tid / 6u, k = tid % 6u;
    const uint32_t i0 = a == 0u ? (uint32_t)ix0 : (a == 1u ? (uint32_t)iy0 : (uint32_t)iz0);
    const float o = frame_origin(P, scene_of_key(P, first), (int)a);
    sh.off[a][k] = frame_corner(P, o, i0 + k - 1u) - frame_corner(P, o, i0);
  }
  if (OWN) Team::sync();
  uint32_t cnt[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t c = r * Team::kSize + tid;
    const bool some = s0[r] != 0xFFFFFFFFu;
    cnt[r] = some ? e0[r] - s0[r] : 0u;
    if (c < (uint32_t)G::NH) sh.gstart[c] = some ? s0[r] : 0u;
    if (OWN && some) {
      const int hx = (int)c / G::SX, hy = ((int)c / G::SY) % G::HY, hz = (int)c % G::HZ;
      if (hx >= 1 && hx <= G::EX && hy >= max(1, y0 + 1) && hy <= min((int)G::EY, y1 - 2) && hz >= 1 && hz <= G::EZ) {
        atomicMin(&sh.g0, s0[r]);
        atomicMax(&sh.g1, e0[r]);
      }
    }
  }
  if constexpr (Team::kSize == 64u) {
    uint32_t carry = 0;
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      uint32_t x = cnt[r];
#pragma unroll
      for (uint32_t o = 1; o < 64u; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
      }
      const uint32_t c = r * 64u + tid;
      if (c < (uint32_t)G::NH) sh.lstart[c] = carry + x - cnt[r];
      carry += __shfl(x, 63);
    }
    if (tid == 0) sh.lstart[G::NH] = carry;
  } else {
    const uint32_t wave = tid >> 6;
    uint32_t x = cnt[0];
#pragma unroll
    for (uint32_t o = 1; o < 64u; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    // the halo cells are held by the first waves (NH <= kTileThreads): only
    // those take part in the scan across waves
    static_assert(G::NH <= (int)kTileThreads, "halo cells fit the first kTileThreads threads");
    if (lane == 63u && wave < kTileThreads / 64u) sh.wsum[wave] = x;
    __syncthreads();
    if (tid < (uint32_t)G::NH) {
      uint32_t pre = 0;
      for (uint32_t w = 0; w < wave; ++w) pre += sh.wsum[w];
      sh.lstart[tid] = pre + x - cnt[0];
      if (tid == (uint32_t)G::NH - 1u) sh.lstart[G::NH] = pre + x;
    }
  }
  Team::sync();
  return sh.lstart[G::NH];
}

// A halo slot as one 16-byte LDS read, also where .w is not used.  Left to itself the
// compiler drops .w and reads 12 bytes, which takes the LDS 1.6 times as long (gfx950,
// clocks per wave read: a scan's addresses, 8 lanes each, 7.1 against 11.1; a list's,
// one per lane, 14.3 against 23.4).
__device__ __forceinline__ float4 slot_read(const float4* s_q, uint32_t j) {
  float4 v = s_q[j];
  asm("" : "+v"(v.x) : "v"(v.w));  // x is used, so w is read
  return v;
}

// Halo cell holding LDS slot i (largest c with lstart[c] <= i).
template <int BITS>
__device__ __forceinline__ int tile_cell_of(const TileShared<BITS>& sh, uint32_t i) {
  int lo = 0, hi = TileGeom<BITS>::NH;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (sh.lstart[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Offset of halo cell c's corner from the block's first cell's corner (c < 216:
// c / 6 and c / 36 by a multiplication, v_mul_hi_u32 is a quarter-rate instruction).
template <int BITS>
__device__ __forceinline__ float3 tile_offset(const TileShared<BITS>& sh, uint32_t c) {
  using G = TileGeom<BITS>;
  static_assert(G::HY == 6 && G::HZ == 6 && G::NH <= 216, "halo cell coordinates");
  const uint32_t xy = __umul24(c, 171u) >> 10, hx = __umul24(xy, 43u) >> 8;
  return make_float3(sh.off[0][hx], sh.off[1][xy - 6u * hx], sh.off[2][c - 6u * xy]);
}

// Own particle g: its halo cell and LDS slot.
template <int BITS>
__device__ __forceinline__ void tile_locate(const TileShared<BITS>& sh, uint32_t key, uint32_t g, int& h,
                                            uint32_t& slot) {
  using G = TileGeom<BITS>;
  // the key's low BITS bits are the cell's coordinates in the block, z, y, x from the LSB
  const uint32_t l = key & ((1u << BITS) - 1u);
  const int hx = (int)(((l >> 2) & 1u) | ((l >> 4) & 2u)) + 1;
  const int hy = (int)(((l >> 1) & 1u) | ((l >> 3) & 2u)) + 1;
  const int hz = (int)((l & 1u) | ((l >> 2) & 2u)) + 1;
  h = hx * G::SX + hy * G::SY + hz;
  slot = sh.lstart[h] + (g - sh.gstart[h]);
}

// Sorted index of the particle in LDS slot j.
template <int BITS>
__device__ __forceinline__ uint32_t tile_global(const TileShared<BITS>& sh, uint32_t j) {
  const int c = tile_cell_of<BITS>(sh, j);
  return sh.gstart[c] + (j - sh.lstart[c]);
}

// Walk the 27 stencil cells of halo cell h; body(j) for every LDS slot j != slot.
template <int BITS, class Body>
__device__ __forceinline__ uint32_t tile_stencil(const TileShared<BITS>& sh, int h, uint32_t slot, Body body) {
  using G = TileGeom<BITS>;
  uint32_t total = 0;
#pragma unroll 1
  for (int dx = -1; dx <= 1; ++dx) {
#pragma unroll 1
    for (int dy = -1; dy <= 1; ++dy) {
      const int hb = h + dx * G::SX + dy * G::SY;
      // the three z cells of a (dx, dy) column are consecutive halo cells: one range
      const uint32_t a = sh.lstart[hb - 1], b = sh.lstart[hb + 2];
      total += b - a;
      for (uint32_t j = a; j < b; ++j) {
        if (j != slot) body(j);
      }
    }
  }
  return total - 1u;  // neighbour count (self excluded)
}

// 27-cell count of a particle (to decide whether the cap binds).
template <int BITS>
__device__ __forceinline__ uint32_t tile_count(const TileShared<BITS>& sh, int h) {
  using G = TileGeom<BITS>;
  uint32_t total = 0;
#pragma unroll
  for (int dx = -1; dx <= 1; ++dx)
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy) {
      const int hb = h + dx * G::SX + dy * G::SY;
      total += sh.lstart[hb + 2] - sh.lstart[hb - 1];
    }
  return total - 1u;
}

// ---------------------------------------------------------------------------
// Block -> tile.  Workgroups are dispatched to the 8 XCDs of the MI355X round
// robin, and each XCD has its own L2.  Tile kernels deal the Morton-ordered tile
// list to the XCDs in chunks of kTileChunk consecutive tiles (chunk c to XCD
// c mod 8), so that the halos of neighbouring tiles (each particle is in ~4.5
// halos) are mostly fetched once per L2 while dense and sparse regions still
// spread evenly over the XCDs.  The grid is a multiple of kXcds * kTileChunk;
// the map from block to rank is a bijection on [0, grid).
constexpr uint32_t kXcds = 8;
static_assert(kTileGridMultiple % (kXcds * kTileChunk) == 0, "tile grid multiple");

// Work items of the tile passes: ranks below nl are large tiles; rank nl + q
// takes small tiles 4q .. 4q + 3, one per wave.  A workgroup takes the ranks
// tile_rank0() + k gridDim.x (k = 0, 1, ...): the grid may be smaller than the
// number of items, and any grid size covers them all.
struct TileItems {
  uint32_t nl, ns, end;  // large tiles, small tiles, ranks
};
__device__ __forceinline__ TileItems tile_items(const TileList& T) {
  const uint32_t nl = T.count[0], ns = T.count[1];
  return TileItems{nl, ns, nl + (ns + 3u) / 4u};
}
__device__ __forceinline__ uint32_t tile_rank0() {
  const uint32_t x = blockIdx.x % kXcds, k = blockIdx.x / kXcds;
  return ((k / kTileChunk) * kXcds + x) * kTileChunk + k % kTileChunk;
}
// The tile of rank r for this thread's team: 1 = large tile `blk` for the whole
// workgroup, 2 = small tile `blk` for this wave, 0 = none (for this wave, none at
// any later rank either).
__device__ __forceinline__ int tile_pick(const TileList& T, const TileItems& it, uint32_t r, uint32_t& blk) {
  // loaded with the counts, not after them (the list has T.cap entries)
  const uint32_t large = T.large[min(r, T.cap - 1u)];
  if (r < it.nl) {
    blk = large;
    return 1;
  }
  if (r >= it.end) return 0;
  const uint32_t i = (r - it.nl) * (kTileThreads / 64u) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i < it.ns) {
    blk = T.small[i];
    return 2;
  }
  return 0;
}

// Halo particles held in LDS; the same for the producing and the consuming pass
// so that a slot names the same particle in both.
template <int BITS>
struct TileCap;
// The capacity decides how many workgroups a CU holds: with 1528 slots (and small tiles'
// 312) a lambda pass has 26 KB and 6 of them, as many as its 73 to 79 VGPRs allow, an omega
// pass (a slot's global index beside it) 32 KB and 5, at 1920 slots 5 and 4.  us a step at
// 1920 / 1352 slots, when it was lowered: 1M column 1060 / 964, 1M splash 1438 / 1285, 16M
// column 14700 / 13650, 64 uneven scenes 7360 / 7110; at 1352 / 1528 / 1560: 1M column 912 /
// 912 / 927, 1M splash 1177 / 1190 / 1225, 16M column 12395 / 12392 / 12650, 64 uneven
// scenes 6930 / 7030 / 7110.  A block with more in its halo (1152 at rest density) is two
// items, its halves.  1528 slots hold a half (96 cells of the 144) of nearly every halo of up
// to 1920 within the neighbour cap; with 1352, layers of 9, 20, 20 and 9 a cell went particle
// by particle from global memory (401K of them 2830 us a step, as halves in the LDS 2193, as
// whole blocks of 1920 slots 2331).
template <>
struct TileCap<5> {
  static constexpr int value = 1528;  // 2x4x4 blocks: 144 halo cells, ~1150 particles at rest density
  // a small tile's halo (one wave, a quarter of the LDS; 64 uneven scenes 6390 us at 272, 6350)
  static constexpr int small = 312;
  static constexpr int adjoint = 1920;  // of the reverse passes' list builders
};
template <>
struct TileCap<6> {
  static constexpr int value = 2880;  // 4x4x4 blocks: 216 halo cells, ~1730 at rest density
  static constexpr int small = 630;
  static constexpr int adjoint = 2880;
};

// ---------------------------------------------------------------------------
// Tile-list compaction: a two-kernel stream compaction of the occupied blocks
// into the large and the small list.  Per-thread and per-block counts are
// packed as large | small << 16 (a block of the compaction covers 4096 flags).
__device__ __forceinline__ uint32_t tile_class(uint32_t b, uint32_t nflags, const uint32_t* __restrict__ start,
                                               const uint32_t* __restrict__ end, uint32_t small_max) {
  if (b >= nflags) return 0u;
  const uint32_t s = start[b];
  if (s == 0u) return 0u;
  if (!(s & kTileCrowded) && end[b] - tile_begin(s) <= small_max) return 0x10000u;
  return s & kTileSplit ? 2u : 1u;
}

// Marks the occupied blocks by their halos and counts the items of every 4096 flags: a
// block of at most small_max particles whose halo is more than a small tile holds is
// large (kTileCrowded; as a small one every pass took it particle by particle from global
// memory: 1M splash with small tiles of up to 64, 1862 us, with the marks 1438; also one of a
// few particles beside a crowd, whose 27 cells of each one lane would walk: with blocks of up
// to 8 left small, steps 11 to 20 of a 262K dam break took 663 us each, with none 521; see
// small_sure), and a
// large one whose halo is more than a tile holds is two items (kTileSplit).  A wave takes F flags, a lane each, and counts
// the halos of those that need it four at a time, kHaloLanes lanes a block, all of a
// lane's cells in flight at once.
constexpr uint32_t kHaloLanes = 16;
// Flags of a wave.  Where the blocks fill few waves, four blocks a wave are one chain of two
// loads (7 us at 32K particles, 17 at 1M); with more flags the chain
// repeats, but the waves that only sweep empty blocks, of a box far larger than its fluid,
// are fewer.  us a step at 4 / 16 / 64 flags: 2K 167 / 173 / 173, 211K splash (45K flags) 472
// / 485 / 509, 1M column (41K) 949 / 951 / 988, 16M column (0.3M) 13557 / 13370 / 13368, 1.2M
// in a 300-cell box (2.2M) 1818 / 1759 / 1795, 5K in a 1024^3-cell box (34M) 3222 / 2502 / 2318.
static uint32_t classify_flags(uint32_t nflags) {
  return nflags <= (1u << 17) ? 4u : nflags <= (1u << 22) ? 16u : 64u;
}
template <int BITS, uint32_t F>
__global__ __launch_bounds__(256) void k_tile_classify(DevParams P, uint32_t nflags, uint32_t* __restrict__ start,
                                                       const uint32_t* __restrict__ end, uint32_t small_max,
                                                       const uint32_t* __restrict__ cs,
                                                       const uint32_t* __restrict__ ce, uint32_t* __restrict__ bcount) {
  using G = TileGeom<BITS>;
  static_assert(F <= 64u && kTileCompactChunk % F == 0u, "a wave's flags lie in one chunk of the compaction");
  const uint32_t lane = threadIdx.x & 63u, l = lane % kHaloLanes;
  const uint32_t base = (blockIdx.x * (blockDim.x / 64u) + (threadIdx.x >> 6)) * F;
  const uint32_t s = lane < F && base + lane < nflags ? start[base + lane] : 0u;
  const uint32_t own = s ? end[base + lane] - tile_begin(s) : 0u;
  uint32_t mark = 0u;
  for (uint64_t todo = __ballot(own > min(small_sure(P.n), small_max)); todo;) {
    // the next four blocks, one for each group of lanes
    uint32_t k = 64u;
#pragma unroll
    for (uint32_t i = 0; i < 64u / kHaloLanes; ++i)
      if (todo) {
        if (lane / kHaloLanes == i) k = (uint32_t)__builtin_ctzll(todo);
        todo &= todo - 1u;
      }
    const uint32_t first = (base + k) << BITS;
    uint32_t halo = 0u;
    if (k < 64u) {
      const int ix0 = (int)compact10(first >> 2), iy0 = (int)compact10(first >> 1), iz0 = (int)compact10(first);
#pragma unroll
      for (uint32_t r = 0; r < ((uint32_t)G::NH + kHaloLanes - 1u) / kHaloLanes; ++r) {
        const uint32_t c = r * kHaloLanes + l;
        if (c >= (uint32_t)G::NH) break;
        const int cx = ix0 - 1 + (int)c / G::SX, cy = iy0 - 1 + ((int)c / G::SY) % G::HY, cz = iz0 - 1 + (int)c % G::HZ;
        if (cx >= 0 && cy >= 0 && cz >= 0 && cx < (int)P.dims[0] && cy < (int)P.dims[1] && cz < (int)P.dims[2]) {
          const uint32_t m = morton3((uint32_t)cx, (uint32_t)cy, (uint32_t)cz);
          const uint32_t a = cs[m], e = ce[m];
          halo += a != 0xFFFFFFFFu ? e - a : 0u;
        }
      }
    }
#pragma unroll
    for (uint32_t o = kHaloLanes / 2u; o; o >>= 1) halo += (uint32_t)__shfl_xor((int)halo, (int)o, (int)kHaloLanes);
    // to the block's own lane
#pragma unroll
    for (uint32_t i = 0; i < 64u / kHaloLanes; ++i) {
      const uint32_t h = (uint32_t)__shfl((int)halo, (int)(i * kHaloLanes)), at = (uint32_t)__shfl((int)k, (int)(i * kHaloLanes));
      if (at != lane) continue;
      if (own <= small_max && h > (uint32_t)TileCap<BITS>::small) mark = kTileCrowded;
      if (BITS == 5 && (own > small_max || mark) && h > (uint32_t)TileCap<BITS>::value) mark |= kTileSplit;
    }
  }
  if (mark) start[base + lane] = s | mark;
  uint32_t c = 0u;
  if (s) c = !(mark & kTileCrowded) && own <= small_max ? 0x10000u : mark & kTileSplit ? 2u : 1u;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) c += (uint32_t)__shfl_xor((int)c, o);
  if (lane == 0u && c) atomicAdd(&bcount[base / kTileCompactChunk], c);
}

__global__ __launch_bounds__(1024) void k_tile_emit(uint32_t nflags, const uint32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ end, uint32_t small_max,
                                                    const uint32_t* __restrict__ bcount, uint32_t* __restrict__ large,
                                                    uint32_t* __restrict__ small, uint32_t* __restrict__ count) {
  __shared__ uint32_t s_w[16][2];
  __shared__ uint32_t s_off[2];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  // offsets of this block: the counts of the blocks before it (unpacked: the
  // totals may exceed 16 bits)
  uint32_t ol = 0, os = 0;
  for (uint32_t i = tid; i < blockIdx.x; i += 1024u) {
    const uint32_t c = bcount[i];
    ol += c & 0xFFFFu;
    os += c >> 16;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    ol += __shfl_xor(ol, d);
    os += __shfl_xor(os, d);
  }
  if (lane == 0) {
    s_w[wave][0] = ol;
    s_w[wave][1] = os;
  }
  __syncthreads();
  if (tid == 0) {
    uint32_t tl = 0, ts = 0;
    for (int w = 0; w < 16; ++w) {
      tl += s_w[w][0];
      ts += s_w[w][1];
    }
    s_off[0] = tl;
    s_off[1] = ts;
  }
  __syncthreads();
  // this thread's blocks and their exclusive scan over the compaction block (packed)
  const uint32_t base = blockIdx.x * kTileCompactChunk + tid * 4u;
  uint32_t f[4], c = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    f[k] = tile_class(base + k, nflags, start, end, small_max);
    c += f[k];
  }
  uint32_t x = c;
#pragma unroll
  for (uint32_t d = 1; d < 64u; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  __syncthreads();
  if (lane == 63u) s_w[wave][0] = x;
  __syncthreads();
  uint32_t pre = 0;
  for (uint32_t w = 0; w < wave; ++w) pre += s_w[w][0];
  const uint32_t ex = pre + x - c;
  uint32_t pl = s_off[0] + (ex & 0xFFFFu), ps = s_off[1] + (ex >> 16);
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    if (f[k] == 1u) {
      large[pl++] = base + k;
    } else if (f[k] == 2u) {
      large[pl++] = (base + k) | (1u << 30);
      large[pl++] = (base + k) | (2u << 30);
    }
    if (f[k] > 2u) small[ps++] = base + k;
  }
  if (blockIdx.x == gridDim.x - 1 && tid == 1023u) {
    const uint32_t tot = pre + x;
    count[0] = s_off[0] + (tot & 0xFFFFu);
    count[1] = s_off[1] + (tot >> 16);
  }
}

hipError_t launch_tile_compact(hipStream_t st, int bits, const DevParams& P, const StepBuffers& B, uint32_t nflags,
                               uint32_t* start, const uint32_t* end, uint32_t small_max, uint32_t* bcount, uint32_t* large, uint32_t* small,
                               uint32_t* count) {
  if (small_max > kTileSmall) return hipErrorInvalidValue;  // a small tile is one wave, one particle per lane
  const uint32_t F = classify_flags(nflags);
  const dim3 g((nflags + 4u * F - 1u) / (4u * F)), t(256);
#define PBD_CLASSIFY(F_)                                                                                          \
  if (bits == 5)                                                                                                  \
    hipLaunchKernelGGL((k_tile_classify<5, F_>), g, t, 0, st, P, nflags, start, end, small_max, B.cstart, B.cend, \
                       bcount);                                                                                   \
  else                                                                                                            \
    hipLaunchKernelGGL((k_tile_classify<6, F_>), g, t, 0, st, P, nflags, start, end, small_max, B.cstart, B.cend, \
                       bcount)
  if (F == 4u) {
    PBD_CLASSIFY(4u);
  } else if (F == 16u) {
    PBD_CLASSIFY(16u);
  } else {
    PBD_CLASSIFY(64u);
  }
#undef PBD_CLASSIFY
  const uint32_t blocks = (nflags + kTileCompactChunk - 1u) / kTileCompactChunk;
  hipLaunchKernelGGL(k_tile_emit, dim3(blocks), dim3(1024), 0, st, nflags, start, end, small_max, bcount, large, small,
                     count);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Neighbour lists.
//
// The lambda pass scans the 27-cell stencil of each particle with a bare
// distance test, keeps the LDS slots of the pairs within R = max(h_poly,
// h_spiky, diameter) (padded for rounding) in a per-thread LDS list, evaluates
// the pass over that list, and writes it out.  The delta-p pass of the same
// Jacobi iteration sees the same positions, the same cells and so the same LDS
// layout: it reads the list instead of scanning.  The omega pass and the final
// (vorticity + XSPH) pass form the same pair.  Pairs outside R contribute
// exactly zero to every term and the list keeps the scan order, so the sums
// are the scan's sums.
//
// A list is padded to a multiple of 8 entries with the sentinel slot CAP (a halo
// entry placed far away, for which every pair term is zero) and stored as
// chunks of 8 u16 slots, chunk-major (NL[c * cap + g]) so that a wave's loads
// of chunk c are contiguous.  A particle with more than kNlMax pairs in range,
// or whose 27-cell count exceeds the neighbour cap, is marked kNlInvalid: its
// passes scan.
constexpr uint32_t kNlMax = 8 * kNlChunks;
constexpr uint16_t kNlInvalid = 0xFFFFu;
constexpr float kFar = 1.0e15f;  // sentinel coordinate: r^2 ~ 3e30 stays finite

struct NeighbourList {
  uint4* nl;      // [kNlChunks][cap] chunks of 8 slots
  uint16_t* cnt;  // [cap] padded entry count, or kNlInvalid
  uint32_t cap;
  unsigned long long* stats;  // PBD_COUNTER_LIST_*
};

// Scan unroll: candidates tested per group in nl_column.
#ifndef PBD_SCAN_UNROLL
#define PBD_SCAN_UNROLL 8
#endif
constexpr uint32_t kScanUnroll = PBD_SCAN_UNROLL;

// LDS of one team: cell table, the halo (CAP entries, the sentinel at CAP and
// kScanUnroll - 1 more that an unrolled scan may read past a cell range; their
// hits are masked off) and, with GI, the global index of every slot.
template <int BITS, int CAP, bool GI>
struct TileRegion {
  TileShared<BITS> sh;
  float4 q[CAP + kScanUnroll];
  uint32_t gi[GI ? CAP + 1 : 1];
};
// A workgroup's LDS: one large tile, or four small tiles in the same bytes.
template <int BITS, bool GI>
union TileLds {
  TileRegion<BITS, TileCap<BITS>::value, GI> big;
  TileRegion<BITS, TileCap<BITS>::small, GI> small[kTileThreads / 64u];
};
constexpr uint32_t kLdsBytes = 160u * 1024u;  // of a CU
static_assert(6 * sizeof(TileLds<5, false>) <= kLdsBytes && 5 * sizeof(TileLds<5, true>) <= kLdsBytes,
              "workgroups per CU of the 2^5-cell passes");
static_assert(3 * sizeof(TileLds<6, false>) <= kLdsBytes && 2 * sizeof(TileLds<6, true>) <= kLdsBytes,
              "workgroups per CU of the 2^6-cell passes");

// Copy the block's halo into LDS (block-local coordinates; .w = payload(i)),
// with s_gi (when not null) the global index of every slot, and place the
// sentinel at slot CAP (s_gi[CAP] = `any`, a valid particle whose pair terms
// the sentinel's position zeroes).  With dk, sh.dmax receives the largest
// dk[i] - dm[i] (dm null: dk[i]) over the halo's particles i, the bound on their
// displacement between two delta-p passes (float bits: the bounds are >= 0, or
// NaN, which exceeds every finite bound).
//
// A workgroup team deals the halo cells to groups of 8 lanes, so a slot's cell is
// known without a search and its offset is looked up once per 8 slots; the first
// 16 particles of every cell of a group are in flight at once (1M dam break, delta-p:
// 70 -> 65 us; 32K: 13.2 -> 9.9 us, with the smaller kernels of TileRest).  A wave team's
// tile is sparse (a few particles in a cell): there a lane takes slots, kLoadUnroll
// in flight, and finds each slot's cell by bisection (the index of a slot past the
// end is clamped to the last slot and its result dropped).
template <int BITS, int CAP, class Team, class Payload>
__device__ __forceinline__ void tile_load(const DevParams& P, TileShared<BITS>& sh, uint32_t total,
                                          const float4* __restrict__ Q, float4* s_q, uint32_t* s_gi, uint32_t any,
                                          Payload payload, const float* __restrict__ dk = nullptr,
                                          const float* __restrict__ dm = nullptr) {
  const uint32_t tid = Team::tid();
  uint32_t dmax = 0u;
  const auto bound = [&](uint32_t gi) { return dk ? __float_as_uint(dk[gi] - (dm ? dm[gi] : 0.0f)) : 0u; };
  if constexpr (Team::kSize == 64u) {
    constexpr uint32_t U = Team::kLoadUnroll;
    for (uint32_t i0 = tid; i0 < total; i0 += U * Team::kSize) {
      int c[U];
      uint32_t gi[U], d[U];
      float4 q[U];
      float w[U];
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint32_t i = min(i0 + u * Team::kSize, total - 1u);
        c[u] = tile_cell_of<BITS>(sh, i);
        gi[u] = sh.gstart[c[u]] + (i - sh.lstart[c[u]]);
        q[u] = Q[gi[u]];
        w[u] = payload(gi[u]);
        d[u] = bound(gi[u]);
      }
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint32_t i = i0 + u * Team::kSize;
        if (i < total) {
          const float3 o = tile_offset<BITS>(sh, (uint32_t)c[u]);
          s_q[i] = make_float4(q[u].x + o.x, q[u].y + o.y, q[u].z + o.z, w[u]);
          if (s_gi) s_gi[i] = gi[u];
        }
      }
      // a clamped slot repeats the last one: its bound may be taken again
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) dmax = max(dmax, d[u]);
    }
  } else {
    constexpr uint32_t NG = Team::kSize / 8u, NH = TileGeom<BITS>::NH, R = (NH + NG - 1u) / NG;
    const uint32_t l8 = tid & 7u;
    uint32_t cell[R], ls[R], n[R], gs[R];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      const uint32_t c = (tid >> 3) + r * NG;
      cell[r] = min(c, NH - 1u);
      ls[r] = sh.lstart[cell[r]];
      n[r] = c < NH ? sh.lstart[cell[r] + 1u] - ls[r] : 0u;
      gs[r] = sh.gstart[cell[r]];
    }
    float4 q[R][2];
    float w[R][2];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
#pragma unroll
      for (uint32_t v = 0; v < 2u; ++v) {
        const uint32_t j = l8 + 8u * v;
        if (j < n[r]) {
          q[r][v] = Q[gs[r] + j];
          w[r][v] = payload(gs[r] + j);
          dmax = max(dmax, bound(gs[r] + j));
        }
      }
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      const float3 o = tile_offset<BITS>(sh, cell[r]);
#pragma unroll
      for (uint32_t v = 0; v < 2u; ++v) {
        const uint32_t j = l8 + 8u * v;
        if (j < n[r]) {
          s_q[ls[r] + j] = make_float4(q[r][v].x + o.x, q[r][v].y + o.y, q[r][v].z + o.z, w[r][v]);
          if (s_gi) s_gi[ls[r] + j] = gs[r] + j;
        }
      }
      for (uint32_t j = l8 + 16u; j < n[r]; j += 8u) {
        const uint32_t gi = gs[r] + j;
        const float4 p = Q[gi];
        s_q[ls[r] + j] = make_float4(p.x + o.x, p.y + o.y, p.z + o.z, payload(gi));
        if (s_gi) s_gi[ls[r] + j] = gi;
        dmax = max(dmax, bound(gi));
      }
    }
  }
  if (dk) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) dmax = max(dmax, (uint32_t)__shfl_xor((int)dmax, o));
    if ((threadIdx.x & 63u) == 0u) atomicMax(&sh.dmax, dmax);
  }
  if (tid < kScanUnroll) s_q[CAP + tid] = make_float4(kFar, kFar, kFar, 0.0f);
  if (s_gi && tid == 0) s_gi[CAP] = any;
}

// Lists carried from pass to pass (StepBuffers::DISP, BUILT, MODE): `pass`
// delta-p passes of the substep are done (a lambda or omega pass), or this is
// delta-p pass `pass` (1-based); disp null: no carry.
struct Carry {
  float* disp;
  uint16_t* built;
  uint16_t* mode;
  uint32_t stride;
  uint32_t pass;
  __device__ __forceinline__ float* bounds(uint32_t p) const {
    return p ? disp + (size_t)(p - 1u) * stride : nullptr;  // after p delta-p passes (p = 0: all zero)
  }
};

// Particles of a tile left to the per-particle global-memory path: thread `tid` of the
// team takes the particles g, g + stride, ... < end whose bit of `bits` is set (bit k:
// the k-th of them; all: every one, for a block whose halo exceeds the tile capacity).
// A tile pass returns them and the kernel walks them once for both teams, so that the
// global path is in a kernel once instead of at every place that takes it (four copies
// made up half of the 50 to 110 KB kernels).
struct TileRest {
  uint32_t g = 0u, end = 0u, stride = 1u, bits = 0u;
  bool all = false;
  template <class Body>
  __device__ __forceinline__ void visit(Body body) const {
    if (!all && bits == 0u) return;
    uint32_t k = 0u;
    for (uint32_t i = g; i < end; i += stride, ++k)
      if (all || ((bits >> k) & 1u)) body(i);
  }
};
// A tile within the capacity has at most 12 rounds (TileCap / team size).
template <class Team>
__device__ __forceinline__ TileRest tile_rest(uint32_t g0, uint32_t g1, bool all) {
  TileRest r;
  r.g = g0 + Team::tid();
  r.end = g1;
  r.stride = Team::kSize;
  r.all = all;
  return r;
}

// Whether a tile keeps the lists it built after an earlier delta-p pass (the
// halo bound of tile_load against P.reuse_max); read after the team barrier
// that follows tile_load.
template <int BITS>
__device__ __forceinline__ bool tile_keeps_lists(const DevParams& P, const TileShared<BITS>& sh) {
  return __uint_as_float(sh.dmax) <= P.reuse_max;  // false for a NaN bound
}

// Delta-p pass C.pass: the particle's bound after it, the one after the
// previous pass plus the length of its move (cell frame).
__device__ __forceinline__ void track_move(const Carry& C, uint32_t g, float4 from, float4 to) {
  if (!C.disp) return;
  const float dx = to.x - from.x, dy = to.y - from.y, dz = to.z - from.z;
  const float* prev = C.bounds(C.pass - 1u);
  C.bounds(C.pass)[g] = (prev ? prev[g] : 0.0f) + sqrtf(dx * dx + dy * dy + dz * dz);
}

// Visit the global list of particle g (n = padded length) in order; w: its first chunk.
template <class Body>
__device__ __forceinline__ void nl_visit(const NeighbourList& L, uint32_t g, uint32_t n, uint4 w, Body body) {
  const uint4* p = L.nl + g;
  const uint32_t nc = n >> 3;
  if (nc == 0) return;
  for (uint32_t c = 1; c <= nc; ++c) {
    // (as a conditional expression this is a flat load from a selected address, with w in
    // scratch, and the next read of the LDS waits for it)
    uint4 nx = w;
    if (c < nc) nx = p[(size_t)c * L.cap];
    body(w.x & 0xFFFFu);
    body(w.x >> 16);
    body(w.y & 0xFFFFu);
    body(w.y >> 16);
    body(w.z & 0xFFFFu);
    body(w.z >> 16);
    body(w.w & 0xFFFFu);
    body(w.w >> 16);
    w = nx;
  }
}

// In-range bits of slots a .. a + len - 1 (len <= 32): bit k is set when slot a + k
// is within the list radius.  The test is the sign of r^2 - r2max, shifted into the
// mask by one v_alignbit: 7 VALU instructions a candidate (compare, select, shift and
// or take 11).  A building lambda pass is bound by VALU issue (86 % busy) and, half as
// much, by the LDS; 1M dam break: 152 -> 122 us, with the 16-byte reads of slot_read.  Unrolled by kScanUnroll: a group may read up to kScanUnroll - 1 slots
// past the range (still inside the LDS array); their bits are masked off.  A position
// that is not a number is +NaN (canonical_nan), whose sign says out of range; the
// caller drops the mask of a particle that is not finite itself (inf - inf is -NaN).
// (The language leaves a NaN's sign open: that the hardware's instructions keep it through
// the subtraction and the fused additions is what the tests of NaN neighbours hold.)
template <uint32_t U = kScanUnroll>
__device__ __forceinline__ uint32_t nl_mask(const float4* s_q, uint32_t a, uint32_t len, float qx, float qy, float qz,
                                            float r2max) {
  static_assert(U <= kScanUnroll && 32u % U == 0u, "whole groups fill a mask");
  uint32_t m = 0u, k = 0u;
  do {
    float4 c[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) c[u] = slot_read(s_q, a + k + u);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const float rx = c[u].x - qx, ry = c[u].y - qy, rz = c[u].z - qz;
      const float d = fmaf(rz, rz, fmaf(ry, ry, fmaf(rx, rx, -r2max)));
      m = __builtin_amdgcn_alignbit(m, __float_as_uint(d), 31u);  // m << 1 | sign of d
    }
    k += U;
  } while (k < len);
  // slot a + j is bit k - 1 - j now
  return (__brev(m) >> (32u - k)) & (0xFFFFFFFFu >> (32u - len));
}

// Appends slots to 8-entry chunks held in four registers and stores each full
// chunk to the global list (chunk-major).
struct ChunkWriter {
  uint32_t w0 = 0u, w1 = 0u, w2 = 0u, w3 = 0u, n = 0u;
  uint4* p;        // the particle's next chunk
  uint32_t stride;  // chunks from one to the next
  __device__ __forceinline__ ChunkWriter(const NeighbourList& L, uint32_t g) : p(L.nl + g), stride(L.cap) {}
  __device__ __forceinline__ void store() {
    *p = make_uint4(w0, w1, w2, w3);
    p += stride;
  }
  __device__ __forceinline__ void push(uint32_t slot) {
    // shift the chunk down one entry; the new slot enters at the top
    w0 = __builtin_amdgcn_alignbit(w1, w0, 16u);
    w1 = __builtin_amdgcn_alignbit(w2, w1, 16u);
    w2 = __builtin_amdgcn_alignbit(w3, w2, 16u);
    w3 = __builtin_amdgcn_alignbit(slot, w3, 16u);
    if ((++n & 7u) == 0u) store();
  }
  // Fills the last chunk up with `pad`; returns the padded length.
  __device__ __forceinline__ uint32_t finish(uint32_t pad) {
    const uint32_t r = (0u - n) & 7u;  // entries to add
    if (r) {
      const uint32_t pp = pad | (pad << 16);
      if (r & 4u) {
        w0 = w2;
        w1 = w3;
        w2 = w3 = pp;
      }
      if (r & 2u) {
        w0 = w1;
        w1 = w2;
        w2 = w3;
        w3 = pp;
      }
      if (r & 1u) {
        w0 = __builtin_amdgcn_alignbit(w1, w0, 16u);
        w1 = __builtin_amdgcn_alignbit(w2, w1, 16u);
        w2 = __builtin_amdgcn_alignbit(w3, w2, 16u);
        w3 = __builtin_amdgcn_alignbit(pp, w3, 16u);
      }
      store();
    }
    return n + r;
  }
};

// A list entry is an LDS slot (< 2^15); with phases, bit 15 marks a solid
// neighbour (the producing pass holds the solid flag in the slot's .w).
constexpr uint32_t kNlSolid = 0x8000u;

// Build the list of the particle at `slot` (halo cell h), the pairs within
// sqrt(r2) in stencil-column then slot order, into the global list, padded to a
// multiple of 8 with the sentinel slot CAP.  Each column is scanned 32 slots at
// a time and its in-range slots are appended at once; the loop over the columns
// is not unrolled (its nine copies, in both teams, made kernels of 70 to 110 KB,
// past the instruction cache).  Returns the padded length, or kNlInvalid when more
// than kNlMax pairs are in range (checked before a segment is appended, so no more
// than kNlMax entries are ever written).
template <int BITS, int CAP, bool PH>
__device__ __forceinline__ uint32_t nl_build(const DevParams& P, const NeighbourList& L, uint32_t g,
                                             const TileShared<BITS>& sh, const float4* s_q, int h, uint32_t slot,
                                             float4 qi, float r2) {
  using G = TileGeom<BITS>;
  const uint32_t valid = fabsf(qi.x) + fabsf(qi.y) + fabsf(qi.z) < __builtin_inff() ? 0xFFFFFFFFu : 0u;
  uint32_t n = 0;
  ChunkWriter cw(L, g);
#pragma unroll 1
  for (int dx = -1; dx <= 1; ++dx) {
#pragma unroll 1
    for (int dy = -1; dy <= 1; ++dy) {
      const int hb = h + dx * G::SX + dy * G::SY;
      const uint32_t a = sh.lstart[hb - 1], b = sh.lstart[hb + 2];
      for (uint32_t s = a; s < b; s += 32u) {
        uint32_t m = nl_mask(s_q, s, min(b - s, 32u), qi.x, qi.y, qi.z, r2) & valid;
        if (slot - s < 32u) m &= ~(1u << (slot - s));  // not the particle itself
        n += __builtin_popcount(m);
        if (n > kNlMax) return kNlInvalid;
        while (m) {
          const uint32_t k = __builtin_ctz(m);
          m &= m - 1u;
          uint32_t e = s + k;
          if (PH && s_q[e].w != 0.0f) e |= kNlSolid;
          cw.push(e);
        }
      }
    }
  }
  return cw.finish((uint32_t)CAP);
}

// lambda over one tile (team: workgroup or wave, CAP: its LDS capacity),
// building the neighbour lists, or, with a carry (a pass after the substep's
// first, in a tile that carries its lists this substep), keeping those the
// tile built after an earlier delta-p pass when its halo has moved less than
// P.reuse_max since.  A carrying tile builds with the skin (P.tile_r2).
template <int BITS, bool FIRST, bool PH, class Team, int CAP>
__device__ __forceinline__ TileRest lambda_tile(const DevParams& P, const TileList& T, uint32_t item, const NeighbourList& L,
                                            const float4* __restrict__ Q, const uint32_t* __restrict__ keys,
                                            const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                                            float* __restrict__ lam, float* __restrict__ dens,
                                            uint32_t* __restrict__ ncnt, uint32_t* __restrict__ ccnt,
                                            const Carry& C, TileShared<BITS>& sh, float4* s_q) {
  constexpr int VAR = PBD_KERNEL_TEXTBOOK;
  const uint32_t tid = Team::tid();
  const TileOwn own = tile_own<BITS>(P, T, item, cs);
  const uint32_t blk = own.blk, g0 = own.g0, g1 = own.g1;
  uint32_t key = 0u;  // of the thread's next particle
  const uint32_t total = tile_setup<BITS, Team, false>(P, blk, cs, ce, sh, [&]() __attribute__((always_inline)) {
    if (g0 + tid < g1) key = keys[g0 + tid];
  }, own.half);
  TileRest rest = tile_rest<Team>(g0, g1, total > (uint32_t)CAP);
  if (total > (uint32_t)CAP) {
    for (uint32_t g = g0 + tid; g < g1; g += Team::kSize) L.cnt[g] = kNlInvalid;
    if (tid == 0) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_BLOCK], (unsigned long long)(g1 - g0));
    return rest;
  }
  // the first pass: whether the tile carries its lists this substep; a later
  // one: the delta-p passes before the tile's lists were built (kNoCarry: none)
  const uint32_t m = C.disp ? (FIRST ? (C.mode[own.carried()] ? 0u : kNoCarry) : C.built[own.carried()]) : kNoCarry;
  const bool carry = !FIRST && m != kNoCarry;
  const float r2 = m != kNoCarry ? P.tile_r2 : P.list_r2;
  // .w: 1 for a solid particle (PH), else 0
  tile_load<BITS, CAP, Team>(P, sh, total, Q, s_q, nullptr, 0u,
                             [&](uint32_t gi) { return PH && P.phs[gi] ? 1.0f : 0.0f; },
                             carry ? C.bounds(C.pass) : nullptr, carry ? C.bounds(m) : nullptr);
  Team::sync();
  const bool keep = carry && tile_keeps_lists<BITS>(P, sh);
  if (tid == 0 && C.disp) {
    if (FIRST) C.built[own.carried()] = (uint16_t)m;  // 0: built now, with the skin
    else if (carry && !keep) C.built[own.carried()] = (uint16_t)C.pass;  // rebuilt now
    if (carry) atomicAdd(&L.stats[keep ? PBD_COUNTER_LIST_CARRIES : PBD_COUNTER_LIST_RESCANS],
                         (unsigned long long)(g1 - g0));
  }
  uint32_t round = 0u;
  for (uint32_t g = g0 + tid; g < g1; g += Team::kSize, ++round) {
    if (round) key = keys[g];
    int h;
    uint32_t slot;
    tile_locate<BITS>(sh, key, g, h, slot);
    uint32_t cnt = 0u, n = kNlInvalid;
    if (keep) {
      // a kept list, or none: a particle over the cap takes the global path as
      // when the list was built, one with a long list scans the stencil
      n = L.cnt[g];
      if (n == kNlInvalid && tile_count<BITS>(sh, h) > P.cap) {
        rest.bits |= 1u << round;
        continue;
      }
    } else {
      cnt = tile_count<BITS>(sh, h);
      if (cnt > P.cap) {
        rest.bits |= 1u << round;
        L.cnt[g] = kNlInvalid;
        atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_CAP], 1ull);
        continue;
      }
    }
    const float4 qi = s_q[slot];
    LambdaAcc a;
    const auto pair = [&](uint32_t j) __attribute__((always_inline)) {
      if (PH && (j & kNlSolid)) return;  // a fluid particle counts fluid neighbours only
      const float4 qj = slot_read(s_q, j);
      if (PH && qj.w != 0.0f) return;
      lambda_pair<VAR, PH>(P, qi.x - qj.x, qi.y - qj.y, qi.z - qj.z, a);
    };
    if (!keep) {
      n = nl_build<BITS, CAP, PH>(P, L, g, sh, s_q, h, slot, qi, r2);
      L.cnt[g] = (uint16_t)n;
      if (n == kNlInvalid) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_LONG], 1ull);
    }
    // a solid particle has no density constraint: after the first pass (which
    // writes its density) it needs its list, for delta-p, but not its pairs here
    if (PH && !FIRST && qi.w != 0.0f) {
      lam[g] = 0.0f;
      continue;
    }
    if (n != kNlInvalid) nl_visit(L, g, n, L.nl[g], pair);
    else tile_stencil<BITS>(sh, h, slot, pair);
    float W;
    const float l = lambda_finish<VAR>(P, a, W, scene_eps(P, key));
    lam[g] = PH && qi.w != 0.0f ? 0.0f : l;
    if (FIRST) {
      dens[g] = W;
      ncnt[g] = cnt;
      ccnt[g] = cnt;
    }
  }
  return rest;
}

template <int BITS, bool FIRST, bool STRIDE, bool PH>
__global__ __launch_bounds__(kTileThreads) void k_tile_lambda(DevParams P, TileList T, NeighbourList L,
                                                              const float4* __restrict__ Q,
                                                              const uint32_t* __restrict__ keys,
                                                              const uint32_t* __restrict__ cs,
                                                              const uint32_t* __restrict__ ce, float* __restrict__ lam,
                                                              float* __restrict__ dens, uint32_t* __restrict__ ncnt,
                                                              uint32_t* __restrict__ ccnt, Carry C) {
  __shared__ TileLds<BITS, false> lds;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&L.stats[PBD_COUNTER_LIST_BUILDS], 1ull);
  const TileItems it = tile_items(T);
  // STRIDE: every gridDim-th rank from tile_rank0(); otherwise the grid covers
  // the ranks and a workgroup takes one
  for (uint32_t r = tile_rank0();; r += gridDim.x) {
    uint32_t blk;
    const int mode = tile_pick(T, it, r, blk);
    if (mode == 0) break;
    TileRest rest;
    if (mode == 1) {
      rest = lambda_tile<BITS, FIRST, PH, TeamBlockN<kTileThreads, STRIDE>, TileCap<BITS>::value>(P, T, blk, L, Q, keys, cs, ce, lam, dens, ncnt,
                                                                       ccnt, C, lds.big.sh, lds.big.q);
    } else {
      auto& reg = lds.small[threadIdx.x >> 6];
      rest = lambda_tile<BITS, FIRST, PH, TeamWaveT<STRIDE>, TileCap<BITS>::small>(P, T, blk, L, Q, keys, cs, ce, lam, dens, ncnt,
                                                                      ccnt, C, reg.sh, reg.q);
    }
    rest.visit([&](uint32_t g) __attribute__((always_inline)) {
      lambda_particle<PBD_KERNEL_TEXTBOOK, FIRST>(P, g, Q, keys, cs, ce, lam, dens, ncnt, ccnt);
    });
    if (!STRIDE) break;
    if (mode == 1) __syncthreads();  // the next rank may be small tiles in the same LDS bytes
  }
}

// Delta-p (+ collisions, apply, update) over one tile, over the lambda pass's
// lists (use_list) or a scan of the stencil; with a carry, each particle's
// displacement bound after the pass is recorded.
template <int BITS, bool COLLIDE, int NS, bool PH, class Team, int CAP>
__device__ __forceinline__ TileRest delta_tile(const DevParams& P, const TileList& T, uint32_t item, const NeighbourList& L, int use_list,
                                           uint32_t flags, const float4* __restrict__ Q,
                                           const float4* __restrict__ QX, const float* __restrict__ lam,
                                           const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                                           const uint32_t* __restrict__ ce, float4* __restrict__ Qo,
                                           float4* __restrict__ QXo, float4* __restrict__ DP,
                                           float4* __restrict__ VS, const Carry& C, TileShared<BITS>& sh,
                                           float4* s_q, uint32_t* s_gi) {
  constexpr int VAR = PBD_KERNEL_TEXTBOOK;
  const uint32_t tid = Team::tid();
  const TileOwn own = tile_own<BITS>(P, T, item, cs);
  const uint32_t blk = own.blk, g0 = own.g0, g1 = own.g1;
  // the thread's next particle: its key, list length and first chunk
  uint32_t key = 0u, n = kNlInvalid;
  uint4 chunk = make_uint4(0u, 0u, 0u, 0u);
  const auto next = [&](uint32_t g) __attribute__((always_inline)) {
    key = keys[g];
    if (use_list) {
      n = L.cnt[g];
      chunk = L.nl[g];
    }
  };
  const uint32_t total = tile_setup<BITS, Team, false>(P, blk, cs, ce, sh, [&]() __attribute__((always_inline)) {
    if (g0 + tid < g1) next(g0 + tid);
  }, own.half);
  TileRest rest = tile_rest<Team>(g0, g1, total > (uint32_t)CAP);
  if (total > (uint32_t)CAP) return rest;
  // s_gi (friction-capable passes): the global index of every slot, for the
  // displacements of a solid contact's partner
  tile_load<BITS, CAP, Team>(P, sh, total, Q, s_q, s_gi, g0, [&](uint32_t gi) { return lam[gi]; });
  Team::sync();
  uint32_t round = 0u;
  for (uint32_t g = g0 + tid; g < g1; g += Team::kSize, ++round) {
    if (round) next(g);
    int h;
    uint32_t slot;
    tile_locate<BITS>(sh, key, g, h, slot);
    // with phases, a particle without a list takes the global path (the tile holds
    // no phases for a scan)
    if (n == kNlInvalid && (PH || tile_count<BITS>(sh, h) > P.cap)) {
      rest.bits |= 1u << round;
      continue;
    }
    const float4 q0 = Q[g], qx = QX[g];  // for the end, loaded beside the walk
    const float4 qb = s_q[slot];
    // phases: delta p between fluid particles only; the contact push on every pair,
    // friction on contacts with a solid (displacements p* - x from the global arrays)
    const bool si = PH && P.phs[g] != 0u;
    const bool fric = PH && COLLIDE && P.mu_s > 0.0f;
    float dix = 0.0f, diy = 0.0f, diz = 0.0f;
    if (fric) {
      dix = q0.x - qx.x;
      diy = q0.y - qx.y;
      diz = q0.z - qx.z;
    }
    DeltaAcc a;
    const auto pair = [&](uint32_t e) __attribute__((always_inline)) {
      const uint32_t j = PH ? (e & ~kNlSolid) : e;
      const float4 qj = s_q[j];
      const float rx = qb.x - qj.x, ry = qb.y - qj.y, rz = qb.z - qj.z;
      if (PH && (si || (e & kNlSolid))) {
        delta_pair<VAR, false, COLLIDE, NS, PH && !COLLIDE>(P, 0.0f, 0.0f, rx, ry, rz, true, a);
        if (fric) {
          const float r2 = length_sq(rx, ry, rz);
          if (r2 > 0.0f) {
            const float il = rsq(r2), len = r2 * il;
            if (len < P.diameter && len > 0.00001f) {
              const uint32_t gj = s_gi ? s_gi[j] : tile_global<BITS>(sh, j);
              const float4 qgj = Q[gj], xj = QX[gj];
              friction_pair(P, rx, ry, rz, len, il, dix, diy, diz, qgj.x - xj.x, qgj.y - xj.y, qgj.z - xj.z, a);
            }
          }
        }
      } else {
        delta_pair<VAR, true, COLLIDE, NS, PH && !COLLIDE>(P, qb.w, qj.w, rx, ry, rz, true, a);
      }
    };
    if (n != kNlInvalid) nl_visit(L, g, n, chunk, pair);
    else tile_stencil<BITS>(sh, h, slot, pair);
    const uint32_t sc = scene_of_key(P, key);
    const float cx = frame_corner(P, frame_origin(P, sc, 0), compact10(key >> 2));
    const float cy = frame_corner(P, frame_origin(P, sc, 1), compact10(key >> 1));
    const float cz = frame_corner(P, frame_origin(P, sc, 2), compact10(key));
    track_move(C, g, q0, delta_finish<VAR, true>(P, flags, g, q0, qx, a, cx, cy, cz, key, Qo, QXo, DP, VS));
  }
  return rest;
}

template <int BITS, bool COLLIDE, int NS, bool STRIDE, bool PH>
__global__ __launch_bounds__(kTileThreads) void k_tile_delta(DevParams P, TileList T, NeighbourList L, int use_list,
                                                             uint32_t flags, const float4* __restrict__ Q,
                                                             const float4* __restrict__ QX,
                                                             const float* __restrict__ lam,
                                                             const uint32_t* __restrict__ keys,
                                                             const uint32_t* __restrict__ cs,
                                                             const uint32_t* __restrict__ ce, float4* __restrict__ Qo,
                                                             float4* __restrict__ QXo, float4* __restrict__ DP,
                                                             float4* __restrict__ VS, Carry C) {
  // friction (phases and collisions) reads the partner's global arrays: keep
  // each slot's global index
  constexpr bool GI = PH && COLLIDE;
  __shared__ TileLds<BITS, GI> lds;
  const TileItems it = tile_items(T);
  // STRIDE: every gridDim-th rank from tile_rank0(); otherwise the grid covers
  // the ranks and a workgroup takes one
  for (uint32_t r = tile_rank0();; r += gridDim.x) {
    uint32_t blk;
    const int mode = tile_pick(T, it, r, blk);
    if (mode == 0) break;
    TileRest rest;
    if (mode == 1) {
      rest = delta_tile<BITS, COLLIDE, NS, PH, TeamBlockN<kTileThreads, STRIDE>, TileCap<BITS>::value>(
          P, T, blk, L, use_list, flags, Q, QX, lam, keys, cs, ce, Qo, QXo, DP, VS, C, lds.big.sh, lds.big.q,
          GI ? lds.big.gi : nullptr);
    } else {
      auto& reg = lds.small[threadIdx.x >> 6];
      rest = delta_tile<BITS, COLLIDE, NS, PH, TeamWaveT<STRIDE>, TileCap<BITS>::small>(P, T, blk, L, use_list, flags, Q, QX, lam,
                                                                           keys, cs, ce, Qo, QXo, DP, VS, C, reg.sh,
                                                                           reg.q, GI ? reg.gi : nullptr);
    }
    rest.visit([&](uint32_t g) __attribute__((always_inline)) {
      const float4 q0 = Q[g];
      track_move(C, g, q0, delta_particle<PBD_KERNEL_TEXTBOOK, true, COLLIDE>(P, flags, g, Q, QX, lam, keys, cs, ce,
                                                                            Qo, QXo, DP, VS));
    });
    if (!STRIDE) break;
    if (mode == 1) __syncthreads();  // the next rank may be small tiles in the same LDS bytes
  }
}

// XSPH: the same neighbour walk also applies XSPH (computeViscosity,
// Density.h:280-310) and writes the velocities to Vo, in the order and with
// the arithmetic of the final pass, which then leaves them alone.  With a
// carry, a carrying tile whose halo has moved less than P.reuse_max since it
// last built its lists keeps them, the others rebuild theirs (for the final
// pass: without the skin), and every tile decides whether it carries its lists
// in the next substep: when its halo has moved less than P.reuse_max since its
// lists were built, or, for a tile that did not carry, over the whole substep.
template <int BITS, bool XSPH, bool PH, class Team, int CAP>
__device__ __forceinline__ TileRest omega_tile(const DevParams& P, const TileList& T, uint32_t item, const NeighbourList& L,
                                           const float4* __restrict__ Q, const float4* __restrict__ VS,
                                           const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                                           const uint32_t* __restrict__ ce, float4* __restrict__ OM,
                                           float4* __restrict__ Vo, const Carry& C, TileShared<BITS>& sh,
                                           float4* s_q, uint32_t* s_gi) {
  constexpr int VAR = PBD_KERNEL_TEXTBOOK;
  const uint32_t tid = Team::tid();
  const TileOwn own = tile_own<BITS>(P, T, item, cs);
  const uint32_t blk = own.blk, g0 = own.g0, g1 = own.g1;
  uint32_t key = 0u;  // of the thread's next particle, and its velocity
  float4 v4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const uint32_t total = tile_setup<BITS, Team, false>(P, blk, cs, ce, sh, [&]() __attribute__((always_inline)) {
    if (g0 + tid < g1) {
      key = keys[g0 + tid];
      v4 = VS[g0 + tid];
    }
  }, own.half);
  TileRest rest = tile_rest<Team>(g0, g1, total > (uint32_t)CAP);
  if (total > (uint32_t)CAP) {
    for (uint32_t g = g0 + tid; g < g1; g += Team::kSize) L.cnt[g] = kNlInvalid;
    if (tid == 0) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_BLOCK], (unsigned long long)(g1 - g0));
    return rest;
  }
  // global index of each slot: velocities are gathered from L2
  // .w: 1 for a solid particle (PH), else 0
  const uint32_t m = C.disp ? C.built[own.carried()] : kNoCarry;
  const bool carry = m != kNoCarry;
  tile_load<BITS, CAP, Team>(P, sh, total, Q, s_q, s_gi, g0,
                             [&](uint32_t gi) { return PH && P.phs[gi] ? 1.0f : 0.0f; },
                             C.disp ? C.bounds(C.pass) : nullptr, carry ? C.bounds(m) : nullptr);
  Team::sync();
  const bool calm = C.disp && tile_keeps_lists<BITS>(P, sh);
  const bool keep = carry && calm;
  if (tid == 0 && C.disp) {
    C.mode[own.carried()] = calm ? 1u : 0u;
    if (carry) atomicAdd(&L.stats[keep ? PBD_COUNTER_LIST_CARRIES : PBD_COUNTER_LIST_RESCANS],
                         (unsigned long long)(g1 - g0));
  }
  uint32_t round = 0u;
  for (uint32_t g = g0 + tid; g < g1; g += Team::kSize, ++round) {
    if (round) {
      key = keys[g];
      v4 = VS[g];
    }
    int h;
    uint32_t slot;
    tile_locate<BITS>(sh, key, g, h, slot);
    // kept lists: a particle without one is over the cap (global path, as when
    // the list was built) or has a long list (stencil scan)
    uint32_t n = keep ? (uint32_t)L.cnt[g] : (uint32_t)kNlInvalid;
    if ((!keep || n == kNlInvalid) && tile_count<BITS>(sh, h) > P.cap) {
      rest.bits |= 1u << round;
      if (!keep) {
        L.cnt[g] = kNlInvalid;
        atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_CAP], 1ull);
      }
      continue;
    }
    const float4 qi = s_q[slot];
    // velocity components as scalars (a float4 aggregate captured by the pair
    // lambda is not promoted to registers)
    const float vx = v4.x, vy = v4.y, vz = v4.z, vw = v4.w;
    OmegaAcc a;
    FinalAcc xa;
    const bool si = PH && qi.w != 0.0f;  // a solid particle: omega 0, no XSPH
    if (si) {
      // no pair of a solid particle counts here, in the final pass or in the
      // reverse passes that walk these lists: an empty list, the sums at zero
      if (!keep) L.cnt[g] = 0u;
      OM[g] = omega_finish<VAR>(P, a);
      if (XSPH) {
        const float c = P.c_visc * P.wc * P.vol;
        Vo[g] = make_float4(vx + c * xa.sx, vy + c * xa.sy, vz + c * xa.sz, vw + c * xa.sw);
      }
      continue;
    }
    const auto pair = [&](uint32_t j) __attribute__((always_inline)) {
      if (PH && (si || (j & kNlSolid))) return;  // fluid neighbours only
      const float4 qj = slot_read(s_q, j);
      if (PH && qj.w != 0.0f) return;
      const float4 vj = VS[s_gi[j]];
      const float rx = qi.x - qj.x, ry = qi.y - qj.y, rz = qi.z - qj.z;
      omega_pair<VAR, PH>(P, rx, ry, rz, vj.x - vx, vj.y - vy, vj.z - vz, a);
      if (XSPH) final_pair_textbook<VAR, PH>(P, false, true, rx, ry, rz, make_float4(vx, vy, vz, vw), vj, 0.0f, 0.0f, xa);
    };
    if (!keep) {
      n = nl_build<BITS, CAP, PH>(P, L, g, sh, s_q, h, slot, qi, P.list_r2);
      L.cnt[g] = (uint16_t)n;
      if (n == kNlInvalid) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_LONG], 1ull);
    }
    if (n != kNlInvalid) nl_visit(L, g, n, L.nl[g], pair);
    else tile_stencil<BITS>(sh, h, slot, pair);
    OM[g] = omega_finish<VAR>(P, a);
    if (XSPH) {
      const float c = P.c_visc * P.wc * P.vol;
      Vo[g] = make_float4(vx + c * xa.sx, vy + c * xa.sy, vz + c * xa.sz, vw + c * xa.sw);
    }
  }
  return rest;
}

template <int BITS, bool XSPH, bool STRIDE, bool PH>
__global__ __launch_bounds__(kTileThreads, STRIDE && BITS == 5 ? 4 : 1) void k_tile_omega(DevParams P, TileList T, NeighbourList L,
                                                             const float4* __restrict__ Q,
                                                             const float4* __restrict__ VS,
                                                             const uint32_t* __restrict__ keys,
                                                             const uint32_t* __restrict__ cs,
                                                             const uint32_t* __restrict__ ce, float4* __restrict__ OM,
                                                             float4* __restrict__ Vo, Carry C) {
  __shared__ TileLds<BITS, true> lds;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&L.stats[PBD_COUNTER_LIST_BUILDS], 1ull);
  const TileItems it = tile_items(T);
  // STRIDE: every gridDim-th rank from tile_rank0(); otherwise the grid covers
  // the ranks and a workgroup takes one
  for (uint32_t r = tile_rank0();; r += gridDim.x) {
    uint32_t blk;
    const int mode = tile_pick(T, it, r, blk);
    if (mode == 0) break;
    TileRest rest;
    if (mode == 1) {
      rest = omega_tile<BITS, XSPH, PH, TeamBlockN<kTileThreads, STRIDE>, TileCap<BITS>::value>(P, T, blk, L, Q, VS, keys, cs, ce, OM, Vo, C,
                                                                     lds.big.sh, lds.big.q, lds.big.gi);
    } else {
      auto& reg = lds.small[threadIdx.x >> 6];
      rest = omega_tile<BITS, XSPH, PH, TeamWaveT<STRIDE>, TileCap<BITS>::small>(P, T, blk, L, Q, VS, keys, cs, ce, OM, Vo, C,
                                                                    reg.sh, reg.q, reg.gi);
    }
    rest.visit([&](uint32_t g) __attribute__((always_inline)) {
      omega_particle<PBD_KERNEL_TEXTBOOK>(P, g, Q, VS, keys, cs, ce, OM);
      if (XSPH) Vo[g] = xsph_particle<PBD_KERNEL_TEXTBOOK>(P, g, Q, VS, keys, cs, ce);
    });
    if (!STRIDE) break;
    if (mode == 1) __syncthreads();  // the next rank may be small tiles in the same LDS bytes
  }
}

template <int BITS, bool VORT, bool XSPH, bool PH, class Team, int CAP>
__device__ __forceinline__ TileRest final_tile(const DevParams& P, const TileList& T, uint32_t item, const NeighbourList& L, int use_list,
                                           uint32_t flags, const float4* __restrict__ Q,
                                           const float4* __restrict__ QX, const float4* __restrict__ VS,
                                           const float4* __restrict__ OM, const uint32_t* __restrict__ keys,
                                           const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                                           const float4* __restrict__ CS, const uint32_t* __restrict__ ncnt,
                                           float4* __restrict__ Xo, float4* __restrict__ Po, float4* __restrict__ Vo,
                                           float4* __restrict__ Co, float4* __restrict__ Fo, TileShared<BITS>& sh,
                                           float4* s_q, uint32_t* s_gi) {
  constexpr int VAR = PBD_KERNEL_TEXTBOOK;
  const uint32_t tid = Team::tid();
  const TileOwn own = tile_own<BITS>(P, T, item, cs);
  const uint32_t blk = own.blk, g0 = own.g0, g1 = own.g1;
  // the thread's next particle: its key, list length and first chunk
  uint32_t key = 0u, n = kNlInvalid;
  uint4 chunk = make_uint4(0u, 0u, 0u, 0u);
  const auto next = [&](uint32_t g) __attribute__((always_inline)) {
    key = keys[g];
    if (use_list) {
      n = L.cnt[g];
      chunk = L.nl[g];
    }
  };
  const uint32_t total = tile_setup<BITS, Team, false>(P, blk, cs, ce, sh, [&]() __attribute__((always_inline)) {
    if (g0 + tid < g1) next(g0 + tid);
  }, own.half);
  constexpr bool vort = VORT, xsph = XSPH;  // flags & FF_VORT, flags & FF_XSPH
  TileRest rest = tile_rest<Team>(g0, g1, total > (uint32_t)CAP);
  if (total > (uint32_t)CAP) {
    for (uint32_t g = g0 + tid; PH && g < g1; g += Team::kSize) P.ph[g] = P.phs[g];  // as below
    return rest;
  }
  // global index of each slot (XSPH only), for the velocity gathers from L2
  const auto omega_len = [&](uint32_t gi) { return vort ? OM[gi].w : 0.0f; };
  tile_load<BITS, CAP, Team>(P, sh, total, Q, s_q, XSPH ? s_gi : nullptr, g0, omega_len);
  Team::sync();
  uint32_t round = 0u;
  for (uint32_t g = g0 + tid; g < g1; g += Team::kSize, ++round) {
    if (PH) P.ph[g] = P.phs[g];  // phases follow the particles into the sorted order
    if (round) next(g);
    int h;
    uint32_t slot;
    tile_locate<BITS>(sh, key, g, h, slot);
    // with phases, a particle without a list takes the global path (the tile holds
    // no phases for a scan)
    if (n == kNlInvalid && (PH || tile_count<BITS>(sh, h) > P.cap)) {
      rest.bits |= 1u << round;
      continue;
    }
    const bool si = PH && P.phs[g] != 0u;  // a solid particle: no vorticity force, no XSPH
    const float4 qb = s_q[slot];
    // velocity components as scalars: copies of the float4 aggregate inside the
    // pair loop are not promoted to registers and end up in scratch
    const float4 v4 = VS[g];
    const float vx = v4.x, vy = v4.y, vz = v4.z, vw = v4.w;
    const float4 oi = vort ? OM[g] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    FinalAcc a;
    if (vort || xsph) {
      const auto pair = [&](uint32_t j) __attribute__((always_inline)) {
        if (PH && (si || (j & kNlSolid))) return;  // fluid neighbours only
        const float4 qj = slot_read(s_q, j);
        const float4 vj = XSPH ? VS[s_gi[j]] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // unused without XSPH
        final_pair_textbook<VAR>(P, vort, xsph, qb.x - qj.x, qb.y - qj.y, qb.z - qj.z, make_float4(vx, vy, vz, vw),
                                 vj, oi.w, qj.w, a);
      };
      if (n != kNlInvalid) nl_visit(L, g, n, chunk, pair);
      else tile_stencil<BITS>(sh, h, slot, pair);
    }
    const uint32_t sc = scene_of_key(P, key);
    const float cx = frame_corner(P, frame_origin(P, sc, 0), compact10(key >> 2));
    const float cy = frame_corner(P, frame_origin(P, sc, 1), compact10(key >> 1));
    const float cz = frame_corner(P, frame_origin(P, sc, 2), compact10(key));
    final_finish<VAR>(P, flags, g, Q[g], make_float4(vx, vy, vz, vw), oi, a, cx, cy, cz, QX, CS, ncnt, Xo, Po, Vo,
                      Co, Fo);
  }
  return rest;
}

template <int BITS, bool VORT, bool XSPH, bool STRIDE, bool PH>
__global__ __launch_bounds__(kTileThreads, STRIDE && BITS == 5 ? 4 : 1) void k_tile_final(
    DevParams P, TileList T, NeighbourList L, int use_list, uint32_t flags, const float4* __restrict__ Q,
    const float4* __restrict__ QX, const float4* __restrict__ VS, const float4* __restrict__ OM,
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
    const float4* __restrict__ CS, const uint32_t* __restrict__ ncnt, float4* __restrict__ Xo,
    float4* __restrict__ Po, float4* __restrict__ Vo, float4* __restrict__ Co, float4* __restrict__ Fo) {
  __shared__ TileLds<BITS, XSPH> lds;
  const TileItems it = tile_items(T);
  // STRIDE: every gridDim-th rank from tile_rank0(); otherwise the grid covers
  // the ranks and a workgroup takes one
  for (uint32_t r = tile_rank0();; r += gridDim.x) {
    uint32_t blk;
    const int mode = tile_pick(T, it, r, blk);
    if (mode == 0) break;
    TileRest rest;
    if (mode == 1) {
      rest = final_tile<BITS, VORT, XSPH, PH, TeamBlockN<kTileThreads, STRIDE>, TileCap<BITS>::value>(
          P, T, blk, L, use_list, flags, Q, QX, VS, OM, keys, cs, ce, CS, ncnt, Xo, Po, Vo, Co, Fo, lds.big.sh, lds.big.q,
          lds.big.gi);
    } else {
      auto& reg = lds.small[threadIdx.x >> 6];
      rest = final_tile<BITS, VORT, XSPH, PH, TeamWaveT<STRIDE>, TileCap<BITS>::small>(P, T, blk, L, use_list, flags, Q, QX, VS, OM,
                                                                          keys, cs, ce, CS, ncnt, Xo, Po, Vo, Co, Fo,
                                                                          reg.sh, reg.q, reg.gi);
    }
    rest.visit([&](uint32_t g) __attribute__((always_inline)) {
      final_particle<PBD_KERNEL_TEXTBOOK>(P, flags, g, Q, QX, VS, OM, keys, cs, ce, CS, ncnt, Xo, Po, Vo, Co, Fo);
    });
    if (!STRIDE) break;
    if (mode == 1) __syncthreads();  // the next rank may be small tiles in the same LDS bytes
  }
}

// ---------------------------------------------------------------------------
// Wide tile passes, for scenes whose blocks are too few to fill the chip: four lanes
// (a quad of the wave) per particle in 1024-thread workgroups, a workgroup per occupied
// block (there are no small tiles).  With a thread per particle a 32K scene runs 128 to 256
// workgroups of one wave per SIMD, and a pass lasts as long as one thread's walk over
// its particle's candidates and pairs.  Here
//   - the lanes of a quad scan two or three of the nine stencil columns each, and write
//     their in-range slots to the particle's list in LDS, each from the place that the
//     counts of the lanes before it give: the list is nl_build's;
//   - a quad takes four list entries at a time, a lane forming each pair's terms; the
//     terms are then added in list order, each lane adding all four (the values cross
//     the quad by DPP), with the fused operations of the one-lane passes, so the sums
//     are theirs bit for bit.
// The VALU work per pair nearly doubles (13 instructions a pair and lane against 29 a
// pair), so the one-lane passes stay the faster ones once the chip is full: wide_tiles
// in kernels.hpp draws the line.  32K column, one lane to four: lambda with its lists
// built 21.5 to 17.4 us, omega 24.6 to 20.2 us.
constexpr uint32_t kQuad = 4;
constexpr uint32_t kWideParticles = kWideThreads / kQuad;  // particles of a round

struct WideLds {
  TileShared<5> sh;
  float4 q[TileCap<5>::value + kScanUnroll];
  uint16_t list[kWideParticles][kNlMax];  // 16-byte chunks, as the global lists'
};
// (the registers, 93 to 99, admit one workgroup of 16 waves a CU)
static_assert(2 * sizeof(WideLds) <= kLdsBytes, "LDS of two workgroups");
static_assert(sizeof(TileShared<5>) % 16 == 0 || alignof(WideLds) >= 16, "alignment of the halo");

// The value that lane p of the quad holds.
template <int p>
__device__ __forceinline__ float quad_get(float x) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(x), p * 0x55, 0xF, 0xF, true));
}
template <int p>
__device__ __forceinline__ uint32_t quad_get(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, p * 0x55, 0xF, 0xF, true);
}

// The block of work item r (every occupied block is a large one).
__device__ __forceinline__ bool wide_pick(const TileList& T, uint32_t r, uint32_t& blk) {
  const uint32_t large = T.large[min(r, T.cap - 1u)];  // with the count, not after it
  if (r >= T.count[0]) return false;
  blk = large;
  return true;
}

// A thread's particles for the global path: the quad's first lane takes those of the
// rounds in `bits`; a block beyond the capacity goes round all threads.
__device__ __forceinline__ TileRest wide_rest(uint32_t g0, uint32_t g1, bool all) {
  TileRest r;
  r.g = g0 + (all ? threadIdx.x : threadIdx.x / kQuad);
  r.end = g1;
  r.stride = all ? kWideThreads : kWideParticles;
  r.all = all;
  return r;
}

// Builds the list of the quad's particle into `list` (LDS) and, chunk by chunk, the
// global lists; as nl_build.  A column's first 64 slots are scanned once, their bits
// kept in registers; what a longer column has more is scanned again when its slots are
// written.
__device__ __forceinline__ uint32_t wide_build(const NeighbourList& L, uint32_t g, const TileShared<5>& sh,
                                               const float4* s_q, uint16_t* list, int h, uint32_t slot, float4 qi,
                                               float r2) {
  using G = TileGeom<5>;
  constexpr uint32_t CAP = TileCap<5>::value;
  const uint32_t sub = threadIdx.x % kQuad;
  const uint32_t valid = fabsf(qi.x) + fabsf(qi.y) + fabsf(qi.z) < __builtin_inff() ? 0xFFFFFFFFu : 0u;
  const auto scan = [&](uint32_t s, uint32_t b) __attribute__((always_inline)) {
    uint32_t m = nl_mask(s_q, s, min(b - s, 32u), qi.x, qi.y, qi.z, r2) & valid;
    if (slot - s < 32u) m &= ~(1u << (slot - s));  // not the particle itself
    return m;
  };
  // columns 2 sub and 2 sub + 1; the last lane column 8 too
  uint32_t a[3], b[3], m0[3], m1[3], cnt = 0u;
#pragma unroll
  for (uint32_t k = 0; k < 3u; ++k) {
    const uint32_t c = 2u * sub + k;
    const int hb = h + ((int)(c / 3u) - 1) * G::SX + ((int)(c % 3u) - 1) * G::SY;
    const bool mine = k < 2u || sub == kQuad - 1u;
    a[k] = mine ? sh.lstart[hb - 1] : 0u;
    b[k] = mine ? sh.lstart[hb + 2] : 0u;
    m0[k] = m1[k] = 0u;
    if (a[k] < b[k]) m0[k] = scan(a[k], b[k]);
    if (a[k] + 32u < b[k]) m1[k] = scan(a[k] + 32u, b[k]);
    cnt += __builtin_popcount(m0[k]) + __builtin_popcount(m1[k]);
    for (uint32_t s = a[k] + 64u; s < b[k]; s += 32u) cnt += __builtin_popcount(scan(s, b[k]));
  }
  const uint32_t c0 = quad_get<0>(cnt), c1 = quad_get<1>(cnt), c2 = quad_get<2>(cnt), c3 = quad_get<3>(cnt);
  const uint32_t n = c0 + c1 + c2 + c3;
  if (n > kNlMax) return kNlInvalid;
  uint32_t i = (sub > 0u ? c0 : 0u) + (sub > 1u ? c1 : 0u) + (sub > 2u ? c2 : 0u);
  const auto put = [&](uint32_t s, uint32_t m) __attribute__((always_inline)) {
    while (m) {
      list[i++] = (uint16_t)(s + (uint32_t)__builtin_ctz(m));
      m &= m - 1u;
    }
  };
#pragma unroll
  for (uint32_t k = 0; k < 3u; ++k) {
    put(a[k], m0[k]);
    put(a[k] + 32u, m1[k]);
    for (uint32_t s = a[k] + 64u; s < b[k]; s += 32u) put(s, scan(s, b[k]));
  }
  const uint32_t np = (n + 7u) & ~7u;
  for (uint32_t k = n + sub; k < np; k += kQuad) list[k] = (uint16_t)CAP;
  TeamWave::sync();
  for (uint32_t c = sub; c < np / 8u; c += kQuad)
    L.nl[(size_t)c * L.cap + g] = *reinterpret_cast<const uint4*>(list + 8u * c);
  return np;
}

// The list of particle g (n entries, a multiple of 8) from the global lists.
__device__ __forceinline__ void wide_fetch(const NeighbourList& L, uint32_t g, uint32_t n, uint16_t* list) {
  for (uint32_t c = threadIdx.x % kQuad; c < n / 8u; c += kQuad)
    *reinterpret_cast<uint4*>(list + 8u * c) = L.nl[(size_t)c * L.cap + g];
  TeamWave::sync();
}

// The quad's walk over the list: pair(j) forms a lane's terms (of slot j), add(get) adds
// those of one lane, get(x) its value of x, lane after lane.
template <class Pair, class Add>
__device__ __forceinline__ void wide_visit(const uint16_t* list, uint32_t n, Pair pair, Add add) {
  const uint32_t sub = threadIdx.x % kQuad;
  const auto quad = [&](const auto& t) __attribute__((always_inline)) {
    add(t, [](auto x) __attribute__((always_inline)) { return quad_get<0>(x); });
    add(t, [](auto x) __attribute__((always_inline)) { return quad_get<1>(x); });
    add(t, [](auto x) __attribute__((always_inline)) { return quad_get<2>(x); });
    add(t, [](auto x) __attribute__((always_inline)) { return quad_get<3>(x); });
  };
  for (uint32_t k = 0; k < n; k += 2u * kQuad) {  // n is a multiple of 8
    const auto t0 = pair((uint32_t)list[k + sub]);
    const auto t1 = pair((uint32_t)list[k + kQuad + sub]);
    quad(t0);
    quad(t1);
  }
}

template <bool FIRST>
__global__ __launch_bounds__(kWideThreads) void k_wide_lambda(DevParams P, TileList T, NeighbourList L,
                                                              const float4* __restrict__ Q,
                                                              const uint32_t* __restrict__ keys,
                                                              const uint32_t* __restrict__ cs,
                                                              const uint32_t* __restrict__ ce,
                                                              float* __restrict__ lam, float* __restrict__ dens,
                                                              uint32_t* __restrict__ ncnt,
                                                              uint32_t* __restrict__ ccnt, Carry C) {
  constexpr int VAR = PBD_KERNEL_TEXTBOOK;
  constexpr int CAP = TileCap<5>::value;
  __shared__ WideLds lds;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&L.stats[PBD_COUNTER_LIST_BUILDS], 1ull);
  uint32_t item;
  if (!wide_pick(T, blockIdx.x, item)) return;
  TileShared<5>& sh = lds.sh;
  const uint32_t tid = threadIdx.x, sub = tid % kQuad;
  const TileOwn own = tile_own<5>(P, T, item, cs);
  const uint32_t blk = own.blk, g0 = own.g0, g1 = own.g1, gf = g0 + tid / kQuad;
  uint32_t key = 0u;  // of the quad's next particle
  const uint32_t total = tile_setup<5, TeamWide, false>(P, blk, cs, ce, sh, [&]() __attribute__((always_inline)) {
    if (gf < g1) key = keys[gf];
  }, own.half);
  TileRest rest = wide_rest(g0, g1, total > (uint32_t)CAP);
  if (total > (uint32_t)CAP) {
    for (uint32_t g = g0 + tid; g < g1; g += kWideThreads) L.cnt[g] = kNlInvalid;
    if (tid == 0) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_BLOCK], (unsigned long long)(g1 - g0));
  } else {
    // as lambda_tile
    const uint32_t m = C.disp ? (FIRST ? (C.mode[own.carried()] ? 0u : kNoCarry) : C.built[own.carried()]) : kNoCarry;
    const bool carry = !FIRST && m != kNoCarry;
    const float r2 = m != kNoCarry ? P.tile_r2 : P.list_r2;
    tile_load<5, CAP, TeamWide>(P, sh, total, Q, lds.q, nullptr, 0u, [](uint32_t) { return 0.0f; },
                                carry ? C.bounds(C.pass) : nullptr, carry ? C.bounds(m) : nullptr);
    __syncthreads();
    const bool keep = carry && tile_keeps_lists<5>(P, sh);
    if (tid == 0 && C.disp) {
      if (FIRST) C.built[own.carried()] = (uint16_t)m;
      else if (carry && !keep) C.built[own.carried()] = (uint16_t)C.pass;
      if (carry) atomicAdd(&L.stats[keep ? PBD_COUNTER_LIST_CARRIES : PBD_COUNTER_LIST_RESCANS],
                           (unsigned long long)(g1 - g0));
    }
    uint16_t* list = lds.list[tid / kQuad];
    uint32_t round = 0u;
    for (uint32_t g = gf; g < g1; g += kWideParticles, ++round) {
      if (round) key = keys[g];
      int h;
      uint32_t slot;
      tile_locate<5>(sh, key, g, h, slot);
      uint32_t cnt = 0u, n = keep ? (uint32_t)L.cnt[g] : (uint32_t)kNlInvalid;
      if (!keep || n == kNlInvalid) {
        cnt = tile_count<5>(sh, h);
        if (cnt > P.cap) {
          if (sub == 0u) {
            rest.bits |= 1u << round;
            if (!keep) {
              L.cnt[g] = kNlInvalid;
              atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_CAP], 1ull);
            }
          }
          continue;
        }
      }
      const float4 qi = lds.q[slot];
      if (!keep) {
        n = wide_build(L, g, sh, lds.q, list, h, slot, qi, r2);
        if (sub == 0u) {
          L.cnt[g] = (uint16_t)n;
          if (n == kNlInvalid) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_LONG], 1ull);
        }
      } else if (n != kNlInvalid) {
        wide_fetch(L, g, n, list);
      }
      LambdaAcc a;
      if (n != kNlInvalid) {
        struct Term {
          float rx, ry, rz, t, t2, g, hr4;
        };
        wide_visit(
            list, n,
            [&](uint32_t j) __attribute__((always_inline)) {
              const float4 qj = slot_read(lds.q, j);
              Term e;
              e.rx = qi.x - qj.x;
              e.ry = qi.y - qj.y;
              e.rz = qi.z - qj.z;
              const float d2 = length_sq(e.rx, e.ry, e.rz);
              e.t = fmaxf(P.hp2 - d2, 0.0f);
              e.t2 = e.t * e.t;
              e.g = grad_factor<VAR>(P, d2, e.hr4);
              return e;
            },
            [&](const Term& e, auto get) __attribute__((always_inline)) {
              const float g1_ = get(e.g);
              a.A = fmaf(get(e.t), get(e.t2), a.A);
              a.gx = fmaf(get(e.rx), g1_, a.gx);
              a.gy = fmaf(get(e.ry), g1_, a.gy);
              a.gz = fmaf(get(e.rz), g1_, a.gz);
              a.B += get(e.hr4);
            });
      } else {  // more pairs than a list holds: every lane scans
        tile_stencil<5>(sh, h, slot, [&](uint32_t j) __attribute__((always_inline)) {
          const float4 qj = slot_read(lds.q, j);
          lambda_pair<VAR>(P, qi.x - qj.x, qi.y - qj.y, qi.z - qj.z, a);
        });
      }
      if (sub != 0u) continue;
      float W;
      lam[g] = lambda_finish_fused(P, a, W, scene_eps(P, key));
      if (FIRST) {
        dens[g] = W;
        ncnt[g] = cnt;
        ccnt[g] = cnt;
      }
    }
  }
  rest.visit([&](uint32_t g) __attribute__((always_inline)) {
    lambda_particle<VAR, FIRST>(P, g, Q, keys, cs, ce, lam, dens, ncnt, ccnt);
  });
}

template <bool XSPH>
__global__ __launch_bounds__(kWideThreads) void k_wide_omega(DevParams P, TileList T, NeighbourList L,
                                                             const float4* __restrict__ Q,
                                                             const float4* __restrict__ VS,
                                                             const uint32_t* __restrict__ keys,
                                                             const uint32_t* __restrict__ cs,
                                                             const uint32_t* __restrict__ ce, float4* __restrict__ OM,
                                                             float4* __restrict__ Vo, Carry C) {
  constexpr int VAR = PBD_KERNEL_TEXTBOOK;
  constexpr int CAP = TileCap<5>::value;
  __shared__ WideLds lds;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&L.stats[PBD_COUNTER_LIST_BUILDS], 1ull);
  uint32_t item;
  if (!wide_pick(T, blockIdx.x, item)) return;
  TileShared<5>& sh = lds.sh;
  const uint32_t tid = threadIdx.x, sub = tid % kQuad;
  const TileOwn own = tile_own<5>(P, T, item, cs);
  const uint32_t blk = own.blk, g0 = own.g0, g1 = own.g1, gf = g0 + tid / kQuad;
  uint32_t key = 0u;  // of the quad's next particle, and its velocity
  float4 v4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const uint32_t total = tile_setup<5, TeamWide, false>(P, blk, cs, ce, sh, [&]() __attribute__((always_inline)) {
    if (gf < g1) {
      key = keys[gf];
      v4 = VS[gf];
    }
  }, own.half);
  TileRest rest = wide_rest(g0, g1, total > (uint32_t)CAP);
  if (total > (uint32_t)CAP) {
    for (uint32_t g = g0 + tid; g < g1; g += kWideThreads) L.cnt[g] = kNlInvalid;
    if (tid == 0) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_BLOCK], (unsigned long long)(g1 - g0));
  } else {
    // as omega_tile; .w: the slot's global index (velocities are gathered from L2), of the
    // sentinel the block's first particle (its pair terms are zero)
    const uint32_t m = C.disp ? C.built[own.carried()] : kNoCarry;
    const bool carry = m != kNoCarry;
    tile_load<5, CAP, TeamWide>(P, sh, total, Q, lds.q, nullptr, 0u,
                                [](uint32_t gi) { return __uint_as_float(gi); }, C.disp ? C.bounds(C.pass) : nullptr,
                                carry ? C.bounds(m) : nullptr);
    __syncthreads();
    const bool calm = C.disp && tile_keeps_lists<5>(P, sh);
    const bool keep = carry && calm;
    if (tid == 0 && C.disp) {
      C.mode[own.carried()] = calm ? 1u : 0u;
      if (carry) atomicAdd(&L.stats[keep ? PBD_COUNTER_LIST_CARRIES : PBD_COUNTER_LIST_RESCANS],
                           (unsigned long long)(g1 - g0));
    }
    uint16_t* list = lds.list[tid / kQuad];
    uint32_t round = 0u;
    for (uint32_t g = gf; g < g1; g += kWideParticles, ++round) {
      if (round) {
        key = keys[g];
        v4 = VS[g];
      }
      int h;
      uint32_t slot;
      tile_locate<5>(sh, key, g, h, slot);
      uint32_t n = keep ? (uint32_t)L.cnt[g] : (uint32_t)kNlInvalid;
      if (n == kNlInvalid && tile_count<5>(sh, h) > P.cap) {
        if (sub == 0u) {
          rest.bits |= 1u << round;
          if (!keep) {
            L.cnt[g] = kNlInvalid;
            atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_CAP], 1ull);
          }
        }
        continue;
      }
      const float4 qi = lds.q[slot];
      const float vx = v4.x, vy = v4.y, vz = v4.z, vw = v4.w;
      if (!keep) {
        n = wide_build(L, g, sh, lds.q, list, h, slot, qi, P.list_r2);
        if (sub == 0u) {
          L.cnt[g] = (uint16_t)n;
          if (n == kNlInvalid) atomicAdd(&L.stats[PBD_COUNTER_UNLISTED_LONG], 1ull);
        }
      } else if (n != kNlInvalid) {
        wide_fetch(L, g, n, list);
      }
      OmegaAcc a;
      FinalAcc xa;
      if (n != kNlInvalid) {
        struct Term {
          float ox, oy, oz, w, dx, dy, dz, dw;
        };
        wide_visit(
            list, n,
            [&](uint32_t j) __attribute__((always_inline)) {
              const float4 qj = lds.q[j];
              const float4 vj = VS[j == (uint32_t)CAP ? g0 : __float_as_uint(qj.w)];
              const float rx = qi.x - qj.x, ry = qi.y - qj.y, rz = qi.z - qj.z;
              const float d2 = length_sq(rx, ry, rz);
              Term e;
              e.dx = vj.x - vx;
              e.dy = vj.y - vy;
              e.dz = vj.z - vz;
              e.dw = vj.w - vw;
              float hr4;
              const float gf = grad_factor<VAR>(P, d2, hr4);
              const float gx = gf * rx, gy = gf * ry, gz = gf * rz;
              e.ox = fmaf(e.dy, gz, -(e.dz * gy));
              e.oy = fmaf(e.dz, gx, -(e.dx * gz));
              e.oz = fmaf(e.dx, gy, -(e.dy * gx));
              e.w = XSPH ? w_unnorm<VAR>(P, d2) : 0.0f;
              return e;
            },
            [&](const Term& e, auto get) __attribute__((always_inline)) {
              a.ox += get(e.ox);
              a.oy += get(e.oy);
              a.oz += get(e.oz);
              if (XSPH) {
                const float w = get(e.w);
                xa.sx = fmaf(get(e.dx), w, xa.sx);
                xa.sy = fmaf(get(e.dy), w, xa.sy);
                xa.sz = fmaf(get(e.dz), w, xa.sz);
                xa.sw = fmaf(get(e.dw), w, xa.sw);
              }
            });
      } else {
        tile_stencil<5>(sh, h, slot, [&](uint32_t j) __attribute__((always_inline)) {
          const float4 qj = lds.q[j];
          const float4 vj = VS[__float_as_uint(qj.w)];
          const float rx = qi.x - qj.x, ry = qi.y - qj.y, rz = qi.z - qj.z;
          omega_pair<VAR>(P, rx, ry, rz, vj.x - vx, vj.y - vy, vj.z - vz, a);
          if (XSPH) final_pair_textbook<VAR>(P, false, true, rx, ry, rz, make_float4(vx, vy, vz, vw), vj, 0.0f, 0.0f, xa);
        });
      }
      if (sub != 0u) continue;
      OM[g] = omega_finish<VAR>(P, a);
      if (XSPH) {
        const float c = P.c_visc * P.wc * P.vol;
        Vo[g] = make_float4(vx + c * xa.sx, vy + c * xa.sy, vz + c * xa.sz, vw + c * xa.sw);
      }
    }
  }
  rest.visit([&](uint32_t g) __attribute__((always_inline)) {
    omega_particle<VAR>(P, g, Q, VS, keys, cs, ce, OM);
    if (XSPH) Vo[g] = xsph_particle<VAR>(P, g, Q, VS, keys, cs, ce);
  });
}

// ---------------------------------------------------------------------------
// Host launchers.
static NeighbourList nlist(const StepBuffers& B) { return NeighbourList{B.NL, B.NLC, B.nl_cap, B.STATS}; }
// pass > 0: carried lists (lambda, omega) or recorded bounds (delta-p) of pass `pass`
static Carry carry_of(const StepBuffers& B, uint32_t pass, bool on) {
  return on ? Carry{B.DISP, B.BUILT, B.MODE, B.nl_cap, pass} : Carry{nullptr, nullptr, nullptr, 0u, 0u};
}

// Phases (P.phased) are supported on 2^5-cell tiles with the direct grid; the
// host keeps other phased configurations on the per-particle kernels.
hipError_t launch_tile_lambda(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P,
                              const TileList& T, const StepBuffers& B, const float4* Q, const uint32_t* keys,
                              bool first, bool carry, uint32_t pass) {
  dim3 g(grid), b(kTileThreads);
  const NeighbourList L = nlist(B);
  // the first pass (pass 0) builds every list; the later ones follow `pass` delta-p passes
  // (carried lists hold the bounds of kCarryPasses passes, any other step has any number)
  if (first != (pass == 0) || (carry && (pass > kCarryPasses || !(B.DISP && B.BUILT && B.MODE))))
    return hipErrorInvalidValue;
  const Carry C = carry_of(B, pass, carry);
#define PBD_LAMBDA(BITS_, F_, S_, PH_)                                                                           \
  hipLaunchKernelGGL((k_tile_lambda<BITS_, F_, S_, PH_>), g, b, 0, st, P, T, L, Q, keys, B.cstart, B.cend, B.LAM, \
                     B.DENS, B.NCNT, B.CCNT, C)
#define PBD_LAMBDA_S(BITS_, F_) \
  if (stride) PBD_LAMBDA(BITS_, F_, true, false); \
  else PBD_LAMBDA(BITS_, F_, false, false)
  if (P.phased) {
    if (bits != 5 || stride) return hipErrorInvalidValue;
    if (first) PBD_LAMBDA(5, true, false, true);
    else PBD_LAMBDA(5, false, false, true);
  } else if (bits == 5) {
    if (first) PBD_LAMBDA_S(5, true);
    else PBD_LAMBDA_S(5, false);
  } else {
    if (first) PBD_LAMBDA_S(6, true);
    else PBD_LAMBDA_S(6, false);
  }
#undef PBD_LAMBDA_S
#undef PBD_LAMBDA
  return hipGetLastError();
}

template <int BITS, bool COLLIDE, int NS, bool PH>
static void launch_delta_t(hipStream_t st, uint32_t grid, bool stride, const DevParams& P, const TileList& T,
                           const StepBuffers& B, int use_list, uint32_t flags, const float4* Q, const float4* QX,
                           float4* Qo, float4* QXo, const uint32_t* keys, const Carry& disp) {
  if constexpr (!PH) {
    if (stride) {
      hipLaunchKernelGGL((k_tile_delta<BITS, COLLIDE, NS, true, false>), dim3(grid), dim3(kTileThreads), 0, st, P, T,
                         nlist(B), use_list, flags, Q, QX, B.LAM, keys, B.cstart, B.cend, Qo, QXo, B.DP, B.VS, disp);
      return;
    }
  }
  hipLaunchKernelGGL((k_tile_delta<BITS, COLLIDE, NS, false, PH>), dim3(grid), dim3(kTileThreads), 0, st, P, T,
                     nlist(B), use_list, flags, Q, QX, B.LAM, keys, B.cstart, B.cend, Qo, QXo, B.DP, B.VS, disp);
}

template <int BITS, bool PH>
static void launch_delta_b(hipStream_t st, uint32_t grid, bool stride, const DevParams& P, const TileList& T,
                           const StepBuffers& B, int use_list, uint32_t flags, bool collide, const float4* Q,
                           const float4* QX, float4* Qo, float4* QXo, const uint32_t* keys, const Carry& disp) {
  const bool n4 = P.n_scorr == 4;  // the s_corr exponent of Macklin & Mueller 2013
  if (collide) {
    if (n4) launch_delta_t<BITS, true, 4, PH>(st, grid, stride, P, T, B, use_list, flags, Q, QX, Qo, QXo, keys, disp);
    else launch_delta_t<BITS, true, 0, PH>(st, grid, stride, P, T, B, use_list, flags, Q, QX, Qo, QXo, keys, disp);
  } else {
    if (n4) launch_delta_t<BITS, false, 4, PH>(st, grid, stride, P, T, B, use_list, flags, Q, QX, Qo, QXo, keys, disp);
    else launch_delta_t<BITS, false, 0, PH>(st, grid, stride, P, T, B, use_list, flags, Q, QX, Qo, QXo, keys, disp);
  }
}

hipError_t launch_tile_delta(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P,
                             const TileList& T, const StepBuffers& B, uint32_t flags, bool collide, bool use_list,
                             const float4* Q, const float4* QX, float4* Qo, float4* QXo, const uint32_t* keys,
                             uint32_t track) {
  const int ul = use_list ? 1 : 0;
  if (track > kCarryPasses || (track && !(B.DISP && B.BUILT))) return hipErrorInvalidValue;
  const Carry disp = carry_of(B, track, track != 0);
  if (P.phased) {
    if (bits != 5 || stride) return hipErrorInvalidValue;
    launch_delta_b<5, true>(st, grid, false, P, T, B, ul, flags, collide, Q, QX, Qo, QXo, keys, disp);
  } else if (bits == 5) {
    launch_delta_b<5, false>(st, grid, stride, P, T, B, ul, flags, collide, Q, QX, Qo, QXo, keys, disp);
  } else {
    launch_delta_b<6, false>(st, grid, stride, P, T, B, ul, flags, collide, Q, QX, Qo, QXo, keys, disp);
  }
  return hipGetLastError();
}

hipError_t launch_tile_omega(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P,
                             const TileList& T, const StepBuffers& B, const float4* Q, const uint32_t* keys,
                             bool xsph, uint32_t carry) {
  dim3 g(grid), b(kTileThreads);
  const NeighbourList L = nlist(B);
  if (carry > kCarryPasses || (carry && !(B.DISP && B.BUILT))) return hipErrorInvalidValue;
  const Carry C = carry_of(B, carry, carry != 0);
#define PBD_OMEGA(BITS_, X_, S_, PH_)                                                                             \
  hipLaunchKernelGGL((k_tile_omega<BITS_, X_, S_, PH_>), g, b, 0, st, P, T, L, Q, B.VS, keys, B.cstart, B.cend, B.OM, \
                     B.V, C)
#define PBD_OMEGA_S(BITS_, X_) \
  if (stride) PBD_OMEGA(BITS_, X_, true, false); \
  else PBD_OMEGA(BITS_, X_, false, false)
  if (P.phased) {
    if (bits != 5 || stride) return hipErrorInvalidValue;
    if (xsph) PBD_OMEGA(5, true, false, true);
    else PBD_OMEGA(5, false, false, true);
  } else if (bits == 5) {
    if (xsph) PBD_OMEGA_S(5, true);
    else PBD_OMEGA_S(5, false);
  } else {
    if (xsph) PBD_OMEGA_S(6, true);
    else PBD_OMEGA_S(6, false);
  }
#undef PBD_OMEGA_S
#undef PBD_OMEGA
  return hipGetLastError();
}

hipError_t launch_tile_final(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P,
                             const TileList& T, const StepBuffers& B, uint32_t flags, bool use_list, const float4* Q,
                             const float4* QX, const uint32_t* keys) {
  dim3 g(grid), b(kTileThreads);
  const NeighbourList L = nlist(B);
  const int ul = use_list ? 1 : 0;
  const bool vort = (flags & FF_VORT) != 0, xsph = (flags & FF_XSPH) != 0;
#define PBD_FINAL(BITS_, V_, X_, S_, PH_)                                                                             \
  hipLaunchKernelGGL((k_tile_final<BITS_, V_, X_, S_, PH_>), g, b, 0, st, P, T, L, ul, flags, Q, QX, B.VS, B.OM, keys, \
                     B.cstart, B.cend, B.CS, B.NCNT, B.X, B.P, B.V, B.C, B.F)
#define PBD_FINAL_S(BITS_, V_, X_) \
  if (stride) PBD_FINAL(BITS_, V_, X_, true, false); \
  else PBD_FINAL(BITS_, V_, X_, false, false)
  if (P.phased) {
    if (bits != 5 || stride) return hipErrorInvalidValue;
    if (vort && xsph) PBD_FINAL(5, true, true, false, true);
    else if (vort) PBD_FINAL(5, true, false, false, true);
    else if (xsph) PBD_FINAL(5, false, true, false, true);
    else PBD_FINAL(5, false, false, false, true);
  } else if (bits == 5) {
    if (vort && xsph) PBD_FINAL_S(5, true, true);
    else if (vort) PBD_FINAL_S(5, true, false);
    else if (xsph) PBD_FINAL_S(5, false, true);
    else PBD_FINAL_S(5, false, false);
  } else {
    if (vort && xsph) PBD_FINAL_S(6, true, true);
    else if (vort) PBD_FINAL_S(6, true, false);
    else if (xsph) PBD_FINAL_S(6, false, true);
    else PBD_FINAL_S(6, false, false);
  }
#undef PBD_FINAL_S
#undef PBD_FINAL
  return hipGetLastError();
}

// The wide passes: `grid` workgroups, one per possible work item.
hipError_t launch_wide_lambda(hipStream_t st, uint32_t grid, const DevParams& P, const TileList& T,
                              const StepBuffers& B, const float4* Q, const uint32_t* keys, bool first, bool carry,
                              uint32_t pass) {
  if (first != (pass == 0) || (carry && (pass > kCarryPasses || !(B.DISP && B.BUILT && B.MODE))) || P.phased)
    return hipErrorInvalidValue;
  const Carry C = carry_of(B, pass, carry);
  if (first)
    hipLaunchKernelGGL(k_wide_lambda<true>, dim3(grid), dim3(kWideThreads), 0, st, P, T, nlist(B), Q, keys, B.cstart,
                       B.cend, B.LAM, B.DENS, B.NCNT, B.CCNT, C);
  else
    hipLaunchKernelGGL(k_wide_lambda<false>, dim3(grid), dim3(kWideThreads), 0, st, P, T, nlist(B), Q, keys, B.cstart,
                       B.cend, B.LAM, B.DENS, B.NCNT, B.CCNT, C);
  return hipGetLastError();
}

hipError_t launch_wide_omega(hipStream_t st, uint32_t grid, const DevParams& P, const TileList& T,
                             const StepBuffers& B, const float4* Q, const uint32_t* keys, bool xsph, uint32_t carry) {
  if (carry > kCarryPasses || (carry && !(B.DISP && B.BUILT)) || P.phased) return hipErrorInvalidValue;
  const Carry C = carry_of(B, carry, carry != 0);
  if (xsph)
    hipLaunchKernelGGL(k_wide_omega<true>, dim3(grid), dim3(kWideThreads), 0, st, P, T, nlist(B), Q, B.VS, keys,
                       B.cstart, B.cend, B.OM, B.V, C);
  else
    hipLaunchKernelGGL(k_wide_omega<false>, dim3(grid), dim3(kWideThreads), 0, st, P, T, nlist(B), Q, B.VS, keys,
                       B.cstart, B.cend, B.OM, B.V, C);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Neighbour lists of the reverse passes (adjoint_list.hpp) on tiles.  The
// halo of a 2^BITS-cell block is copied to LDS once, and one thread per own
// particle walks its 27 cells there in stencil order (threads of one cell read
// the same slots; each (x, y) column's three z cells as one slot range),
// dealing the candidates within the list radius to its lanes in turn: entry c
// to lane c mod kAdjLanes.  The lanes hold other shares of the
// candidates than a scan's, so the reverse passes add the same terms in
// another order.  A particle with more than kAdjLanes x kAdjListMax is marked
// kAdjScan; a block whose halo exceeds the LDS capacity uses adj_list_lane.
static_assert(kAdjLanes == 8, "the tile list builder writes rows of 8 entries as two 16-byte stores");

// The list builders tally their counters per workgroup in LDS (tally[0]:
// PBD_COUNTER_ADJ_LISTED_TILE, [1]: PBD_COUNTER_ADJ_SCANNED, [2]:
// PBD_COUNTER_ADJ_FROM_FORWARD) and add them to the context's once at the end:
// atomics on one address from every wave would queue in the L2.
constexpr uint32_t kAdjTallies = 3;
__device__ __forceinline__ void wave_tally(uint32_t* t, bool pred) {
  const uint64_t m = __ballot(pred);
  const uint64_t act = __ballot(true);
  if (m && (uint32_t)(__ffsll((unsigned long long)act) - 1) == (threadIdx.x & 63u)) atomicAdd(t, (uint32_t)__popcll(m));
}
__device__ __forceinline__ void tally_begin(uint32_t* t) {
  if (threadIdx.x < kAdjTallies) t[threadIdx.x] = 0u;
}
// The halo's .w for the list builders: 1 for a solid particle of a phased step
// (P.phs), whose entries carry kAdjSolid.
__device__ __forceinline__ auto adj_solid_payload(const DevParams& P) {
  const uint32_t* ph = P.phs;
  return [ph](uint32_t gi) { return ph && ph[gi] ? 1.0f : 0.0f; };
}
__device__ __forceinline__ uint32_t adj_solid_bit(const DevParams& P, const float4* s_q, uint32_t slot) {
  return P.phs && s_q[slot].w != 0.0f ? kAdjSolid : 0u;
}
// after a barrier that follows the last wave_tally
__device__ __forceinline__ void tally_flush(const uint32_t* t, unsigned long long* stats) {
  constexpr uint32_t kCounter[kAdjTallies] = {PBD_COUNTER_ADJ_LISTED_TILE, PBD_COUNTER_ADJ_SCANNED,
                                              PBD_COUNTER_ADJ_FROM_FORWARD};
  if (stats && threadIdx.x < kAdjTallies && t[threadIdx.x])
    atomicAdd(stats + kCounter[threadIdx.x], (unsigned long long)t[threadIdx.x]);
}

// In-range bits (lo, hi) of slots a .. b - 1 (1 <= b - a <= 64).  Four candidates a group:
// these builders keep a window of entries and two masks beside them, and eight take them
// from four waves a SIMD to three (165 VGPRs; the reverse of two substeps of 729K particles
// with its lists built here 4520 us, 4410 so with the team's opaque index).
__device__ __forceinline__ void nl_column(const float4* s_q, uint32_t a, uint32_t b, float4 q, float r2max,
                                          uint32_t& lo, uint32_t& hi) {
  const uint32_t valid = fabsf(q.x) + fabsf(q.y) + fabsf(q.z) < __builtin_inff() ? 0xFFFFFFFFu : 0u;
  const uint32_t len = b - a;
  lo = nl_mask<4u>(s_q, a, min(len, 32u), q.x, q.y, q.z, r2max) & valid;
  hi = len > 32u ? nl_mask<4u>(s_q, a + 32u, len - 32u, q.x, q.y, q.z, r2max) & valid : 0u;
}

// One particle's list: entries dealt to its lanes in turn, the last kAdjLanes
// of them in a shift window w[0..7]; each full row (entries 8k .. 8k+7, one per
// lane) is written as 32 bytes, and rows past kAdjListMax are dropped (the
// particle is then marked kAdjScan).
struct AdjRows {
  static constexpr uint32_t kMax = kAdjLanes * kAdjListMax;
  uint32_t w[kAdjLanes];
  uint32_t c = 0;
  uint32_t* e;  // the lists (AdjList::e) of n particles; this is particle g's
  uint32_t n, g;
  __device__ __forceinline__ AdjRows(const AdjList& L, uint32_t n_, uint32_t g_) : e(L.e), n(n_), g(g_) {
#pragma unroll
    for (uint32_t i = 0; i < kAdjLanes; ++i) w[i] = 0u;
  }
  __device__ __forceinline__ void put_row(uint32_t row) {
    uint4* dst = reinterpret_cast<uint4*>(e + ((size_t)row * n + g) * kAdjLanes);
    dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
    dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
  }
  __device__ __forceinline__ void push(uint32_t entry) {
#pragma unroll
    for (uint32_t i = 0; i + 1 < kAdjLanes; ++i) w[i] = w[i + 1];
    w[kAdjLanes - 1] = entry;
    ++c;
    if ((c & (kAdjLanes - 1u)) == 0u && c <= kMax) put_row(c / kAdjLanes - 1u);
  }
  // the last, partial row (its r entries to lanes 0 .. r-1) and the lane counts
  __device__ __forceinline__ void finish(const AdjList& L, uint32_t g) {
    const uint32_t r = c & (kAdjLanes - 1u);
    if (r != 0u && c < kMax) {
      for (uint32_t i = r; i < kAdjLanes; ++i) {
#pragma unroll
        for (uint32_t k = 0; k + 1 < kAdjLanes; ++k) w[k] = w[k + 1];
        w[kAdjLanes - 1] = 0u;
      }
      put_row(c / kAdjLanes);
    }
    uint32_t cl[kAdjLanes];
#pragma unroll
    for (uint32_t lane = 0; lane < kAdjLanes; ++lane) cl[lane] = c > kMax ? kAdjScan : (c + kAdjLanes - 1u - lane) / kAdjLanes;
    uint4* cdst = reinterpret_cast<uint4*>(L.cnt + (size_t)g * kAdjLanes);
    cdst[0] = make_uint4(cl[0], cl[1], cl[2], cl[3]);
    cdst[1] = make_uint4(cl[4], cl[5], cl[6], cl[7]);
  }
};

// The list of own particle g (halo cell h, LDS slot `slot`) from the halo in
// LDS, as adjlist_tile builds it.  Per (x, y) column the three z cells are one slot range [a0, e), tested
// 64 slots at a time into in-range masks (branch-free, nl_column); the in-range
// slots are then pushed in slot order.  A slot's z offset and sorted index
// follow from a1, a2.  Returns the number of candidates in range.
template <int BITS>
__device__ __forceinline__ uint32_t adjlist_particle(const DevParams& P, const TileShared<BITS>& sh,
                                                     const float4* s_q, const AdjList& L, uint32_t g, int h,
                                                     uint32_t slot) {
  using G = TileGeom<BITS>;
  const float4 qb = s_q[slot];
  AdjRows R(L, P.n, g);
#pragma unroll
  for (int dx = -1; dx <= 1; ++dx) {
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy) {
      const int hb = h + dx * G::SX + dy * G::SY;
      const uint32_t a0 = sh.lstart[hb - 1], a1 = sh.lstart[hb], a2 = sh.lstart[hb + 1], e = sh.lstart[hb + 2];
      const uint32_t b0 = sh.gstart[hb - 1] - a0, b1 = sh.gstart[hb] - a1, b2 = sh.gstart[hb + 1] - a2;
      const uint32_t oc = (uint32_t)((dx + 1) * 9 + (dy + 1) * 3);
      for (uint32_t s0 = a0; s0 < e; s0 += 64u) {
        uint32_t lo, hi;
        nl_column(s_q, s0, e < s0 + 64u ? e : s0 + 64u, qb, P.list_r2, lo, hi);
        const uint32_t k = slot - s0;  // the particle itself (when in this segment)
        if (k < 32u) lo &= ~(1u << k);
        else if (k < 64u) hi &= ~(1u << (k - 32u));
#pragma unroll
        for (uint32_t half = 0; half < 2u; ++half) {
          uint32_t m = half ? hi : lo;
          while (m) {
            const uint32_t j = s0 + 32u * half + (uint32_t)__builtin_ctz(m);
            m &= m - 1u;
            const uint32_t z = j < a1 ? 0u : (j < a2 ? 1u : 2u);
            const uint32_t base = z == 0u ? b0 : (z == 1u ? b1 : b2);  // sorted index of slot j: base + j
            R.push((base + j) | ((oc + z) << 27) | adj_solid_bit(P, s_q, j));
          }
        }
      }
    }
  }
  R.finish(L, g);
  return R.c;
}

template <int BITS>
__device__ __forceinline__ void adjlist_tile(const DevParams& P, uint32_t blk, const float4* __restrict__ Q,
                                             const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                                             const uint32_t* __restrict__ ce, const AdjList& L,
                                             uint32_t* __restrict__ flag, unsigned long long* __restrict__ stats,
                                             uint32_t* tally, TileShared<BITS>& sh, float4* s_q) {
  using G = TileGeom<BITS>;
  constexpr int CAP = TileCap<BITS>::adjoint;
  constexpr uint32_t kMax = kAdjLanes * kAdjListMax;
  const uint32_t total = tile_setup<BITS, TeamBlockN<kTileThreads, true>>(P, blk, cs, ce, sh);
  const uint32_t g0 = sh.g0, g1 = sh.g1;
  if (total > (uint32_t)CAP) {
    // whole particles per pass of the loop: a particle's lanes are active together
    const uint32_t m = (g1 - g0) * kAdjLanes;
    for (uint32_t u = threadIdx.x; u < m; u += kTileThreads)
      adj_list_lane(P, Q, keys, cs, ce, L, flag, stats, g0 + u / kAdjLanes, u % kAdjLanes);
    return;
  }
  tile_load<BITS, CAP, TeamBlockN<kTileThreads, true>>(P, sh, total, Q, s_q, nullptr, 0u, adj_solid_payload(P));
  __syncthreads();
  const uint32_t n = P.n;
  for (uint32_t g = g0 + threadIdx.x; g < g1; g += kTileThreads) {
    int h;
    uint32_t slot;
    tile_locate<BITS>(sh, keys[g], g, h, slot);
    const float4 qb = s_q[slot];
    // the last kAdjLanes entries in a shift window w[0..7]; each full row of
    // the list (entries 8k .. 8k+7, one per lane) is written as 32 bytes
    uint32_t w[kAdjLanes];
#pragma unroll
    for (uint32_t i = 0; i < kAdjLanes; ++i) w[i] = 0u;
    const auto put_row = [&](uint32_t row) {
      uint4* dst = reinterpret_cast<uint4*>(L.e + ((size_t)row * n + g) * kAdjLanes);
      dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
      dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
    };
    uint32_t c = 0;
    const auto push = [&](uint32_t entry) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t i = 0; i + 1 < kAdjLanes; ++i) w[i] = w[i + 1];
      w[kAdjLanes - 1] = entry;
      ++c;
      if ((c & (kAdjLanes - 1u)) == 0u && c <= kMax) put_row(c / kAdjLanes - 1u);
    };
    // per (x, y) column the three z cells are one slot range [a0, e), tested 64
    // slots at a time into in-range masks (branch-free, nl_column); the in-range
    // slots are then pushed in slot order.  A slot's z offset and sorted index
    // follow from a1, a2.
#pragma unroll
    for (int dx = -1; dx <= 1; ++dx) {
#pragma unroll
      for (int dy = -1; dy <= 1; ++dy) {
        const int hb = h + dx * G::SX + dy * G::SY;
        const uint32_t a0 = sh.lstart[hb - 1], a1 = sh.lstart[hb], a2 = sh.lstart[hb + 1], e = sh.lstart[hb + 2];
        const uint32_t b0 = sh.gstart[hb - 1] - a0, b1 = sh.gstart[hb] - a1, b2 = sh.gstart[hb + 1] - a2;
        const uint32_t oc = (uint32_t)((dx + 1) * 9 + (dy + 1) * 3);
        for (uint32_t s0 = a0; s0 < e; s0 += 64u) {
          uint32_t lo, hi;
          nl_column(s_q, s0, e < s0 + 64u ? e : s0 + 64u, qb, P.list_r2, lo, hi);
          const uint32_t k = slot - s0;  // the particle itself (when in this segment)
          if (k < 32u) lo &= ~(1u << k);
          else if (k < 64u) hi &= ~(1u << (k - 32u));
#pragma unroll
          for (uint32_t half = 0; half < 2u; ++half) {
            uint32_t m = half ? hi : lo;
            while (m) {
              const uint32_t j = s0 + 32u * half + (uint32_t)__builtin_ctz(m);
              m &= m - 1u;
              const uint32_t z = j < a1 ? 0u : (j < a2 ? 1u : 2u);
              const uint32_t base = z == 0u ? b0 : (z == 1u ? b1 : b2);  // sorted index of slot j: base + j
              push((base + j) | ((oc + z) << 27) | adj_solid_bit(P, s_q, j));
            }
          }
        }
      }
    }
    const uint32_t r = c & (kAdjLanes - 1u);
    if (r != 0u && c < kMax) {  // the last, partial row: its r entries to lanes 0 .. r-1
      for (uint32_t i = r; i < kAdjLanes; ++i) {
#pragma unroll
        for (uint32_t k = 0; k + 1 < kAdjLanes; ++k) w[k] = w[k + 1];
        w[kAdjLanes - 1] = 0u;
      }
      put_row(c / kAdjLanes);
    }
    uint32_t cl[kAdjLanes];
#pragma unroll
    for (uint32_t lane = 0; lane < kAdjLanes; ++lane) cl[lane] = c > kMax ? kAdjScan : (c + kAdjLanes - 1u - lane) / kAdjLanes;
    uint4* cdst = reinterpret_cast<uint4*>(L.cnt + (size_t)g * kAdjLanes);
    cdst[0] = make_uint4(cl[0], cl[1], cl[2], cl[3]);
    cdst[1] = make_uint4(cl[4], cl[5], cl[6], cl[7]);
    if (tile_count<BITS>(sh, h) >= P.cap) flag[0] = 1u;
    wave_tally(tally + 0, c <= kMax);
    wave_tally(tally + 1, c > kMax);
  }
}

// The lists of one block taken from the forward's tile lists of the same
// positions (F: those a recorded step's lambda pass built for an iteration,
// without a skin, or its omega pass for the final positions, on the same
// 2^BITS-cell blocks).  A forward list holds the candidates within the list
// radius in stencil-column then slot order, the order adjlist_particle deals
// them to the lanes in, so the lists come out the same without the halo's
// positions or a distance test: only the block's cell table is set up (the
// omega pass leaves a solid particle's list empty: the reverse passes read no
// pair of a solid particle at the final positions).  The
// slots of a list increase, so a walk over the nine columns gives each slot's
// halo cell; slots at or past the halo size are the forward's padding, and the
// forward's solid bit becomes kAdjSolid.  A particle without a forward list
// (over the neighbour cap, more pairs than a forward list holds, or in a tile or half
// beyond its capacity) is left to k_tile_adjlist_redo, and so is a block beyond the
// builders' capacity: the block is appended to redo (redo[0]: the count).  A block beyond
// the tile capacity is taken as its two halves, whose cell tables the forward's slots
// count in (all of it left to the redo pass, the reverse of two substeps of 729K particles
// at 1.6 times their rest density took 18.8 ms, as halves 14.2).
//
// adjlist_forward_tile: a thread per particle, which deals the entries as
// adjlist_particle does.
template <int BITS>
__device__ __forceinline__ void adjlist_forward_tile(const DevParams& P, uint32_t blk,
                                                     const uint32_t* __restrict__ keys,
                                                     const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                                                     const NeighbourList& F, const AdjList& L,
                                                     uint32_t* __restrict__ flag, uint32_t* tally,
                                                     uint32_t* __restrict__ redo, TileShared<BITS>& sh) {
  using G = TileGeom<BITS>;
  constexpr int CAP = TileCap<BITS>::value;
  uint32_t total = tile_setup<BITS, TeamBlockN<kTileThreads, true>>(P, blk, cs, ce, sh);
  if (total > (uint32_t)TileCap<BITS>::adjoint) {
    if (threadIdx.x == 0) redo[1u + atomicAdd(redo, 1u)] = blk;
    return;
  }
  const uint32_t last = total > (uint32_t)CAP ? 2u : 0u;
  int missing = 0;
#pragma unroll 1
  for (uint32_t half = last ? 1u : 0u; half <= last; ++half) {
    if (half) {
      __syncthreads();
      total = tile_setup<BITS, TeamBlockN<kTileThreads, true>>(P, blk, cs, ce, sh, NoLoads(), half);
    }
    const uint32_t g0 = sh.g0, g1 = sh.g1;
    if (g0 >= g1) continue;  // an empty half
    for (uint32_t g = g0 + threadIdx.x; g < g1; g += kTileThreads) {
      const uint32_t fn = F.cnt[g];
      if (fn == kNlInvalid) {
        missing = 1;
        continue;
      }
      int h;
      uint32_t slot;
      tile_locate<BITS>(sh, keys[g], g, h, slot);
      AdjRows R(L, P.n, g);
      if (fn > AdjRows::kMax) {
        R.c = AdjRows::kMax + 1u;  // more candidates than the lanes hold: scan
      } else {
        // column `col` (dx = col / 3 - 1, dy = col % 3 - 1): slots [a0, e), z cells from a1, a2
        int col = 0;
        uint32_t a1 = 0, a2 = 0, e = 0, b0 = 0, b1 = 0, b2 = 0, oc = 0;
        const auto column = [&](int c3) __attribute__((always_inline)) {
          const int hb = h + (c3 / 3 - 1) * G::SX + (c3 % 3 - 1) * G::SY;
          const uint32_t a0 = sh.lstart[hb - 1];
          a1 = sh.lstart[hb];
          a2 = sh.lstart[hb + 1];
          e = sh.lstart[hb + 2];
          b0 = sh.gstart[hb - 1] - a0;
          b1 = sh.gstart[hb] - a1;
          b2 = sh.gstart[hb + 1] - a2;
          oc = (uint32_t)((c3 / 3) * 9 + (c3 % 3) * 3);
        };
        column(0);
        // chunk k + 1 is loaded while chunk k is taken apart
        const uint4* p = F.nl + g;
        const uint32_t nc = fn / 8u;
        bool done = nc == 0u;
        uint4 v = nc ? p[0] : make_uint4(0u, 0u, 0u, 0u);
        for (uint32_t k = 0; k < nc && !done; ++k) {
          uint4 nx = v;  // as nl_visit
          if (k + 1u < nc) nx = p[(size_t)(k + 1u) * F.cap];
          const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
          v = nx;
#pragma unroll
          for (uint32_t i = 0; i < 8u; ++i) {
            const uint32_t raw = (wd[i / 2u] >> (16u * (i & 1u))) & 0xFFFFu;
            const uint32_t j = raw & (kNlSolid - 1u);
            if (done || j >= total) {  // the padding, after the last entry
              done = true;
              continue;
            }
            while (j >= e && col < 8) column(++col);
            const uint32_t z = j < a1 ? 0u : (j < a2 ? 1u : 2u);
            const uint32_t base = z == 0u ? b0 : (z == 1u ? b1 : b2);
            R.push((base + j) | ((oc + z) << 27) | ((raw & kNlSolid) ? kAdjSolid : 0u));
          }
        }
      }
      R.finish(L, g);
      if (tile_count<BITS>(sh, h) >= P.cap) flag[0] = 1u;
      wave_tally(tally + 0, R.c <= AdjRows::kMax);
      wave_tally(tally + 1, R.c > AdjRows::kMax);
      wave_tally(tally + 2, true);
    }
  }
  if (__syncthreads_or(missing) && threadIdx.x == 0) redo[1u + atomicAdd(redo, 1u)] = blk;
}

// adjlist_forward_tile_wide, for scenes whose blocks are too few to fill the
// CUs with a thread per particle: entry c goes to lane c mod 8 of row c / 8,
// so chunk k of a forward list (its entries 8k .. 8k+7) is row k, and a thread
// per (particle, chunk) converts one row.  It finds the column of the chunk's
// first slot, then walks the columns with the slots; the padding is zero in
// the row, as in the builder's last row.  The thread of a particle's last
// chunk writes the lane counts.
template <int BITS>
__device__ __forceinline__ void adjlist_forward_tile_wide(const DevParams& P, uint32_t blk,
                                                          const uint32_t* __restrict__ keys,
                                                     const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                                                     const NeighbourList& F, const AdjList& L,
                                                     uint32_t* __restrict__ flag, uint32_t* tally,
                                                     uint32_t* __restrict__ redo, TileShared<BITS>& sh) {
  using G = TileGeom<BITS>;
  constexpr int CAP = TileCap<BITS>::value;
  static_assert(kNlRecordChunks == kAdjLanes && kAdjListMax == kAdjLanes, "a forward chunk is a row of the lanes");
  uint32_t total = tile_setup<BITS, TeamBlockN<kWideThreads, true>>(P, blk, cs, ce, sh);
  if (total > (uint32_t)TileCap<BITS>::adjoint) {
    if (threadIdx.x == 0) redo[1u + atomicAdd(redo, 1u)] = blk;
    return;
  }
  const uint32_t n = P.n, last = total > (uint32_t)CAP ? 2u : 0u;
  int missing = 0;
#pragma unroll 1
  for (uint32_t half = last ? 1u : 0u; half <= last; ++half) {
    if (half) {
      __syncthreads();
      total = tile_setup<BITS, TeamBlockN<kWideThreads, true>>(P, blk, cs, ce, sh, NoLoads(), half);
    }
    const uint32_t g0 = sh.g0, g1 = sh.g1;
    if (g0 >= g1) continue;  // an empty half
    for (uint32_t u = threadIdx.x; u < (g1 - g0) * kAdjLanes; u += kWideThreads) {
      const uint32_t g = g0 + u / kAdjLanes, k = u % kAdjLanes;
      const uint32_t fn = F.cnt[g];
      if (fn == kNlInvalid) {
        missing = 1;
        continue;
      }
      const uint32_t nc = fn / 8u;
      // the thread that writes the counts: the last chunk's, or chunk 0's without a row
      const bool counter = fn > AdjRows::kMax || nc == 0u ? k == 0u : k + 1u == nc;
      uint32_t c = 0;
      int h = 0;
      if (fn <= AdjRows::kMax && k < nc) {
        uint32_t slot;
        tile_locate<BITS>(sh, keys[g], g, h, slot);
        const uint4 v = F.nl[(size_t)k * F.cap + g];
        const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
        int col = -1;
        uint32_t a1 = 0, a2 = 0, e = 0, b0 = 0, b1 = 0, b2 = 0, oc = 0;
        const auto column = [&](int c3) __attribute__((always_inline)) {
          const int hb = h + (c3 / 3 - 1) * G::SX + (c3 % 3 - 1) * G::SY;
          const uint32_t a0 = sh.lstart[hb - 1];
          a1 = sh.lstart[hb];
          a2 = sh.lstart[hb + 1];
          e = sh.lstart[hb + 2];
          b0 = sh.gstart[hb - 1] - a0;
          b1 = sh.gstart[hb] - a1;
          b2 = sh.gstart[hb + 1] - a2;
          oc = (uint32_t)((c3 / 3) * 9 + (c3 % 3) * 3);
        };
        column(++col);
        uint32_t w[kAdjLanes];
#pragma unroll
        for (uint32_t i = 0; i < kAdjLanes; ++i) {
          const uint32_t raw = (wd[i / 2u] >> (16u * (i & 1u))) & 0xFFFFu;
          const uint32_t j = raw & (kNlSolid - 1u);
          w[i] = 0u;
          if (j >= total) continue;  // the padding, after the last entry
          ++c;
          while (j >= e && col < 8) column(++col);
          const uint32_t z = j < a1 ? 0u : (j < a2 ? 1u : 2u);
          const uint32_t base = z == 0u ? b0 : (z == 1u ? b1 : b2);
          w[i] = (base + j) | ((oc + z) << 27) | ((raw & kNlSolid) ? kAdjSolid : 0u);
        }
        uint4* dst = reinterpret_cast<uint4*>(L.e + ((size_t)k * n + g) * kAdjLanes);
        dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
        dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
      }
      if (counter) {
        if (fn > AdjRows::kMax) {
          c = AdjRows::kMax + 1u;  // more candidates than the lanes hold: scan
        } else if (nc) {
          c += 8u * (nc - 1u);
        }
        uint32_t cl[kAdjLanes];
#pragma unroll
        for (uint32_t lane = 0; lane < kAdjLanes; ++lane)
          cl[lane] = c > AdjRows::kMax ? kAdjScan : (c + kAdjLanes - 1u - lane) / kAdjLanes;
        uint4* cdst = reinterpret_cast<uint4*>(L.cnt + (size_t)g * kAdjLanes);
        cdst[0] = make_uint4(cl[0], cl[1], cl[2], cl[3]);
        cdst[1] = make_uint4(cl[4], cl[5], cl[6], cl[7]);
        if (fn > AdjRows::kMax || nc == 0u) {
          uint32_t slot;
          tile_locate<BITS>(sh, keys[g], g, h, slot);
        }
        if (tile_count<BITS>(sh, h) >= P.cap) flag[0] = 1u;
      }
      wave_tally(tally + 0, counter && c <= AdjRows::kMax);
      wave_tally(tally + 1, counter && c > AdjRows::kMax);
      wave_tally(tally + 2, counter);
    }
  }
  if (__syncthreads_or(missing) && threadIdx.x == 0) redo[1u + atomicAdd(redo, 1u)] = blk;
}

// The blocks adjlist_forward_tile appended to redo: its particles without a
// forward list built by adjlist_particle on the block's halo, or, in a block
// beyond the tile capacity, every particle by adj_list_lane.
template <int BITS>
__global__ __launch_bounds__(kTileThreads, 4) void k_tile_adjlist_redo(DevParams P, const float4* __restrict__ Q,
                                                                    const uint32_t* __restrict__ keys,
                                                                    const uint32_t* __restrict__ cs,
                                                                    const uint32_t* __restrict__ ce, NeighbourList F,
                                                                    AdjList L, uint32_t* __restrict__ flag,
                                                                    unsigned long long* __restrict__ stats,
                                                                    const uint32_t* __restrict__ redo) {
  constexpr int CAP = TileCap<BITS>::adjoint;
  __shared__ TileRegion<BITS, TileCap<BITS>::adjoint, false> lds;
  __shared__ uint32_t s_tally[kAdjTallies];
  tally_begin(s_tally);
  const uint32_t count = redo[0];
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    __syncthreads();  // the previous block's halo is done with (and the tallies are cleared)
    TileShared<BITS>& sh = lds.sh;
    float4* s_q = lds.q;
    const uint32_t total = tile_setup<BITS, TeamBlockN<kTileThreads, true>>(P, redo[1u + i], cs, ce, sh);
    if (total > (uint32_t)CAP) {
      const uint32_t m = (sh.g1 - sh.g0) * kAdjLanes;
      for (uint32_t u = threadIdx.x; u < m; u += kTileThreads)
        adj_list_lane(P, Q, keys, cs, ce, L, flag, stats, sh.g0 + u / kAdjLanes, u % kAdjLanes);
      continue;
    }
    tile_load<BITS, CAP, TeamBlockN<kTileThreads, true>>(P, sh, total, Q, s_q, nullptr, 0u, adj_solid_payload(P));
    __syncthreads();
    for (uint32_t g = sh.g0 + threadIdx.x; g < sh.g1; g += kTileThreads) {
      if (F.cnt[g] != kNlInvalid) continue;  // converted
      int h;
      uint32_t slot;
      tile_locate<BITS>(sh, keys[g], g, h, slot);
      const uint32_t c = adjlist_particle<BITS>(P, sh, s_q, L, g, h, slot);
      if (tile_count<BITS>(sh, h) >= P.cap) flag[0] = 1u;
      wave_tally(s_tally + 0, c <= AdjRows::kMax);
      wave_tally(s_tally + 1, c > AdjRows::kMax);
    }
  }
  __syncthreads();
  tally_flush(s_tally, stats);
}

// The same lists for small scenes, whose blocks are too few to fill the CUs
// with one thread per particle: a 1024-thread workgroup, four threads per
// particle (part k of the 9 stencil columns: 0-2, 3-4, 5-6, 7-8).  Each thread
// keeps its columns' in-range masks (the first 64-slot segment of each; longer
// columns are tested again when written), the parts' entry counts are combined
// in LDS into offsets, and every entry is written at its index in the list of
// the one-thread builder: the lists are identical.
constexpr uint32_t kWideParts = kWideThreads / kTileThreads;
static_assert(kWideParts == 4, "four threads per particle");
template <int BITS>
__device__ __forceinline__ void adjlist_tile_wide(const DevParams& P, uint32_t blk, const float4* __restrict__ Q,
                                                  const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                                                  const uint32_t* __restrict__ ce, const AdjList& L,
                                                  uint32_t* __restrict__ flag, unsigned long long* __restrict__ stats,
                                                  uint32_t* tally, TileShared<BITS>& sh, float4* s_q,
                                                  uint32_t (*s_part)[kTileThreads]) {
  using G = TileGeom<BITS>;
  constexpr int CAP = TileCap<BITS>::adjoint;
  constexpr uint32_t kMax = kAdjLanes * kAdjListMax;
  const uint32_t total = tile_setup<BITS, TeamBlockN<kWideThreads, true>>(P, blk, cs, ce, sh);
  const uint32_t g0 = sh.g0, g1 = sh.g1;
  if (total > (uint32_t)CAP) {
    const uint32_t m = (g1 - g0) * kAdjLanes;
    for (uint32_t u = threadIdx.x; u < m; u += kWideThreads)
      adj_list_lane(P, Q, keys, cs, ce, L, flag, stats, g0 + u / kAdjLanes, u % kAdjLanes);
    return;
  }
  tile_load<BITS, CAP, TeamBlockN<kWideThreads, true>>(P, sh, total, Q, s_q, nullptr, 0u, adj_solid_payload(P));
  __syncthreads();
  const uint32_t n = P.n;
  const uint32_t part = threadIdx.x / kTileThreads, pl = threadIdx.x % kTileThreads;
  const int cbeg = part == 0u ? 0 : 1 + 2 * (int)part, cend = part == 0u ? 3 : 3 + 2 * (int)part;
  // every thread of the workgroup takes each round (the counts are exchanged)
  for (uint32_t base = g0; base < g1; base += kTileThreads) {
    const uint32_t g = base + pl;
    const bool valid = g < g1;
    int h = 0;
    uint32_t slot = 0;
    float4 qb = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t lo[3] = {0u, 0u, 0u}, hi[3] = {0u, 0u, 0u}, cnt = 0;
    if (valid) {
      tile_locate<BITS>(sh, keys[g], g, h, slot);
      qb = s_q[slot];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int c = cbeg + k;
        if (c >= cend) break;
        const int hb = h + (c / 3 - 1) * G::SX + (c % 3 - 1) * G::SY;
        const uint32_t a0 = sh.lstart[hb - 1], e = sh.lstart[hb + 2];
        for (uint32_t s0 = a0; s0 < e; s0 += 64u) {
          uint32_t l, u;
          nl_column(s_q, s0, e < s0 + 64u ? e : s0 + 64u, qb, P.list_r2, l, u);
          const uint32_t d = slot - s0;  // the particle itself (when in this segment)
          if (d < 32u) l &= ~(1u << d);
          else if (d < 64u) u &= ~(1u << (d - 32u));
          if (s0 == a0) {
            lo[k] = l;
            hi[k] = u;
          }
          cnt += __builtin_popcount(l) + __builtin_popcount(u);
        }
      }
    }
    s_part[part][pl] = cnt;
    __syncthreads();
    uint32_t off = 0, all = 0;
#pragma unroll
    for (uint32_t k = 0; k < kWideParts; ++k) {
      const uint32_t v = s_part[k][pl];
      off += k < part ? v : 0u;
      all += v;
    }
    if (valid) {
      uint32_t c = off;
      const auto put = [&](uint32_t entry) __attribute__((always_inline)) {
        if (c < kMax) L.e[((size_t)(c / kAdjLanes) * n + g) * kAdjLanes + c % kAdjLanes] = entry;
        ++c;
      };
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int col = cbeg + k;
        if (col >= cend) break;
        const int dx = col / 3 - 1, dy = col % 3 - 1;
        const int hb = h + dx * G::SX + dy * G::SY;
        const uint32_t a0 = sh.lstart[hb - 1], a1 = sh.lstart[hb], a2 = sh.lstart[hb + 1], e = sh.lstart[hb + 2];
        const uint32_t b0 = sh.gstart[hb - 1] - a0, b1 = sh.gstart[hb] - a1, b2 = sh.gstart[hb + 1] - a2;
        const uint32_t oc = (uint32_t)((dx + 1) * 9 + (dy + 1) * 3);
        for (uint32_t s0 = a0; s0 < e; s0 += 64u) {
          uint32_t l = lo[k], u = hi[k];
          if (s0 != a0) {  // a column of more than 64 slots: its later segments again
            nl_column(s_q, s0, e < s0 + 64u ? e : s0 + 64u, qb, P.list_r2, l, u);
            const uint32_t d = slot - s0;
            if (d < 32u) l &= ~(1u << d);
            else if (d < 64u) u &= ~(1u << (d - 32u));
          }
#pragma unroll
          for (uint32_t half = 0; half < 2u; ++half) {
            uint32_t m = half ? u : l;
            while (m) {
              const uint32_t j = s0 + 32u * half + (uint32_t)__builtin_ctz(m);
              m &= m - 1u;
              const uint32_t z = j < a1 ? 0u : (j < a2 ? 1u : 2u);
              const uint32_t b = z == 0u ? b0 : (z == 1u ? b1 : b2);  // sorted index of slot j: b + j
              put((b + j) | ((oc + z) << 27) | adj_solid_bit(P, s_q, j));
            }
          }
        }
      }
      if (part == 0u) {
        uint32_t cl[kAdjLanes];
#pragma unroll
        for (uint32_t lane = 0; lane < kAdjLanes; ++lane)
          cl[lane] = all > kMax ? kAdjScan : (all + kAdjLanes - 1u - lane) / kAdjLanes;
        uint4* cdst = reinterpret_cast<uint4*>(L.cnt + (size_t)g * kAdjLanes);
        cdst[0] = make_uint4(cl[0], cl[1], cl[2], cl[3]);
        cdst[1] = make_uint4(cl[4], cl[5], cl[6], cl[7]);
        if (tile_count<BITS>(sh, h) >= P.cap) flag[0] = 1u;
      }
    }
    if (part == 0u) {
      wave_tally(tally + 0, valid && all <= kMax);
      wave_tally(tally + 1, valid && all > kMax);
    }
    __syncthreads();  // s_part is written again by the next round
  }
}

template <int BITS>
__global__ __launch_bounds__(kWideThreads) void k_tile_adjlist_wide(DevParams P, uint32_t nblocks, uint32_t table,
                                                                    const float4* __restrict__ Q,
                                                                    const uint32_t* __restrict__ keys,
                                                                    const uint32_t* __restrict__ cs,
                                                                    const uint32_t* __restrict__ ce, AdjList L,
                                                                    uint32_t* __restrict__ flag,
                                                                    unsigned long long* __restrict__ stats) {
  __shared__ TileRegion<BITS, TileCap<BITS>::adjoint, false> lds;
  __shared__ uint32_t s_part[kWideParts][kTileThreads];
  __shared__ uint32_t s_occ;
  __shared__ uint32_t s_tally[kAdjTallies];
  constexpr uint32_t kCells = 1u << BITS;
  constexpr uint32_t kPer = kWideThreads / kCells;
  static_assert(kPer <= 32u, "occupancy bits of one batch");
  tally_begin(s_tally);
  for (uint32_t i0 = 0; blockIdx.x + i0 * gridDim.x < nblocks; i0 += kPer) {
    if (threadIdx.x == 0) s_occ = 0u;
    __syncthreads();
    const uint32_t k = threadIdx.x / kCells;
    const uint32_t b = blockIdx.x + (i0 + k) * gridDim.x;
    const uint32_t cell = b * kCells + threadIdx.x % kCells;
    if (b < nblocks && cell < table && cs[cell] != 0xFFFFFFFFu) atomicOr(&s_occ, 1u << k);
    __syncthreads();
    const uint32_t occ = s_occ;
    for (uint32_t i = 0; i < kPer; ++i) {
      if (!((occ >> i) & 1u)) continue;
      adjlist_tile_wide<BITS>(P, blockIdx.x + (i0 + i) * gridDim.x, Q, keys, cs, ce, L, flag, stats, s_tally,
                              lds.sh, lds.q, s_part);
      __syncthreads();
    }
    __syncthreads();
  }
  __syncthreads();
  tally_flush(s_tally, stats);
}

// Workgroup w takes the blocks w + i gridDim.x, kTileThreads / 2^BITS of them
// at a time, finds the occupied ones from their own cells' starts and builds
// those one by one; interleaved so that the occupied blocks, which lie in a
// few Morton ranges, spread over all workgroups.
template <int BITS>
__global__ __launch_bounds__(kTileThreads, 4) void k_tile_adjlist(DevParams P, uint32_t nblocks, uint32_t table,
                                                               const float4* __restrict__ Q,
                                                               const uint32_t* __restrict__ keys,
                                                               const uint32_t* __restrict__ cs,
                                                               const uint32_t* __restrict__ ce, AdjList L,
                                                               uint32_t* __restrict__ flag,
                                                               unsigned long long* __restrict__ stats) {
  __shared__ TileRegion<BITS, TileCap<BITS>::adjoint, false> lds;
  __shared__ uint32_t s_occ;
  __shared__ uint32_t s_tally[kAdjTallies];
  constexpr uint32_t kCells = 1u << BITS;
  constexpr uint32_t kPer = kTileThreads / kCells;
  static_assert(kPer <= 32u, "occupancy bits of one batch");
  tally_begin(s_tally);
  for (uint32_t i0 = 0; blockIdx.x + i0 * gridDim.x < nblocks; i0 += kPer) {
    if (threadIdx.x == 0) s_occ = 0u;
    __syncthreads();
    const uint32_t k = threadIdx.x / kCells;
    const uint32_t b = blockIdx.x + (i0 + k) * gridDim.x;
    const uint32_t cell = b * kCells + threadIdx.x % kCells;
    if (b < nblocks && cell < table && cs[cell] != 0xFFFFFFFFu) atomicOr(&s_occ, 1u << k);
    __syncthreads();
    const uint32_t occ = s_occ;
    for (uint32_t i = 0; i < kPer; ++i) {
      if (!((occ >> i) & 1u)) continue;
      adjlist_tile<BITS>(P, blockIdx.x + (i0 + i) * gridDim.x, Q, keys, cs, ce, L, flag, stats, s_tally,
                         lds.sh, lds.q);
      __syncthreads();
    }
    __syncthreads();
  }
  __syncthreads();
  tally_flush(s_tally, stats);
}

size_t adjoint_record_chunks(uint32_t n, uint32_t iters) {
  static_assert(kNlRecordChunks <= kNlChunks, "a recorded set holds a prefix of a forward list");
  return ((size_t)kNlRecordChunks * (iters + 1u) + (kNlChunks - kNlRecordChunks)) * n;
}

// The walk over the blocks of k_tile_adjlist, taking the lists from the
// forward's (F), with only the blocks' cell tables in LDS: k_tile_adjlist_forward
// a thread per particle; k_tile_adjlist_forward_wide 1024-thread workgroups, a
// thread per (particle, chunk), held to 64 VGPRs (8 waves per SIMD) so that two
// workgroups share a CU.
template <int BITS>
__global__ __launch_bounds__(kWideThreads, 8) void k_tile_adjlist_forward_wide(DevParams P, uint32_t nblocks, uint32_t table,
                                                                       const uint32_t* __restrict__ keys,
                                                                       const uint32_t* __restrict__ cs,
                                                                       const uint32_t* __restrict__ ce,
                                                                       NeighbourList F, AdjList L,
                                                                       uint32_t* __restrict__ flag,
                                                                       unsigned long long* __restrict__ stats,
                                                                       uint32_t* __restrict__ redo) {
  __shared__ TileShared<BITS> sh;
  __shared__ uint32_t s_occ;
  __shared__ uint32_t s_tally[kAdjTallies];
  constexpr uint32_t kCells = 1u << BITS;
  constexpr uint32_t kPer = kWideThreads / kCells;
  static_assert(kPer <= 32u, "occupancy bits of one batch");
  tally_begin(s_tally);
  for (uint32_t i0 = 0; blockIdx.x + i0 * gridDim.x < nblocks; i0 += kPer) {
    if (threadIdx.x == 0) s_occ = 0u;
    __syncthreads();
    const uint32_t k = threadIdx.x / kCells;
    const uint32_t b = blockIdx.x + (i0 + k) * gridDim.x;
    const uint32_t cell = b * kCells + threadIdx.x % kCells;
    if (b < nblocks && cell < table && cs[cell] != 0xFFFFFFFFu) atomicOr(&s_occ, 1u << k);
    __syncthreads();
    const uint32_t occ = s_occ;
    for (uint32_t i = 0; i < kPer; ++i) {
      if (!((occ >> i) & 1u)) continue;
      adjlist_forward_tile_wide<BITS>(P, blockIdx.x + (i0 + i) * gridDim.x, keys, cs, ce, F, L, flag, s_tally, redo, sh);
      __syncthreads();
    }
    __syncthreads();
  }
  __syncthreads();
  tally_flush(s_tally, stats);
}

template <int BITS>
__global__ __launch_bounds__(kTileThreads) void k_tile_adjlist_forward(DevParams P, uint32_t nblocks, uint32_t table,
                                                                       const uint32_t* __restrict__ keys,
                                                                       const uint32_t* __restrict__ cs,
                                                                       const uint32_t* __restrict__ ce,
                                                                       NeighbourList F, AdjList L,
                                                                       uint32_t* __restrict__ flag,
                                                                       unsigned long long* __restrict__ stats,
                                                                       uint32_t* __restrict__ redo) {
  __shared__ TileShared<BITS> sh;
  __shared__ uint32_t s_occ;
  __shared__ uint32_t s_tally[kAdjTallies];
  constexpr uint32_t kCells = 1u << BITS;
  constexpr uint32_t kPer = kTileThreads / kCells;
  static_assert(kPer <= 32u, "occupancy bits of one batch");
  tally_begin(s_tally);
  for (uint32_t i0 = 0; blockIdx.x + i0 * gridDim.x < nblocks; i0 += kPer) {
    if (threadIdx.x == 0) s_occ = 0u;
    __syncthreads();
    const uint32_t k = threadIdx.x / kCells;
    const uint32_t b = blockIdx.x + (i0 + k) * gridDim.x;
    const uint32_t cell = b * kCells + threadIdx.x % kCells;
    if (b < nblocks && cell < table && cs[cell] != 0xFFFFFFFFu) atomicOr(&s_occ, 1u << k);
    __syncthreads();
    const uint32_t occ = s_occ;
    for (uint32_t i = 0; i < kPer; ++i) {
      if (!((occ >> i) & 1u)) continue;
      adjlist_forward_tile<BITS>(P, blockIdx.x + (i0 + i) * gridDim.x, keys, cs, ce, F, L, flag, s_tally, redo, sh);
      __syncthreads();
    }
    __syncthreads();
  }
  __syncthreads();
  tally_flush(s_tally, stats);
}

hipError_t launch_adjoint_list_tiles(hipStream_t st, const DevParams& P, uint32_t table, const float4* Q,
                                     const uint32_t* keys, const uint32_t* cs, const uint32_t* ce, AdjList L,
                                     uint32_t* flag, unsigned long long* stats, const uint4* fwd_lists,
                                     const uint16_t* fwd_counts, uint32_t fwd_stride, uint32_t* redo) {
  if (P.n == 0 || table == 0) return hipSuccess;
  constexpr int BITS = 5;
  const uint32_t nblocks = ((table - 1u) >> BITS) + 1u;
  // a workgroup per block up to 4096 of them (small scenes still fill the CUs)
  const uint32_t grid = nblocks < 4096u ? nblocks : 4096u;
  if (fwd_lists) {
    if (!fwd_counts || fwd_stride < P.n || !redo) return hipErrorInvalidValue;
    const NeighbourList F{const_cast<uint4*>(fwd_lists), const_cast<uint16_t*>(fwd_counts), fwd_stride, nullptr};
    const hipError_t e = launch_fill_u32(st, redo, 0u, 1u);
    if (e != hipSuccess) return e;
    if (P.n < kAdjWideMaxParticles) {
      const uint32_t fgrid = nblocks < 2048u ? nblocks : 2048u;
      hipLaunchKernelGGL(k_tile_adjlist_forward_wide<BITS>, dim3(fgrid), dim3(kWideThreads), 0, st, P, nblocks, table,
                         keys, cs, ce, F, L, flag, stats, redo);
    } else {
      hipLaunchKernelGGL(k_tile_adjlist_forward<BITS>, dim3(grid), dim3(kTileThreads), 0, st, P, nblocks, table, keys,
                         cs, ce, F, L, flag, stats, redo);
    }
    // workgroups past the count of appended blocks return at once
    const uint32_t rgrid = nblocks < 256u ? nblocks : 256u;
    hipLaunchKernelGGL(k_tile_adjlist_redo<BITS>, dim3(rgrid), dim3(kTileThreads), 0, st, P, Q, keys, cs, ce, F, L,
                       flag, stats, redo);
  } else if (P.n < kAdjWideMaxParticles) {
    // one 16-wave workgroup per CU, each looping over its share of the blocks
    const uint32_t wgrid = nblocks < 256u ? nblocks : 256u;
    hipLaunchKernelGGL(k_tile_adjlist_wide<BITS>, dim3(wgrid), dim3(kWideThreads), 0, st, P, nblocks, table, Q, keys,
                       cs, ce, L, flag, stats);
  } else {
    hipLaunchKernelGGL(k_tile_adjlist<BITS>, dim3(grid), dim3(kTileThreads), 0, st, P, nblocks, table, Q, keys, cs,
                       ce, L, flag, stats);
  }
  return hipGetLastError();
}

}  // namespace pbd
