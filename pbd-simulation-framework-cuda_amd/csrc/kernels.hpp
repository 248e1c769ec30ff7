// kernels.hpp - host launchers of the PBF step kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "params.hpp"

namespace pbd {

// k_delta flags
enum : uint32_t { DF_APPLY = 1u, DF_UPDATE = 2u, DF_WRITE_DP = 4u };
// k_final flags
// FF_XSPH_DONE: the omega pass already wrote the XSPH velocities to the output
enum : uint32_t { FF_VORT = 1u, FF_XSPH = 2u, FF_UPDATED = 4u, FF_XSPH_DONE = 8u };

// Device buffers of one context (see kernels.hip for the layout).
struct StepBuffers {
  // public, particle order of the previous step on entry, sorted order on exit
  float4* X;   // positions4
  float4* P;   // predictedPositions4
  float4* V;   // velocities4
  float4* C;   // colors4
  float4* F;   // externalForces (by slot)
  // step-internal, sorted order
  float4* Q[2];
  float4* QX[2];
  float4* VS;
  float4* CS;
  float4* DP;
  float4* OM;
  float* LAM;
  float* DENS;
  uint32_t* NCNT;
  uint32_t* CCNT;
  uint32_t* keys_in;    // unsorted cell ids
  uint32_t* cstart;     // cell table
  uint32_t* cend;
  uint32_t table_size;
  // neighbour lists of the tile passes (tiles.hip)
  uint4* NL;            // [kNlChunks][nl_cap] chunks of 8 u16 LDS slots
  uint16_t* NLC;        // padded list lengths (0xFFFF = scan instead)
  uint32_t nl_cap;
  unsigned long long* STATS;  // work counters (PBD_COUNTER_*)
  // Tile lists carried from pass to pass: DISP[(p - 1) nl_cap + i] bounds the
  // displacement of particle i over the substep's first p delta-p passes (the
  // sum of the lengths of its moves; p = 1 .. kCarryPasses, and 0 for p = 0),
  // BUILT[2 b] is the number of delta-p passes before tile b last built its lists
  // (kNoCarry: the tile rebuilds them every pass this substep), MODE[2 b] whether
  // tile b carries its lists in the next substep (its halo stayed within the
  // skin in the last one).  Of a block of two items, 2 b is the first's place and
  // 2 b + 1 the second's.
  float* DISP;
  uint16_t* BUILT;
  uint16_t* MODE;
};
constexpr uint32_t kNoCarry = 0xFFFFu;

// Occupied Morton blocks of the current step in Morton order (the reorder
// kernel marks them, launch_tile_compact lists them).  Blocks of at most
// kTileSmall particles are "small": four of them share one workgroup, one wave
// each; the others take a whole workgroup.
struct TileList {
  const uint32_t* large;  // block ids (cell id >> bits) of the large tiles, ascending; a split block twice, its halves' marks in bits 30, 31
  const uint32_t* small;  // block ids of the small tiles, ascending
  const uint32_t* count;  // count[0] large tiles, count[1] small tiles
  const uint32_t* start;  // per occupied block: 1 + its first sorted index, | its marks
  const uint32_t* end;    // per occupied block: 1 + its last
  uint32_t cap;           // entries of large
};

constexpr uint32_t kTileSmall = 64;           // particles of a small tile (one wave)
// Blocks of up to this many particles are small whatever their halo.  None, by the times: ms
// for 200 steps of a dam break with blocks of up to 8 left small / none: 110K 91.2 / 86.8, 262K
// 122.1 / 116.6, 512K 193.0 / 183.8, 1M 375.2 / 373.8; and 64K with a threshold of 64 set 85.0
// / 80.1.  Up to 2^16 particles, where small tiles are only made for a shape that asks for
// them, 8 stays all the same: those blocks have no lists, and the comparison of the reverse
// mode's lists from the forward with built ones needs blocks without.
__host__ __device__ inline uint32_t small_sure(uint32_t n) { return n <= (1u << 16) ? 8u : 0u; }
constexpr uint32_t kTileCrowded = 1u << 31;   // a block that is large for its halo
constexpr uint32_t kTileSplit = 1u << 30;     // a block that is two items for its halo
// Blocks that are two items: a halo of more than 1528 particles; a particle is in at most 8 (1528 / 8 = 191).
inline uint32_t split_bound(uint32_t ntiles, uint32_t n) { return n / 191u + 1u < ntiles ? n / 191u + 1u : ntiles; }
// The small-tile threshold a context starts with, by particle count.  Measured
// over 100 frames of the dam break (ms per substep at 0 / 32 / 64): up to 2^16
// particles the occupied blocks are too few to fill the chip, and packing four
// sparse blocks into one workgroup only takes parallelism away (32K: 0.45 /
// 0.46 / 0.51, 64K: 0.48 / 0.50 / 0.58); below 2^21 a threshold of 32 is
// fastest (128K: 0.55 / 0.53 / 0.67, 512K: 1.27 / 1.13 / 1.26, 1M: 2.17 / 1.90
// / 1.95); from 2^21 on, 64 (2M: 3.72 at 32, 3.66 at 64; 16.7M: equal).
inline uint32_t default_small_max(uint32_t n) {
  return n <= (1u << 16) ? 0u : n < (1u << 21) ? 32u : kTileSmall;
}
// The largest block that is small under a threshold: from 32 on, blocks of up to kTileSmall
// are, where their halo fits a small tile: a workgroup of its own leaves three of its waves
// idle.  us a step with small tiles up to 32 / 48 / 64: 211K splash 588 / 573 / 521, 1M
// splash 1669 / 1544 / 1438, 64 scenes of 2K to 32K 7960 / 7530 / 7355, 1M column 1060 /
// 1065 / 1064; a 32K frame 223 without, 238 with them.  A rule of the threshold alone, so
// that a shape read and set again launches the same step.
inline uint32_t small_tile_limit(uint32_t small_max) { return small_max < 32u ? small_max : kTileSmall; }
constexpr uint32_t kNlChunks = 12;            // neighbour-list chunks of 8 slots: lists of up to 96 pairs
constexpr uint32_t kTileCompactChunk = 4096;  // flags per block of the compaction
#ifndef PBD_TILE_CHUNK
#define PBD_TILE_CHUNK 4
#endif
constexpr uint32_t kTileChunk = PBD_TILE_CHUNK;        // consecutive tiles per XCD turn (tiles.hip tile_rank0)
constexpr uint32_t kTileGridMultiple = 8 * kTileChunk;  // tile grids are a multiple of (XCDs x tile chunk)
// A tile grid covers the work items (one per workgroup) up to kTileGridDirect
// workgroups (a 256x128x128-cell grid bounds 327,680).  Above that (a batch's
// cell table bounds the items far above the occupied blocks: ~2M workgroups for
// 256 scenes) the passes run on kTileGridStride workgroups, each taking every
// gridDim-th item.
constexpr uint32_t kTileGridDirect = 1u << 20;
constexpr uint32_t kTileGridStride = 16384;
// Skin of the forward tile lists, in percent of the list radius: the first
// lambda pass of a substep lists every pair within (1 + skin) times the radius,
// and the later passes keep a tile's lists while no particle of its halo has
// moved by more than 0.45 skin radius since then.
constexpr uint32_t kListSkinPct = 10;
constexpr uint32_t kListSkinPctMax = 50;
constexpr uint32_t kCarryPasses = 8;  // solver iterations up to which lists are carried
static_assert(kTileGridStride % kTileGridMultiple == 0 && kTileGridDirect % kTileGridMultiple == 0, "tile grids");
// Work items (large tiles + small tiles / 4) <= occupied blocks <= min(ntiles, n), and the
// second halves of split blocks.  Whether a step takes the capped grid is decided by the
// blocks alone: phased scenes have no capped form, and the halves of those just below the
// line lie past it.  A direct grid is a multiple of XCDs x tile chunk, so that tile_rank0
// maps it onto [0, grid).
inline uint32_t tile_grid_round(uint32_t items) {
  return (items + kTileGridMultiple - 1u) / kTileGridMultiple * kTileGridMultiple;
}
inline bool capped_grid(uint32_t ntiles, uint32_t n) {
  return tile_grid_round(ntiles < n ? ntiles : n) > kTileGridDirect;
}
inline uint32_t direct_grid(uint32_t ntiles, uint32_t n) {
  return tile_grid_round((ntiles < n ? ntiles : n) + split_bound(ntiles, n));
}
// Splits the occupied blocks (start[b] != 0) into large[] and small[] by their
// particle count end[b] - (start[b] - 1) (small: at most small_max <= kTileSmall),
// both ascending; count[0..1] = their lengths.  bcount holds
// ceil(nflags / kTileCompactChunk) packed block counts.
// A block of more than small_sure(n) particles is small only if its halo fits a small tile,
// and one whose halo exceeds a tile is two items.  bcount starts at zero.
hipError_t launch_tile_compact(hipStream_t st, int bits, const DevParams& P, const StepBuffers& B, uint32_t nflags,
                               uint32_t* start, const uint32_t* end, uint32_t small_max, uint32_t* bcount, uint32_t* large, uint32_t* small,
                               uint32_t* count);

hipError_t launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t v, uint32_t n);
// Several device arrays copied (src null: zeroed) by one launch; sizes are multiples of 4.
struct CopySet {
  static constexpr uint32_t kMax = 10;
  void* dst[kMax];
  const void* src[kMax];
  size_t bytes[kMax];
  uint32_t count = 0;
  CopySet& add(void* d, const void* s, size_t b) {
    dst[count] = d;
    src[count] = s;
    bytes[count++] = b;
    return *this;
  }
};
hipError_t launch_copy_set(hipStream_t st, const CopySet& c);
// cstart[0, ts) = UINT_MAX, cend[0, ts) = n, flags[0, nflags) = 0 (flags may be null)
hipError_t launch_cell_reset(hipStream_t st, uint32_t* cstart, uint32_t* cend, uint32_t ts, uint32_t n,
                             uint32_t* flags, uint32_t nflags, uint32_t* bcount);
// applyForces + initializeCellIds; the keys' digits of `passes` 8-bit passes are
// added to copy (workgroup mod copies) of the sort's histogram (SortPlan::hist).
hipError_t launch_predict_keys(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, uint32_t* hist,
                               uint32_t passes, uint32_t copies);
// For every occupied Morton block b of 2^tile_bits cells (tile_bits != 0):
// tile_start[b] = 1 + its first sorted index, tile_end[b] = 1 + its last.
hipError_t launch_reorder(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B,
                          const uint32_t* keys_s, const uint32_t* ids_s, uint32_t tile_bits, uint32_t* tile_start,
                          uint32_t* tile_end);
hipError_t launch_lambda(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, const float4* Q,
                         const uint32_t* keys_s, bool first);
hipError_t launch_count(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B,
                        const uint32_t* keys_s);
hipError_t launch_delta(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, uint32_t flags,
                        bool delta, bool collide, const float4* Q, const float4* QX, float4* Qo, float4* QXo,
                        const uint32_t* keys_s);
hipError_t launch_update(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, const float4* Q,
                         float4* QX);
hipError_t launch_omega(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, const float4* Q,
                        const uint32_t* keys_s);
hipError_t launch_final(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, uint32_t flags,
                        const float4* Q, const float4* QX, const uint32_t* keys_s);
// collisionType 1: one stabilization iteration of `batches` contact batches,
// in place on Q / QX (solved: n x words bit rows, minc: n, partner: n).
hipError_t launch_collide_batches(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B,
                                  float4* Q, float4* QX, const uint32_t* keys, uint32_t batches, uint32_t* solved,
                                  uint32_t words, unsigned long long* minc, uint32_t* partner);
// The wide lambda and omega passes (tiles.hip): four lanes per particle, for scenes whose
// blocks do not fill the chip.  Measured (us a step, four lanes / one lane in these two
// passes; every pass builds its lists, a splash's from crowded cells): 2K
// column 230 / 254, 32K column 251 / 263, 30K splash 281 / 379, 64K column 287 / 286, 64K
// splash 381 / 422; 125K column 405 / 328, 125K splash 455 / 462.  The other passes walk
// kept lists, and a 32K scene's take 11.1 us (delta p) and 9.6 (final) with four lanes,
// 9.9 and 8.9 with one.  Four lanes want a workgroup per block, so a launch shape with
// small tiles keeps one lane, and the phased tiles have no fourfold form.
constexpr uint32_t kWideMax = 1u << 16;
constexpr uint32_t kWideGridMax = 8192;  // possible work items (workgroups of 16 waves, most of them empty)
inline bool wide_tiles(const DevParams& P, int bits, uint32_t small_max, uint32_t bound) {
  return bits == 5 && small_max == 0u && !P.phased && P.n <= kWideMax && bound <= kWideGridMax;
}
hipError_t launch_wide_lambda(hipStream_t st, uint32_t grid, const DevParams& P, const TileList& T,
                              const StepBuffers& B, const float4* Q, const uint32_t* keys, bool first, bool carry,
                              uint32_t pass);
hipError_t launch_wide_omega(hipStream_t st, uint32_t grid, const DevParams& P, const TileList& T,
                             const StepBuffers& B, const float4* Q, const uint32_t* keys, bool xsph, uint32_t carry);
// The neighbour passes with a wave per particle (wave.hip), for the particle counts and
// stencils that wave_passes names; the launchers above take them by that rule.  The line
// lies where a thread per particle becomes the faster one (reference parameters, whole
// step, thread / wave, us): 1,000 particles 555 / 128, 13,824 601 / 186, 46,656 617 / 339,
// 74,088 624 / 468, 110,592 635 / 638.
constexpr uint32_t kWaveParticles = 3u << 15;
bool wave_passes(const DevParams& P);
hipError_t launch_wave_lambda(hipStream_t st, const DevParams& P, const StepBuffers& B, const float4* Q,
                              const uint32_t* keys, bool first);
hipError_t launch_wave_delta(hipStream_t st, const DevParams& P, const StepBuffers& B, uint32_t flags, bool delta,
                             bool collide, const float4* Q, const float4* QX, float4* Qo, float4* QXo,
                             const uint32_t* keys);
hipError_t launch_wave_omega(hipStream_t st, const DevParams& P, const StepBuffers& B, const float4* Q,
                             const uint32_t* keys);
hipError_t launch_wave_final(hipStream_t st, const DevParams& P, const StepBuffers& B, uint32_t flags, const float4* Q,
                             const float4* QX, const uint32_t* keys);
hipError_t launch_check_finite(hipStream_t st, uint32_t n, const float4* X, const float4* V, uint32_t* bad);

// ---- LDS cell-block tiles (tiles.hip), textbook variant, 27-cell stencil ----
// The lambda and omega passes write the neighbour lists that the following
// delta-p and final passes read when use_list is set.  With carry, the first
// lambda pass (pass 0) builds the lists of the tiles that carry them this
// substep with the skin (B.MODE); a later lambda pass, after `pass` delta-p
// passes, or the omega pass after `carry` of them, keeps a carrying tile's
// lists while its halo has moved less than P.reuse_max since the tile last
// built them (B.DISP, B.BUILT) and rebuilds the others; delta-p pass
// `track` > 0 records the bounds after it (0: no carry).  The omega pass
// chooses which tiles carry their lists in the next substep.
hipError_t launch_tile_lambda(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P, const TileList& T,
                              const StepBuffers& B, const float4* Q, const uint32_t* keys, bool first, bool carry,
                              uint32_t pass);
hipError_t launch_tile_delta(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P, const TileList& T,
                             const StepBuffers& B, uint32_t flags, bool collide, bool use_list, const float4* Q,
                             const float4* QX, float4* Qo, float4* QXo, const uint32_t* keys, uint32_t track);
// xsph: also apply XSPH (computeViscosity) and write the velocities to B.V
hipError_t launch_tile_omega(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P, const TileList& T,
                             const StepBuffers& B, const float4* Q, const uint32_t* keys, bool xsph, uint32_t carry);
hipError_t launch_tile_final(hipStream_t st, int bits, uint32_t grid, bool stride, const DevParams& P, const TileList& T,
                             const StepBuffers& B, uint32_t flags, bool use_list, const float4* Q, const float4* QX,
                             const uint32_t* keys);

// ---- sort (sort.hip) ----
struct SortPlan {
  uint32_t n_max;       // capacity in items
  uint32_t passes;      // 8-bit digit passes (1..4)
  uint32_t tiles_max;   // tiles for n_max at the smallest tile
  uint32_t items;       // keys per thread of a onesweep tile: 4, 8 or 16 (0: sort_items_for(n))
  // device scratch
  uint32_t* hist;       // [4][256] exclusive digit offsets, then kSortHistCopies x [4][256] partial counts
  uint32_t* tile_ctr;   // [4] tile tickets
  uint32_t* status;     // [4][tiles_max][256] look-back words
  uint32_t* err;        // look-back spin-limit flag (device or pinned host memory)
  uint32_t* keys_alt;   // ping-pong buffers (n_max)
  uint32_t* vals_alt;
  uint32_t* keys_out;
  uint32_t* vals_out;
};

constexpr uint32_t kSortThreads = 256;
constexpr uint32_t kSortItemsMin = 4;                       // the smallest onesweep tile: 1024 keys
constexpr uint32_t kSortTileMin = kSortThreads * kSortItemsMin;
// copies of the digit histogram that the counting workgroups add into (by
// workgroup index), so that no more than 1/32 of them add to the same word
constexpr uint32_t kSortHistCopies = 32;
constexpr uint32_t kSortHistWords = (1u + kSortHistCopies) * 4u * 256u;

// Number of 8-bit passes covering keys < key_bound.
uint32_t sort_passes_for(uint32_t key_bound);
// Keys per thread of the onesweep tiles for n items: the largest of 16, 8, 4
// that still gives 512 tiles (two per CU), else 4.
uint32_t sort_items_for(uint32_t n);
// The sort of a step is split around the kernel that makes the keys:
//   launch_sort_prepare  zeroes the digit histogram, tile tickets and look-back words;
//   (the key kernel adds its keys' digits to the histogram: launch_predict_keys)
//   launch_sort_ranks    scans the histogram and runs the onesweep passes: a stable
//                        LSD sort of (keys_in[i], i), left in *keys_res / *vals_res.
hipError_t launch_sort_prepare(hipStream_t st, const SortPlan& plan, uint32_t n);
hipError_t launch_sort_ranks(hipStream_t st, const SortPlan& plan, uint32_t n, const uint32_t* keys_in,
                             const uint32_t** keys_res, const uint32_t** vals_res);
// Histogram copies the key kernel adds into for n items at tpb threads per workgroup.
uint32_t sort_hist_copies(uint32_t n, uint32_t tpb);

}  // namespace pbd
