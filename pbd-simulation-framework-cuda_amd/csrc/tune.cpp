// tune.cpp - the autotuner of the step's launch shape.
//
// The reference fixes its launch shape from Application.Cuda.threadsPerBlock
// alone (kernel/Initialize.h:73-85, kernel/Globals.h:117-120).  Here a context's
// shape has six coordinates, none of which changes what the step computes:
//   threads per block of the per-particle kernels, the neighbour-pass tile
//   (2^5 or 2^6 cells), the onesweep sort tile (256 x 4, 8 or 16 keys), the
//   largest block that takes one wave instead of a workgroup, the workgroups
//   of the capped tile grid of large batches, and the skin of the tile
//   neighbour lists (pairs beyond the interaction radius add exact zeros, so
//   a longer list sums the same terms in the same order).
// autotune() times each candidate over a few graph-launched steps from the
// context's current state, one coordinate at a time with the others at their
// best so far, restoring the state after every trial; the fastest shape is
// kept.  Choices are cached per workload key in the process and, when the
// environment variable PBD_TUNE_CACHE names a file, in that file.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "fluid.hpp"

namespace pbd {

namespace {

std::mutex g_cache_mutex;
std::map<std::string, Fluid::LaunchShape> g_cache;
bool g_cache_loaded = false;

// "key tpb tile_bits sort_items small_max stride_grid skin_pct" per line
void load_cache_file() {
  if (g_cache_loaded) return;
  g_cache_loaded = true;
  const char* path = std::getenv("PBD_TUNE_CACHE");
  if (!path || !*path) return;
  FILE* f = std::fopen(path, "r");
  if (!f) return;
  char key[256];
  Fluid::LaunchShape s{};
  while (std::fscanf(f, "%255s %u %u %u %u %u %u", key, &s.tpb, &s.tile_bits, &s.sort_items, &s.small_max,
                     &s.stride_grid, &s.skin_pct) == 7)
    g_cache[key] = s;
  std::fclose(f);
}

void store_cache(const std::string& key, const Fluid::LaunchShape& s) {
  g_cache[key] = s;
  const char* path = std::getenv("PBD_TUNE_CACHE");
  if (!path || !*path) return;
  if (FILE* f = std::fopen(path, "a")) {
    std::fprintf(f, "%s %u %u %u %u %u %u\n", key.c_str(), s.tpb, s.tile_bits, s.sort_items, s.small_max, s.stride_grid,
                 s.skin_pct);
    std::fclose(f);
  }
}

}  // namespace

Fluid::LaunchShape Fluid::launch_shape() const {
  return LaunchShape{tpb_, params_.tile_bits, sort_.items, small_max(), stride_grid_, skin_pct_};
}

int Fluid::set_launch_shape(const LaunchShape& s) {
  if (s.tpb < 64 || s.tpb > 1024 || s.tpb % 64 != 0) return fail(PBD_ERR_INVALID, "threads per block: 64 .. 1024, a multiple of 64");
  if (s.tile_bits != 0 && s.tile_bits != 5 && s.tile_bits != 6) return fail(PBD_ERR_INVALID, "tile bits must be 0, 5 or 6");
  if (s.sort_items != 0 && s.sort_items != 4 && s.sort_items != 8 && s.sort_items != 16)
    return fail(PBD_ERR_INVALID, "sort items must be 0, 4, 8 or 16");
  if (s.small_max > kTileSmall) return fail(PBD_ERR_INVALID, "small tiles hold at most 64 particles");
  if (s.stride_grid == 0 || s.stride_grid % kTileGridMultiple != 0 || s.stride_grid > kTileGridDirect)
    return fail(PBD_ERR_INVALID, "the stride grid must be a positive multiple of 32 up to 2^20");
  if (s.skin_pct > kListSkinPctMax) return fail(PBD_ERR_INVALID, "the list skin is 0 .. 50 percent");
  if (int rc = sync()) return rc;
  tpb_ = s.tpb;
  params_.threads_per_block = s.tpb;
  params_.tile_bits = s.tile_bits;
  sort_.items = s.sort_items;
  small_max_ = s.small_max;
  small_auto_ = false;
  stride_grid_ = s.stride_grid;
  skin_pct_ = s.skin_pct;
  dev_valid_ = false;
  invalidate_graph();
  return PBD_OK;
}

// The workload a shape is chosen for: particle count to a power of two, grid,
// variant, phases, solver shape and scene count.
std::string Fluid::tune_key() const {
  uint32_t lg = 0;
  while ((1u << lg) < n_ && lg < 31) ++lg;
  std::ostringstream os;
  os << "n" << lg << "_g" << params_.grid_dims[0] << "x" << params_.grid_dims[1] << "x" << params_.grid_dims[2] << "_v"
     << params_.kernel_variant << "_kw" << params_.kernel_width_neighbours << "_it" << params_.solver_iterations << "_ph"
     << (phased() ? 1 : 0) << "_s" << scene_count_ << "_t" << (params_.tile_bits ? 1 : 0);
  return os.str();
}

int Fluid::time_shape(const LaunchShape& s, uint32_t steps, double* ms) {
  if (int rc = set_launch_shape(s)) return rc;
  if (int rc = ensure_graph()) return rc;
  hipEvent_t a = nullptr, b = nullptr;
  hipError_t e = hipEventCreate(&a);
  if (e == hipSuccess) e = hipEventCreate(&b);
  // one untimed launch (first touch of the shape's code and data), then the trial
  if (e == hipSuccess) e = hipGraphLaunch(graph_exec_, stream_);
  if (e == hipSuccess) e = hipEventRecord(a, stream_);
  for (uint32_t i = 0; i < steps && e == hipSuccess; ++i) e = hipGraphLaunch(graph_exec_, stream_);
  if (e == hipSuccess) e = hipEventRecord(b, stream_);
  if (e == hipSuccess) e = hipEventSynchronize(b);
  float t = 0.0f;
  if (e == hipSuccess) e = hipEventElapsedTime(&t, a, b);
  if (a) (void)hipEventDestroy(a);
  if (b) (void)hipEventDestroy(b);
  if (hip_check(e, "autotune trial")) return status_;
  *ms = (double)t / (double)steps;
  return PBD_OK;
}

int Fluid::autotune(uint32_t trial_steps, LaunchShape* chosen, double* ms_chosen, double* ms_default) {
  if (status_ != PBD_OK) return status_;
  if (trial_steps == 0) trial_steps = 8;
  const LaunchShape start = launch_shape();
  if (n_ == 0) {
    if (chosen) *chosen = start;
    return PBD_OK;
  }
  if (int rc = sync()) return rc;
  const std::string key = tune_key();
  {
    std::lock_guard<std::mutex> lk(g_cache_mutex);
    load_cache_file();
    auto it = g_cache.find(key);
    if (it != g_cache.end()) {  // chosen before for this workload: not timed again
      tuned_ = true;
      if (chosen) *chosen = it->second;
      if (ms_chosen) *ms_chosen = 0.0;
      if (ms_default) *ms_default = 0.0;
      return set_launch_shape(it->second);
    }
  }
  // the state every trial starts from: the public arrays, the phases, the
  // persistent per-slot arrays and the work counters
  const size_t n = n_;
  struct Saved {
    void* dst;
    const void* src;
    size_t bytes;
  };
  std::vector<Saved> keep = {{nullptr, B_.X, n * 16}, {nullptr, B_.P, n * 16},  {nullptr, B_.V, n * 16},
                             {nullptr, B_.C, n * 16}, {nullptr, B_.F, n * 16},  {nullptr, B_.LAM, n * 4},
                             {nullptr, B_.DP, n * 16}, {nullptr, B_.OM, n * 16}, {nullptr, ph_, n * 4},
                             {nullptr, B_.STATS, PBD_COUNTER_COUNT * 8}};
  auto release = [&]() {
    for (auto& k : keep)
      if (k.dst) (void)hipFree(k.dst);
  };
  hipError_t e = hipSuccess;
  for (auto& k : keep)
    if (e == hipSuccess) e = hipMalloc(&k.dst, k.bytes);
  for (auto& k : keep)
    if (e == hipSuccess) e = hipMemcpyAsync(k.dst, k.src, k.bytes, hipMemcpyDeviceToDevice, stream_);
  if (e == hipSuccess) e = hipStreamSynchronize(stream_);
  if (e != hipSuccess) {
    release();
    return hip_check(e, "autotune snapshot");
  }
  auto restore = [&]() {
    hipError_t r = hipSuccess;
    for (auto& k : keep)
      if (r == hipSuccess) r = hipMemcpyAsync(const_cast<void*>(k.src), k.dst, k.bytes, hipMemcpyDeviceToDevice, stream_);
    if (r == hipSuccess) r = hipStreamSynchronize(stream_);
    return r;
  };
  constexpr double kTuneMargin = 0.02;
  // candidates per coordinate; a coordinate the step does not use is not searched
  const bool tiles = params_.tile_bits != 0 && params_.kernel_variant == PBD_KERNEL_TEXTBOOK &&
                     params_.kernel_width_neighbours == 1 && params_.active_find_contacts;
  const uint32_t ntiles = ((B_.table_size - 1u) >> 5) + 1u;
  const bool stride = tiles && capped_grid(ntiles, n_);
  LaunchShape best = start;
  double best_ms = 0.0, first_ms = 0.0;
  int rc = time_shape(best, trial_steps, &best_ms);
  if (rc == PBD_OK) {
    first_ms = best_ms;
    e = restore();
    if (e != hipSuccess) rc = hip_check(e, "autotune restore");
  }
  auto trial = [&](LaunchShape s) {
    if (rc != PBD_OK) return;
    double ms = 0.0;
    rc = time_shape(s, trial_steps, &ms);
    if (rc != PBD_OK) return;
    e = restore();
    if (e != hipSuccess) {
      rc = hip_check(e, "autotune restore");
      return;
    }
    // a candidate replaces the shape in hand only when it is clearly faster:
    // trial windows are short, and a choice made on noise can cost later
    // steps (small tiles, for one, matter only once the flow has spread)
    if (ms < best_ms * (1.0 - kTuneMargin)) {
      best_ms = ms;
      best = s;
    }
  };
  for (uint32_t v : {4u, 8u, 16u}) {
    LaunchShape s = best;
    s.sort_items = v;
    if (v != best.sort_items) trial(s);
  }
  if (tiles && !phased()) {
    for (uint32_t v : {5u, 6u}) {
      LaunchShape s = best;
      s.tile_bits = v;
      if (v != best.tile_bits) trial(s);
    }
  }
  if (tiles) {
    // not 0 (small tiles off): they pay once the flow has spread into sparse
    // blocks, which trial steps from an earlier state may not see (off was 3 %
    // faster over steps 21-28 of the 1M dam break and 14 % slower over 21-220)
    LaunchShape s = best;
    s.small_max = kTileSmall;
    if (small_tile_limit(best.small_max) != kTileSmall) trial(s);
  }
  for (uint32_t v : {128u, 256u, 512u}) {
    LaunchShape s = best;
    s.tpb = v;
    if (v != best.tpb) trial(s);
  }
  if (stride) {
    for (uint32_t v : {8192u, 16384u, 32768u}) {
      LaunchShape s = best;
      s.stride_grid = v;
      if (v != best.stride_grid) trial(s);
    }
  }
  if (tiles) {
    for (uint32_t v : {0u, 5u, 10u, 20u}) {
      LaunchShape s = best;
      s.skin_pct = v;
      if (v != best.skin_pct) trial(s);
    }
  }
  release();
  if (rc != PBD_OK) {
    (void)set_launch_shape(start);
    return rc;
  }
  if (int r = set_launch_shape(best)) return r;
  tuned_ = true;
  {
    std::lock_guard<std::mutex> lk(g_cache_mutex);
    store_cache(key, best);
  }
  if (chosen) *chosen = best;
  if (ms_chosen) *ms_chosen = best_ms;
  if (ms_default) *ms_default = first_ms;
  return PBD_OK;
}

}  // namespace pbd
