// fluid.cpp - host orchestrator of the PBF step (Fluid::compute, Fluid.cu:14-97).
#include "fluid.hpp"

#include <algorithm>
#include <cstring>
#include <sstream>

namespace pbd {

const char* const kStageNames[ST_NUM] = {"predict_keys", "cell_reset", "sort",  "reorder", "tile_list", "lambda",
                                         "delta",        "collide",    "update", "count",  "omega",     "final",
                                         "lambda_carry"};

Fluid::~Fluid() {
  if (stream_ && owns_stream_) (void)hipStreamSynchronize(stream_);
  adj_release();
  invalidate_graph();
  for (auto& p : pending_) {
    (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  for (auto e : event_pool_) (void)hipEventDestroy(e);
  for (void* p : allocations_) (void)hipFree(p);
  if (host_err_) (void)hipHostFree(host_err_);
  if (stream_ && owns_stream_) (void)hipStreamDestroy(stream_);
}

int Fluid::fail(int code, const std::string& msg) {
  status_ = code;
  error_ = msg;
  return code;
}

int Fluid::hip_check(hipError_t e, const char* what) {
  if (e == hipSuccess) return PBD_OK;
  std::ostringstream os;
  os << what << ": " << hipGetErrorString(e);
  return fail(e == hipErrorOutOfMemory ? PBD_ERR_NOMEM : PBD_ERR_HIP, os.str());
}

void Fluid::invalidate_graph() {
  if (graph_exec_) (void)hipGraphExecDestroy(graph_exec_);
  if (graph_) (void)hipGraphDestroy(graph_);
  graph_exec_ = nullptr;
  graph_ = nullptr;
  graph_valid_ = false;
}

template <class T>
static int dev_alloc(std::vector<void*>& list, T** p, size_t count) {
  void* q = nullptr;
  if (hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) return PBD_ERR_NOMEM;
  list.push_back(q);
  *p = static_cast<T*>(q);
  return PBD_OK;
}

// A buffer of the context: its own hipMalloc, or, for a context set up in a
// caller's region (init_in_place), the next 256-byte-aligned piece of it.
template <class T>
int Fluid::take(T** p, size_t count) {
  if (!region_) return dev_alloc(allocations_, p, count);
  const size_t off = (region_used_ + 255u) & ~(size_t)255u;
  const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
  if (off > region_size_ || bytes > region_size_ - off) return PBD_ERR_NOMEM;
  *p = reinterpret_cast<T*>(region_ + off);
  region_used_ = off + bytes;
  return PBD_OK;
}

int Fluid::alloc_table() {
  const uint32_t ts = host_morton(params_.grid_dims[0] - 1u, params_.grid_dims[1] - 1u, params_.grid_dims[2] - 1u) + 1u;
  if (B_.cstart && ts == B_.table_size) return PBD_OK;
  if (region_) {  // a region's table is laid out once, for its largest grid
    if (ts > region_table_) return fail(PBD_ERR_INVALID, "the grid's cell table exceeds the region's");
    B_.table_size = ts;
    sort_.passes = sort_passes_for(ts);
    if (B_.cstart) return PBD_OK;
  } else if (B_.cstart) {
    for (void* q : {(void*)B_.cstart, (void*)B_.cend, (void*)tile_flag_, (void*)tile_end_, (void*)tile_bcount_,
                    (void*)B_.BUILT, (void*)B_.MODE}) {
      (void)hipFree(q);
      allocations_.erase(std::remove(allocations_.begin(), allocations_.end(), q), allocations_.end());
    }
    B_.cstart = B_.cend = nullptr;
    tile_flag_ = tile_end_ = tile_bcount_ = nullptr;
    B_.BUILT = B_.MODE = nullptr;
  }
  // tile starts and ends for the smallest tile (2^5 cells) and the compaction's block counts
  const uint32_t tt = region_ ? region_table_ : ts;
  const uint32_t nt = ((tt - 1u) >> 5) + 1u;
  if (take(&B_.cstart, tt) || take(&B_.cend, tt) || take(&tile_flag_, nt) || take(&tile_end_, nt) ||
      take(&tile_bcount_, (nt + kTileCompactChunk - 1u) / kTileCompactChunk) || take(&B_.BUILT, 2 * (size_t)nt) ||
      take(&B_.MODE, 2 * (size_t)nt))
    return fail(PBD_ERR_NOMEM, "cell table allocation failed");
  // no tile carries its lists before its halo has been seen to stay within the skin
  // (a region is zeroed whole by init_in_place)
  if (!region_ && hip_check(hipMemsetAsync(B_.MODE, 0, (size_t)nt * 4, stream_), "tile mode zeroing")) return status_;
  B_.table_size = ts;
  sort_.passes = sort_passes_for(ts);
  return PBD_OK;
}

int Fluid::init(const pbd_params& p, uint32_t capacity) {
  params_ = p;
  const char* why = nullptr;
  DevParams probe;
  if (derive_device_params(p, 0, probe, &why) != PBD_OK) return fail(PBD_ERR_INVALID, why);
  if (capacity == 0) capacity = p.texture_width * p.texture_width;
  if (capacity == 0 || capacity >= (1u << 30)) return fail(PBD_ERR_INVALID, "capacity must be in [1, 2^30)");
  cap_ = capacity;
  tpb_ = p.threads_per_block ? p.threads_per_block : 256;
  if (tpb_ < 64 || tpb_ > 1024 || (tpb_ % 64) != 0) tpb_ = 256;
  if (hip_check(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate")) return status_;
  owns_stream_ = true;
  if (int rc = layout()) return rc;
  // initializeDensity zeroes lambdas, deltaPositions, externalForces, omegas (Density.h:321-330)
  const size_t c = cap_;
  hipError_t e = hipSuccess;
  for (void* q : {(void*)B_.X, (void*)B_.P, (void*)B_.V, (void*)B_.C, (void*)B_.F, (void*)B_.DP, (void*)B_.OM,
                  (void*)B_.VS, (void*)B_.CS})
    if (e == hipSuccess) e = hipMemsetAsync(q, 0, c * 16, stream_);
  for (void* q : {(void*)B_.LAM, (void*)B_.DENS, (void*)B_.NCNT, (void*)B_.CCNT, (void*)ph_, (void*)phs_})
    if (e == hipSuccess) e = hipMemsetAsync(q, 0, c * 4, stream_);
  if (e == hipSuccess) e = hipMemsetAsync(d_scratch_, 0, 16, stream_);
  if (e == hipSuccess) e = hipMemsetAsync(tile_count_, 0, 8, stream_);
  if (e == hipSuccess) e = hipMemsetAsync(B_.STATS, 0, PBD_COUNTER_COUNT * 8, stream_);
  if (e == hipSuccess) e = hipStreamSynchronize(stream_);
  if (hip_check(e, "initial zeroing")) return status_;
  stage_ms_.assign(ST_NUM, 0.0);
  stage_launches_.assign(ST_NUM, 0);
  return PBD_OK;
}

// The context's device buffers for cap_ particles (public arrays too, unless
// the caller lends them per step) and the cell table of the parameters' grid.
int Fluid::layout() {
  const size_t c = cap_;
  int rc = 0;
  if (!region_) {
    rc |= take(&B_.X, c);
    rc |= take(&B_.P, c);
    rc |= take(&B_.V, c);
    rc |= take(&B_.C, c);
    rc |= take(&B_.F, c);
  }
  rc |= take(&B_.Q[0], c);
  rc |= take(&B_.Q[1], c);
  rc |= take(&B_.QX[0], c);
  rc |= take(&B_.QX[1], c);
  rc |= take(&B_.VS, c);
  rc |= take(&B_.CS, c);
  rc |= take(&B_.DP, c);
  rc |= take(&B_.OM, c);
  rc |= take(&B_.LAM, c);
  rc |= take(&B_.DENS, c);
  rc |= take(&B_.NCNT, c);
  rc |= take(&B_.CCNT, c);
  rc |= take(&B_.DISP, c * kCarryPasses);
  rc |= take(&B_.keys_in, c);
  rc |= take(&ph_, c);
  rc |= take(&phs_, c);
  sort_.n_max = cap_;
  sort_.tiles_max = (cap_ + kSortTileMin - 1) / kSortTileMin;
  rc |= take(&sort_.hist, kSortHistWords);
  rc |= take(&sort_.tile_ctr, 4);
  rc |= take(&sort_.status, (size_t)4 * sort_.tiles_max * 256);
  if (region_) {
    rc |= take(&sort_.err, 1);
  } else {
    // The sort's error flag lies in pinned host memory: kernels write it on failure only,
    // and sync() reads it in place (a copy of 4 bytes took 10 us of every sync).
    rc |= hipHostMalloc(reinterpret_cast<void**>(&host_err_), sizeof(uint32_t), hipHostMallocDefault) != hipSuccess ||
          hipHostGetDevicePointer(reinterpret_cast<void**>(&sort_.err), host_err_, 0) != hipSuccess;
    if (!rc) *host_err_ = 0u;
  }
  rc |= take(&sort_.keys_alt, c);
  rc |= take(&sort_.vals_alt, c);
  rc |= take(&sort_.keys_out, c);
  rc |= take(&sort_.vals_out, c);
  rc |= take(&d_scratch_, 4);
  rc |= take(&tile_list_, (size_t)2 * c);
  rc |= take(&tile_count_, 2);
  rc |= take(&B_.NL, c * kNlChunks);  // up to 8 kNlChunks slots per particle
  rc |= take(&B_.NLC, c);
  B_.nl_cap = cap_;
  rc |= take(&B_.STATS, PBD_COUNTER_COUNT);
  if (rc) return fail(PBD_ERR_NOMEM, region_ ? "the region is too small for the context" : "device allocation failed");
  if (alloc_table()) return status_;
  keys_sorted_ = sort_.keys_out;
  ids_sorted_ = sort_.vals_out;
  return PBD_OK;
}

int Fluid::init_in_place(const pbd_params& p, uint32_t capacity, uint32_t table_cap, unsigned char* region,
                         size_t bytes, hipStream_t st) {
  params_ = p;
  const char* why = nullptr;
  DevParams probe;
  if (derive_device_params(p, 0, probe, &why) != PBD_OK) return fail(PBD_ERR_INVALID, why);
  if (capacity == 0 || table_cap == 0 || !region) return fail(PBD_ERR_INVALID, "empty region");
  cap_ = capacity;
  tpb_ = 256;
  region_ = region;
  region_size_ = bytes;
  region_used_ = 0;
  region_table_ = table_cap;
  stream_ = st;
  owns_stream_ = false;
  if (int rc = layout()) return rc;
  // everything starts at zero, like a new context's buffers (kernels only: the
  // caller's stream may be capturing a graph)
  return hip_check(launch_fill_u32(st, reinterpret_cast<uint32_t*>(region_), 0u, (uint32_t)(region_used_ / 4u)),
                   "region zeroing");
}

// One substep on the caller's arrays, stream-ordered on st (a context set up
// by init_in_place).  What a step reads before it writes (lambdas, delta p,
// omega, densities, the sort's error flag) is cleared first, so every call
// steps as a new context's first compute would.
int Fluid::compute_in_place(const pbd_params& p, uint32_t n, float4* X, float4* P, float4* V, float4* C, float4* F,
                            hipStream_t st) {
  clear_status();
  if (!region_) return fail(PBD_ERR_INVALID, "not a context in a caller's region");
  if (n > cap_) return fail(PBD_ERR_CAPACITY, "more particles than the region holds");
  if (std::memcmp(&p, &params_, sizeof p) != 0) {
    const char* why = nullptr;
    DevParams probe;
    if (derive_device_params(p, n, probe, &why) != PBD_OK) return fail(PBD_ERR_INVALID, why);
    params_ = p;
    tpb_ = p.threads_per_block ? p.threads_per_block : 256;
    if (tpb_ < 64 || tpb_ > 1024 || (tpb_ % 64) != 0) tpb_ = 256;
    if (int rc = alloc_table()) return rc;  // no allocation: checks the table against the region's
    dev_valid_ = false;
  }
  if (n != n_) dev_valid_ = false;
  n_ = n;
  stream_ = st;
  B_.X = X;
  B_.P = P;
  B_.V = V;
  B_.C = C;
  B_.F = F;
  if (n == 0) return PBD_OK;
  CopySet zero;  // one launch: as five they took 9 us of a small scene's step
  zero.add(B_.LAM, nullptr, (size_t)n * 4).add(B_.DENS, nullptr, (size_t)n * 4);
  zero.add(B_.DP, nullptr, (size_t)n * 16).add(B_.OM, nullptr, (size_t)n * 16).add(sort_.err, nullptr, 4);
  const hipError_t e = launch_copy_set(st, zero);
  if (hip_check(e, "clearing the region")) return status_;
  compute();
  return status_;
}

int Fluid::set_params(const pbd_params& p) {
  const char* why = nullptr;
  DevParams probe;
  if (derive_device_params(p, n_, probe, &why) != PBD_OK) return fail(PBD_ERR_INVALID, why);
  if (hip_check(hipStreamSynchronize(stream_), "sync")) return status_;
  params_ = p;
  tpb_ = p.threads_per_block ? p.threads_per_block : 256;
  if (tpb_ < 64 || tpb_ > 1024 || (tpb_ % 64) != 0) tpb_ = 256;
  dev_valid_ = false;
  tuned_ = false;
  invalidate_graph();
  return alloc_table();
}

int Fluid::add_particles(uint32_t n, const float* pos4, const float* vel4, const float* col4) {
  if (n == 0) return PBD_OK;
  if (!pos4) return fail(PBD_ERR_INVALID, "positions are required");
  if ((uint64_t)n_ + n > cap_) {
    std::ostringstream os;
    os << "capacity exceeded: " << n_ << " + " << n << " > " << cap_;
    return fail(PBD_ERR_CAPACITY, os.str());
  }
  if (hip_check(hipStreamSynchronize(stream_), "sync")) return status_;
  const size_t off = n_, bytes = (size_t)n * 16;
  std::vector<float> zeros, white;
  if (!vel4) {
    zeros.assign((size_t)n * 4, 0.0f);
    vel4 = zeros.data();
  }
  if (!col4) {
    white.assign((size_t)n * 4, 1.0f);
    col4 = white.data();
  }
  std::vector<float> f0((size_t)n * 4, 0.0f);
  hipError_t e = hipMemcpy(B_.X + off, pos4, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(B_.P + off, pos4, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(B_.V + off, vel4, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(B_.C + off, col4, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(B_.F + off, f0.data(), bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(ph_ + off, 0, (size_t)n * 4);  // new particles are fluid
  if (hip_check(e, "add_particles upload")) return status_;
  n_ += n;
  dev_valid_ = false;
  tuned_ = false;
  invalidate_graph();
  return PBD_OK;
}

int Fluid::clear_particles() {
  if (hip_check(hipStreamSynchronize(stream_), "sync")) return status_;
  n_ = 0;
  dev_valid_ = false;
  invalidate_graph();
  return PBD_OK;
}

// ---------------------------------------------------------------------------
// timing
void Fluid::stage_begin(int stage) {
  if (!timing_) return;
  (void)stage;
  hipEvent_t a;
  if (!event_pool_.empty()) {
    a = event_pool_.back();
    event_pool_.pop_back();
  } else {
    (void)hipEventCreate(&a);
  }
  (void)hipEventRecord(a, stream_);
  cur_begin_ = a;
}

void Fluid::stage_end(int stage) {
  if (!timing_ || !cur_begin_) return;
  hipEvent_t b;
  if (!event_pool_.empty()) {
    b = event_pool_.back();
    event_pool_.pop_back();
  } else {
    (void)hipEventCreate(&b);
  }
  (void)hipEventRecord(b, stream_);
  pending_.push_back({stage, cur_begin_, b});
  cur_begin_ = nullptr;
}

int Fluid::collect_timings() {
  for (auto& p : pending_) {
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
      stage_ms_[p.stage] += ms;
      stage_launches_[p.stage] += 1;
    }
    event_pool_.push_back(p.a);
    event_pool_.push_back(p.b);
  }
  pending_.clear();
  return PBD_OK;
}

int Fluid::timings(const char** names, double* ms, uint64_t* launches, uint32_t cap, uint32_t* count) {
  if (int rc = sync()) return rc;
  for (uint32_t i = 0; i < (uint32_t)ST_NUM && i < cap; ++i) {
    if (names) names[i] = kStageNames[i];
    if (ms) ms[i] = stage_ms_[i];
    if (launches) launches[i] = stage_launches_[i];
  }
  if (count) *count = ST_NUM;
  return PBD_OK;
}

void Fluid::reset_timings() {
  std::fill(stage_ms_.begin(), stage_ms_.end(), 0.0);
  std::fill(stage_launches_.begin(), stage_launches_.end(), 0);
}

int Fluid::counters(uint64_t* values, uint32_t cap, uint32_t* count) {
  if (count) *count = PBD_COUNTER_COUNT;
  if (!values || cap == 0) return PBD_OK;
  unsigned long long h[PBD_COUNTER_COUNT] = {};
  hipError_t e = hipMemcpyAsync(h, B_.STATS, sizeof(h), hipMemcpyDeviceToHost, stream_);
  if (e == hipSuccess) e = hipStreamSynchronize(stream_);
  if (hip_check(e, "counters")) return status_;
  for (uint32_t i = 0; i < std::min<uint32_t>(cap, PBD_COUNTER_COUNT); ++i) values[i] = h[i];
  return PBD_OK;
}

int Fluid::reset_counters() {
  hipError_t e = launch_fill_u32(stream_, reinterpret_cast<uint32_t*>(B_.STATS), 0u, 2 * PBD_COUNTER_COUNT);
  if (e == hipSuccess) e = hipStreamSynchronize(stream_);
  return hip_check(e, "reset counters");
}

void Fluid::set_scenes(const SceneParams* table, const uint32_t* first, uint32_t n, uint32_t slot_log2) {
  scene_table_ = table;
  scene_first_ = first;
  scene_count_ = n;
  slot_log2_ = slot_log2;
  dev_valid_ = false;
  invalidate_graph();
}

// Context tables the derived parameters point to: the phases (when the context
// holds solid particles or friction is on) and a batched context's scene table.
void Fluid::apply_context() {
  // tile lists with a skin: carried from pass to pass while the halos stay
  // within it (0.45 skin per particle: two particles close in by 0.9 skin at
  // most, the rest is the margin for rounding)
  if (skin_pct_ > 0) {
    const float skin = dev_.list_r * (float)skin_pct_ * 0.01f;
    const float rl = dev_.list_r + skin;
    dev_.tile_r2 = rl * rl * 1.0001f;
    dev_.reuse_max = 0.45f * skin;
  } else {
    dev_.tile_r2 = dev_.list_r2;
    dev_.reuse_max = -1.0f;
  }
  dev_.phased = (has_solids_ || params_.friction_static > 0.0f) ? 1u : 0u;
  dev_.phs = dev_.phased ? phs_ : nullptr;
  dev_.ph = dev_.phased ? ph_ : nullptr;
  if (!scene_table_) return;
  dev_.scenes = scene_table_;
  dev_.scene_first = scene_first_;
  dev_.n_scenes = scene_count_;
  dev_.slot_log2 = slot_log2_;
  dev_.local_mask = (1u << slot_log2_) - 1u;
}

// collisionType 1 state: a solved bit per neighbour-table slot, the smallest
// offer and the candidate partner per particle; allocated on first use.
int Fluid::ensure_batch_buffers() {
  const uint32_t words = (params_.max_neighbours_per_particle + 31u) / 32u;
  if (batch_solved_ && words <= batch_words_) return PBD_OK;
  if ((uint64_t)cap_ * words >= (1ull << 32)) return fail(PBD_ERR_INVALID, "collisionType 1: contact table too large");
  for (void* q : {(void*)batch_solved_, (void*)batch_min_, (void*)batch_partner_}) {
    if (!q) continue;
    (void)hipFree(q);
    allocations_.erase(std::remove(allocations_.begin(), allocations_.end(), q), allocations_.end());
  }
  batch_solved_ = nullptr;
  batch_min_ = nullptr;
  batch_partner_ = nullptr;
  if (dev_alloc(allocations_, &batch_solved_, (size_t)cap_ * words) || dev_alloc(allocations_, &batch_min_, cap_) ||
      dev_alloc(allocations_, &batch_partner_, cap_))
    return fail(PBD_ERR_NOMEM, "collisionType 1 buffers");
  batch_words_ = words;
  return PBD_OK;
}

// ---------------------------------------------------------------------------
// The step.
#define PBD_LAUNCH(stage, call)                                   \
  do {                                                            \
    stage_begin(stage);                                           \
    hipError_t e_ = (call);                                       \
    stage_end(stage);                                             \
    if (e_ != hipSuccess) return hip_check(e_, kStageNames[stage]); \
  } while (0)

int Fluid::enqueue_substep() {
  const DevParams& P = dev_;
  const hipStream_t st = stream_;
  const uint32_t tpb = tpb_;
  const uint32_t g = P.gates;
  // LDS tiles for the 27-cell stencil of the textbook kernels (tiles.hip)
  const int bits = (int)params_.tile_bits;
  bool tiles = bits != 0 && P.variant == PBD_KERNEL_TEXTBOOK && P.kw == 1 && (g & G_FIND_CONTACTS);
  uint32_t tgrid = 0, ntiles = 0;
  bool tstride = false;
  if (tiles) {
    ntiles = ((B_.table_size - 1u) >> bits) + 1u;
    tstride = capped_grid(ntiles, P.n);
    tgrid = tstride ? stride_grid_ : direct_grid(ntiles, P.n);
    // phases on tiles: 2^5-cell blocks with the direct grid only
    if (P.phased && (bits != 5 || tstride)) tiles = false;
  }
  const uint32_t wgrid = std::min(ntiles, P.n) + split_bound(ntiles, P.n);  // the wide passes': a workgroup per block
  const bool wide = tiles && wide_tiles(P, bits, small_max(), std::min(ntiles, P.n));
  const TileList TL{tile_list_, tile_list_ + cap_, tile_count_, tile_flag_, tile_end_, cap_};
  // Lists carried over the substep: in the tiles whose halo stayed within the
  // skin over the last substep, the first lambda pass builds them with the
  // skin, and the later lambda passes and the omega pass keep them while the
  // halo has moved less than the skin allows since the tile last built them.
  // Every move of Q between them must be a tile delta-p pass that records the
  // displacement bounds: one delta-p pass per iteration, its collisions fused
  // (stabilizationIterations <= 1), contacts not in batches, and at most
  // kCarryPasses iterations (the bounds of each pass are kept).  The omega pass
  // picks the carrying tiles of the next substep, so it must run.
  // A recorded step keeps the tile lists of its position sets for the reverse
  // passes (AdjTape::NL): iteration k's lambda pass (and its delta-p pass) and
  // the omega pass (and the final pass) use set k and set iters of the record,
  // and every one of those passes builds its lists, without a skin.
  const bool rec_lists = rec_ && rec_->NL && tiles && bits == 5;
  if (rec_) rec_->nl_recorded = rec_lists;
  const auto list_set = [&](uint32_t k) {
    StepBuffers b = B_;
    if (rec_lists) {
      b.NL = rec_->NL + (size_t)k * kNlRecordChunks * P.n;
      b.NLC = rec_->NLC + (size_t)k * P.n;
      b.nl_cap = P.n;
    }
    return b;
  };
  const bool carry = !rec_lists && tiles && P.reuse_max > 0.0f && (g & G_LAMBDA) && (g & G_DELTA) && (g & G_OMEGA) &&
                     params_.stabilization_iterations <= 1 &&
                     !(params_.collision_type == 1 && params_.stabilization_iterations > 0) &&
                     params_.solver_iterations > 0 && params_.solver_iterations <= kCarryPasses;
  const size_t n16 = (size_t)P.n * 16, n4 = (size_t)P.n * 4;
  // the sort's histogram, tickets and look-back words start at zero
  PBD_LAUNCH(ST_SORT, launch_sort_prepare(st, sort_, P.n));
  // 1-2. applyForces + initializeCellIds (Fluid.cu:21-25), with the sort's digit counts
  PBD_LAUNCH(ST_PREDICT, launch_predict_keys(st, tpb, P, B_, sort_.hist, sort_.passes, kSortHistCopies));
  // resetCellInfo (Fluid.cu:31): empty = {UINT_MAX, N}
  PBD_LAUNCH(ST_CELL_RESET, launch_cell_reset(st, B_.cstart, B_.cend, B_.table_size, P.n, tiles ? tile_flag_ : nullptr,
                                              tiles ? ntiles : 0u, tile_bcount_));
  // 3. sortIds (Fluid.cu:27)
  PBD_LAUNCH(ST_SORT, launch_sort_ranks(st, sort_, P.n, B_.keys_in, &keys_sorted_, &ids_sorted_));
  // 4-5. reorderStorage + computeCellInfo (Fluid.cu:29,33)
  // Where a recorded step's delta-p passes write whole new positions, they write them (and
  // x, and the lambdas) to the record instead of to buffers that are copied there.
  const uint32_t S = params_.stabilization_iterations;
  const uint32_t iters = params_.solver_iterations;
  const bool batched = params_.collision_type == 1 && S > 0;
  const bool direct = rec_ && (g & G_DELTA) && !batched && iters > 0;
  float4* Q = direct ? rec_->Q : B_.Q[0];
  float4* QX = direct && rec_->QX ? rec_->QX : B_.QX[0];
  StepBuffers sorted = B_;
  sorted.Q[0] = Q;
  sorted.QX[0] = QX;
  PBD_LAUNCH(ST_REORDER, launch_reorder(st, tpb, P, sorted, keys_sorted_, ids_sorted_, tiles ? (uint32_t)bits : 0u,
                                        tile_flag_, tile_end_));
  if (tiles)
    PBD_LAUNCH(ST_TILES, launch_tile_compact(st, bits, P, B_, ntiles, tile_flag_, tile_end_, small_tiles(), tile_bcount_, tile_list_,
                                             tile_list_ + cap_, tile_count_));
  const uint32_t* keys = keys_sorted_;
  if (rec_) {
    // the step's input state (for the reverse of the predict stage; nothing has written to
    // it yet), its order and its cells
    const size_t tb = (size_t)B_.table_size * 4;
    CopySet set;
    set.add(rec_->Xin, B_.X, n16).add(rec_->Vin, B_.V, n16).add(rec_->Fin, B_.F, n16);
    set.add(rec_->keys, keys_sorted_, n4).add(rec_->perm, ids_sorted_, n4);
    set.add(rec_->cs, B_.cstart, tb).add(rec_->ce, B_.cend, tb);
    if (rec_->PH) set.add(rec_->PH, phs_, n4);  // the step's phases, sorted
    if (!direct) set.add(rec_->Q, Q, n16);
    if (tape_copy(set)) return status_;
  }

  // 6-7. solver loop (Fluid.cu:49-80); contacts/neighbours are walked inside the passes
  const bool lambda_on = g & G_LAMBDA, delta_on = g & G_DELTA, apply_on = g & G_APPLY_DELTA;
  const bool update_on = g & G_UPDATE;
  bool counted = false, updated = false;
  if (batched) {
    // allocated ahead of any capture (ensure_graph); the eager path allocates on first use
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hip_check(hipStreamIsCapturing(st, &cs), "hipStreamIsCapturing")) return status_;
    if (cs != hipStreamCaptureStatusNone && !batch_solved_)
      return fail(PBD_ERR_INVALID, "collisionType 1 buffers must exist before a graph capture");
    if (cs == hipStreamCaptureStatusNone) {
      if (int rc = ensure_batch_buffers()) return rc;
    }
  }
  for (uint32_t it = 0; it < iters; ++it) {
    const bool last_it = it + 1 == iters;
    bool listed = false;  // the lambda pass left the neighbour lists of Q
    // x at the iteration's start, for the reverse of the friction
    if (rec_ && rec_->QX && !direct && tape_copy(CopySet().add(rec_->QX + (size_t)it * P.n, QX, n16))) return status_;
    // the last iteration's lambdas stay in the context's buffer too
    const bool lam_direct = direct && !last_it && lambda_on;
    StepBuffers B = list_set(it);
    if (lam_direct) B.LAM = rec_->LAM + (size_t)it * P.n;
    if (lambda_on) {
      if (tiles) {
        PBD_LAUNCH(carry && counted ? ST_LAMBDA_CARRY : ST_LAMBDA,
                   wide ? launch_wide_lambda(st, wgrid, P, TL, B, Q, keys, !counted, carry, it)
                        : launch_tile_lambda(st, bits, tgrid, tstride, P, TL, B, Q, keys, !counted, carry,
                                      it));
        listed = true;
      } else {
        PBD_LAUNCH(ST_LAMBDA, launch_lambda(st, tpb, P, B, Q, keys, !counted));
      }
      counted = true;
      if (rec_ && !lam_direct && tape_copy(CopySet().add(rec_->LAM + (size_t)it * P.n, B_.LAM, n4))) return status_;
    }
    // the Q-writing kernels of this iteration
    struct K {
      bool delta, collide;
      uint32_t flags;
      bool batches = false;  // collisionType 1: one stabilization iteration of contact batches, in place
    };
    K ks[128];
    uint32_t nk = 0;
    const uint32_t ncoll = std::min<uint32_t>(S, 100);
    if (batched) {
      // Fluid.cu:52-78 with collisionType 1: delta p computed first, the batches
      // move p* and x in place, delta p applied last
      if (delta_on) ks[nk++] = {true, false, DF_WRITE_DP};
      for (uint32_t c = 0; c < ncoll; ++c) ks[nk++] = {false, false, 0u, true};
      if (apply_on) ks[nk++] = {false, false, DF_APPLY};
    } else if (delta_on) {
      uint32_t fl = 0;
      if (apply_on && ncoll <= 1) fl |= DF_APPLY;
      if (ncoll >= 2 || !apply_on || last_it) fl |= DF_WRITE_DP;
      ks[nk++] = {true, ncoll >= 1, fl};
      for (uint32_t c = 1; c < ncoll; ++c) ks[nk++] = {false, true, (apply_on && c + 1 == ncoll) ? DF_APPLY : 0u};
    } else {
      for (uint32_t c = 0; c < ncoll; ++c) ks[nk++] = {false, true, (apply_on && c + 1 == ncoll) ? DF_APPLY : 0u};
      if (ncoll == 0 && apply_on) ks[nk++] = {false, false, DF_APPLY};
    }
    for (uint32_t k = 0; k < nk; ++k) {
      if (ks[k].batches) {
        PBD_LAUNCH(ST_COLLIDE, launch_collide_batches(st, tpb, P, B_, Q, QX, keys,
                                                      params_.max_collision_batches, batch_solved_, batch_words_,
                                                      batch_min_, batch_partner_));
        continue;
      }
      uint32_t fl = ks[k].flags;
      if (last_it && k + 1 == nk && update_on) {
        fl |= DF_UPDATE;
        updated = true;
      }
      const int stage = ks[k].delta ? ST_DELTA : ST_COLLIDE;
      const bool to_rec = direct && k + 1 == nk;
      float4* Qo = to_rec ? rec_->Q + (size_t)(it + 1) * P.n : B_.Q[Q == B_.Q[0] ? 1 : 0];
      float4* QXo = to_rec && rec_->QX && !last_it ? rec_->QX + (size_t)(it + 1) * P.n : B_.QX[QX == B_.QX[0] ? 1 : 0];
      if (tiles && ks[k].delta) {
        PBD_LAUNCH(stage, launch_tile_delta(st, bits, tgrid, tstride, P, TL, B, fl, ks[k].collide, listed && k == 0, Q, QX,
                                            Qo, QXo, keys, carry ? it + 1u : 0u));
      } else {
        PBD_LAUNCH(stage, launch_delta(st, tpb, P, B, fl, ks[k].delta, ks[k].collide, Q, QX, Qo, QXo, keys));
      }
      Q = Qo;
      QX = QXo;
    }
    if (rec_ && !direct && tape_copy(CopySet().add(rec_->Q + (size_t)(it + 1) * P.n, Q, n16))) return status_;
  }
  if (!counted) PBD_LAUNCH(ST_COUNT, launch_count(st, tpb, P, B_, keys));
  // 8. updatePositions (Fluid.cu:82-84) when not fused into the last solver pass
  if (update_on && !updated) {
    PBD_LAUNCH(ST_UPDATE, launch_update(st, tpb, P, B_, Q, QX));
    updated = true;
  }
  // 9. computeOmega (Fluid.cu:86-88)
  const bool omega_listed = tiles && (g & G_OMEGA);  // the omega pass leaves the lists of Q
  // the tile omega pass also applies XSPH: it walks the same neighbours with their velocities
  const bool xsph_in_omega = omega_listed && (g & G_VISCOSITY);
  if (g & G_OMEGA) {
    if (tiles) {
      PBD_LAUNCH(ST_OMEGA,
                 wide ? launch_wide_omega(st, wgrid, P, TL, list_set(iters), Q, keys, xsph_in_omega,
                                          carry ? iters : 0u)
                      : launch_tile_omega(st, bits, tgrid, tstride, P, TL, list_set(iters), Q, keys, xsph_in_omega,
                                   carry ? iters : 0u));
    } else {
      PBD_LAUNCH(ST_OMEGA, launch_omega(st, tpb, P, B_, Q, keys));
    }
  }
  if (rec_ && tape_copy(CopySet().add(rec_->U, B_.VS, n16).add(rec_->OM, B_.OM, n16))) return status_;
  // 10-11. computeVorticity + computeViscosity (Fluid.cu:90-96) and the output
  uint32_t ff = 0;
  if (g & G_VORTICITY) ff |= FF_VORT;
  if (g & G_VISCOSITY) ff |= xsph_in_omega ? FF_XSPH_DONE : FF_XSPH;
  if (updated) ff |= FF_UPDATED;
  if (tiles)
    PBD_LAUNCH(ST_FINAL, launch_tile_final(st, bits, tgrid, tstride, P, TL, list_set(iters), ff, omega_listed, Q, QX, keys));
  else
    PBD_LAUNCH(ST_FINAL, launch_final(st, tpb, P, B_, ff, Q, QX, keys));
  return PBD_OK;
}

void Fluid::compute() {
  if (status_ != PBD_OK) return;
  if (n_ == 0) return;  // Fluid.cu:19
  if (!dev_valid_) {
    const char* why = nullptr;
    if (derive_device_params(params_, n_, dev_, &why) != PBD_OK) {
      fail(PBD_ERR_INVALID, why);
      return;
    }
    apply_context();
    dev_valid_ = true;
  }
  enqueue_substep();
}

int Fluid::step(uint32_t frames, bool graph) {
  if (status_ != PBD_OK) return status_;
  const uint32_t sub = params_.substeps ? params_.substeps : 1;
  if (n_ == 0) return PBD_OK;
  if (params_.autotune && !tuned_ && !rec_ && frames > 0) {
    if (int rc = autotune(8, nullptr, nullptr, nullptr)) return rc;
  }
  if (!graph || timing_) {
    for (uint32_t f = 0; f < frames; ++f)
      for (uint32_t s = 0; s < sub; ++s) {
        compute();
        if (status_ != PBD_OK) return status_;
      }
    return PBD_OK;
  }
  if (int rc = ensure_graph()) return rc;
  for (uint32_t f = 0; f < frames; ++f)
    for (uint32_t s = 0; s < sub; ++s)
      if (hip_check(hipGraphLaunch(graph_exec_, stream_), "hipGraphLaunch")) return status_;
  return PBD_OK;
}

// Capture one substep into graph_exec_ (once per parameter / particle-count change).
int Fluid::ensure_graph() {
  if (graph_valid_) return PBD_OK;
  if (!dev_valid_) {
    const char* why = nullptr;
    if (derive_device_params(params_, n_, dev_, &why) != PBD_OK) return fail(PBD_ERR_INVALID, why);
    apply_context();
    dev_valid_ = true;
  }
  // everything the substep needs is allocated before the capture: no allocation
  // or free may happen while the stream captures
  if (params_.collision_type == 1 && params_.stabilization_iterations > 0) {
    if (int rc = ensure_batch_buffers()) return rc;
  }
  if (hip_check(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture"))
    return status_;
  AdjTape* rec = rec_;
  rec_ = nullptr;  // a graph never records
  int rc = enqueue_substep();
  rec_ = rec;
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(stream_, &g);
  if (rc != PBD_OK) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (hip_check(e, "hipStreamEndCapture")) return status_;
  graph_ = g;
  if (hip_check(hipGraphInstantiate(&graph_exec_, graph_, nullptr, nullptr, 0), "hipGraphInstantiate"))
    return status_;
  graph_valid_ = true;
  return PBD_OK;
}

int Fluid::tape_copy(const CopySet& set) { return hip_check(launch_copy_set(stream_, set), "adjoint record copy"); }

int Fluid::sync() {
  if (!stream_ || !sort_.err) return status_;  // not initialised: nothing queued
  if (hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize")) return status_;
  if (timing_ || !pending_.empty()) collect_timings();
  uint32_t err = 0;
  if (host_err_) err = *static_cast<volatile uint32_t*>(host_err_);
  else if (hip_check(hipMemcpy(&err, sort_.err, 4, hipMemcpyDeviceToHost), "read sort flag")) return status_;
  if (err) return fail(PBD_ERR_HIP, "sort look-back exceeded its spin limit");
  return status_;
}

// ---------------------------------------------------------------------------
// buffers
static int elem_info(int which, size_t* elem, bool* table) {
  *table = false;
  switch (which) {
    case PBD_BUF_POSITIONS:
    case PBD_BUF_PREDICTED:
    case PBD_BUF_VELOCITIES:
    case PBD_BUF_COLORS:
    case PBD_BUF_EXTERNAL_FORCES:
    case PBD_BUF_OMEGAS:
    case PBD_BUF_DELTA_POSITIONS:
      *elem = 16;
      return PBD_OK;
    case PBD_BUF_DENSITIES:
    case PBD_BUF_LAMBDAS:
    case PBD_BUF_CELL_IDS:
    case PBD_BUF_PARTICLE_IDS:
    case PBD_BUF_NEIGHBOUR_COUNTERS:
    case PBD_BUF_CONTACT_COUNTERS:
      *elem = 4;
      return PBD_OK;
    case PBD_BUF_CELL_STARTS:
    case PBD_BUF_CELL_ENDINGS:
      *elem = 4;
      *table = true;
      return PBD_OK;
    case PBD_BUF_PHASES:
      *elem = 4;
      return PBD_OK;
    default:
      return PBD_ERR_INVALID;
  }
}

int Fluid::buffer_bytes(int which, size_t* bytes) const {
  size_t elem;
  bool table;
  if (elem_info(which, &elem, &table)) return PBD_ERR_INVALID;
  *bytes = elem * (table ? B_.table_size : n_);
  return PBD_OK;
}

int Fluid::download(int which, void* dst, size_t bytes) {
  size_t need;
  if (buffer_bytes(which, &need) || bytes > need || (bytes && !dst))
    return fail(PBD_ERR_INVALID, "download: bad buffer id or size");
  if (int rc = sync()) return rc;
  const void* src = nullptr;
  switch (which) {
    case PBD_BUF_POSITIONS: src = B_.X; break;
    case PBD_BUF_PREDICTED: src = B_.P; break;
    case PBD_BUF_VELOCITIES: src = B_.V; break;
    case PBD_BUF_COLORS: src = B_.C; break;
    case PBD_BUF_EXTERNAL_FORCES: src = B_.F; break;
    case PBD_BUF_DENSITIES: src = B_.DENS; break;
    case PBD_BUF_LAMBDAS: src = B_.LAM; break;
    case PBD_BUF_CELL_IDS: src = keys_sorted_; break;
    case PBD_BUF_PARTICLE_IDS: src = ids_sorted_; break;
    case PBD_BUF_CELL_STARTS: src = B_.cstart; break;
    case PBD_BUF_CELL_ENDINGS: src = B_.cend; break;
    case PBD_BUF_NEIGHBOUR_COUNTERS: src = B_.NCNT; break;
    case PBD_BUF_CONTACT_COUNTERS: src = B_.CCNT; break;
    case PBD_BUF_OMEGAS: src = B_.OM; break;
    case PBD_BUF_DELTA_POSITIONS: src = B_.DP; break;
    case PBD_BUF_PHASES: src = ph_; break;
  }
  if (bytes == 0) return PBD_OK;
  return hip_check(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "download");
}

int Fluid::download_range(int which, uint32_t first, uint32_t count, void* dst) {
  size_t esz = 0;
  const void* src = nullptr;
  switch (which) {
    case PBD_BUF_POSITIONS: src = B_.X; esz = 16; break;
    case PBD_BUF_PREDICTED: src = B_.P; esz = 16; break;
    case PBD_BUF_VELOCITIES: src = B_.V; esz = 16; break;
    case PBD_BUF_COLORS: src = B_.C; esz = 16; break;
    case PBD_BUF_EXTERNAL_FORCES: src = B_.F; esz = 16; break;
    case PBD_BUF_DENSITIES: src = B_.DENS; esz = 4; break;
    case PBD_BUF_LAMBDAS: src = B_.LAM; esz = 4; break;
    case PBD_BUF_NEIGHBOUR_COUNTERS: src = B_.NCNT; esz = 4; break;
    case PBD_BUF_CONTACT_COUNTERS: src = B_.CCNT; esz = 4; break;
    case PBD_BUF_OMEGAS: src = B_.OM; esz = 16; break;
    case PBD_BUF_DELTA_POSITIONS: src = B_.DP; esz = 16; break;
    case PBD_BUF_CELL_IDS: src = keys_sorted_; esz = 4; break;
    case PBD_BUF_PARTICLE_IDS: src = ids_sorted_; esz = 4; break;
    case PBD_BUF_PHASES: src = ph_; esz = 4; break;
    default: return fail(PBD_ERR_INVALID, "download: not a per-particle buffer");
  }
  if ((uint64_t)first + count > n_ || (count && !dst)) return fail(PBD_ERR_INVALID, "download: range exceeds particle count");
  if (int rc = sync()) return rc;
  if (count == 0) return PBD_OK;
  return hip_check(hipMemcpy(dst, static_cast<const char*>(src) + (size_t)first * esz, (size_t)count * esz,
                             hipMemcpyDeviceToHost),
                   "download");
}

int Fluid::set_phases(uint32_t first, uint32_t count, const uint32_t* phases) {
  if ((uint64_t)first + count > n_ || (count && !phases)) return fail(PBD_ERR_INVALID, "phases: range exceeds particle count");
  bool solid = false;
  for (uint32_t i = 0; i < count; ++i) {
    if (phases[i] > PBD_PHASE_SOLID) return fail(PBD_ERR_INVALID, "phases: values must be PBD_PHASE_FLUID or PBD_PHASE_SOLID");
    solid |= phases[i] == PBD_PHASE_SOLID;
  }
  if (int rc = sync()) return rc;
  if (count && hip_check(hipMemcpy(ph_ + first, phases, (size_t)count * 4, hipMemcpyHostToDevice), "phases upload"))
    return status_;
  // the per-particle path with phase masks stays on once a solid particle was seen
  if (solid && !has_solids_) {
    has_solids_ = true;
    dev_valid_ = false;
    invalidate_graph();
  }
  return PBD_OK;
}

int Fluid::upload(int which, const void* src, size_t bytes) {
  if (which == PBD_BUF_PHASES) {
    if (bytes > (size_t)n_ * 4 || (bytes % 4) != 0) return fail(PBD_ERR_INVALID, "upload: size exceeds particle count");
    return set_phases(0, (uint32_t)(bytes / 4), static_cast<const uint32_t*>(src));
  }
  void* dst = nullptr;
  switch (which) {
    case PBD_BUF_POSITIONS: dst = B_.X; break;
    case PBD_BUF_PREDICTED: dst = B_.P; break;
    case PBD_BUF_VELOCITIES: dst = B_.V; break;
    case PBD_BUF_COLORS: dst = B_.C; break;
    case PBD_BUF_EXTERNAL_FORCES: dst = B_.F; break;
    default: return fail(PBD_ERR_INVALID, "upload: only particle state buffers can be uploaded");
  }
  if (bytes > (size_t)n_ * 16 || (bytes && !src)) return fail(PBD_ERR_INVALID, "upload: size exceeds particle count");
  if (int rc = sync()) return rc;
  if (bytes == 0) return PBD_OK;
  return hip_check(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "upload");
}

int Fluid::check_finite(uint32_t* bad) {
  if (hip_check(hipMemsetAsync(d_scratch_, 0, 4, stream_), "memset")) return status_;
  if (hip_check(launch_check_finite(stream_, n_, B_.X, B_.V, d_scratch_), "check_finite")) return status_;
  uint32_t b = 0;
  if (hip_check(hipMemcpyAsync(&b, d_scratch_, 4, hipMemcpyDeviceToHost, stream_), "copy")) return status_;
  if (hip_check(hipStreamSynchronize(stream_), "sync")) return status_;
  if (bad) *bad = b;
  return b ? PBD_ERR_NONFINITE : PBD_OK;
}

void Fluid::get_buffers(pbd_buffers* out) const {
  out->positions4 = B_.X;
  out->predicted_positions4 = B_.P;
  out->velocities4 = B_.V;
  out->colors4 = B_.C;
  out->external_forces4 = B_.F;
  out->num_particles = n_;
  out->capacity = cap_;
}

}  // namespace pbd
