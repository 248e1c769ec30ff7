// fluid.hpp - host orchestrator of the PBF step.
//
// Mirrors the reference's step interface: Cuda_Computable::compute()
// (src/cuda/Cuda_Computable.h:8-18) implemented by Fluid (src/app/simulation/
// Fluid.h, Fluid.cu:4-97).  The constructor's allocation replaces
// cudaInitializeKernels (kernel/Initialize.h:122-130) and the GL-owned particle
// buffers of Particles (src/app/rendering/Particles.cc:26-143); compute() runs
// the stages of Fluid.cu:14-97 on one HIP stream with the same Active.* gates.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "adjoint.hpp"
#include "kernels.hpp"
#include "params.hpp"
#include "pbd/pbd.h"

namespace pbd {

class Cuda_Computable {
 public:
  virtual ~Cuda_Computable() = default;
  virtual void compute() = 0;
};

class Fluid : public Cuda_Computable {
 public:
  Fluid() = default;
  ~Fluid() override;
  Fluid(const Fluid&) = delete;
  Fluid& operator=(const Fluid&) = delete;

  // Allocate for `capacity` particles on the current device.
  int init(const pbd_params& p, uint32_t capacity);
  // Set up in a caller's device region instead (no allocation, no stream of
  // its own): up to `capacity` particles and a cell table of up to table_cap
  // entries; the public arrays are lent per step (compute_in_place).
  int init_in_place(const pbd_params& p, uint32_t capacity, uint32_t table_cap, unsigned char* region, size_t bytes,
                    hipStream_t st);
  int compute_in_place(const pbd_params& p, uint32_t n, float4* X, float4* P, float4* V, float4* C, float4* F,
                       hipStream_t st);
  int set_params(const pbd_params& p);
  const pbd_params& params() const { return params_; }

  // One substep (Fluid::compute).  Errors are kept in status().
  void compute() override;
  // frames x substeps calls of compute(); graph = replay a captured substep.
  int step(uint32_t frames, bool graph);
  int sync();

  int add_particles(uint32_t n, const float* pos4, const float* vel4, const float* col4);
  int clear_particles();
  uint32_t num_particles() const { return n_; }
  uint32_t capacity() const { return cap_; }

  int download(int which, void* dst, size_t bytes);
  // count elements of a per-particle buffer from index first (sorted order)
  int download_range(int which, uint32_t first, uint32_t count, void* dst);
  int upload(int which, const void* src, size_t bytes);
  // phases of particles [first, first + count) (PBD_PHASE_*)
  int set_phases(uint32_t first, uint32_t count, const uint32_t* phases);
  bool phased() const { return has_solids_ || params_.friction_static > 0.0f; }
  int buffer_bytes(int which, size_t* bytes) const;
  int check_finite(uint32_t* bad);
  void get_buffers(pbd_buffers* out) const;

  void set_timing(bool on) { timing_ = on; }
  int timings(const char** names, double* ms, uint64_t* launches, uint32_t cap, uint32_t* count);
  void reset_timings();
  int counters(uint64_t* values, uint32_t cap, uint32_t* count);
  int reset_counters();

  // Launch shape (tune.cpp): how the step is launched, never what it computes.
  struct LaunchShape {
    uint32_t tpb, tile_bits, sort_items, small_max, stride_grid, skin_pct;
  };
  LaunchShape launch_shape() const;
  int set_launch_shape(const LaunchShape& s);
  // Time trial_steps graph launches per candidate from the current state
  // (restored after each trial) and keep the fastest; ms_* may be null.
  int autotune(uint32_t trial_steps, LaunchShape* chosen, double* ms_chosen, double* ms_default);

  // Batched scenes: the device table of n scene constants and the slot size
  // (owned by the caller, alive as long as the context).
  void set_scenes(const SceneParams* table, const uint32_t* first, uint32_t n, uint32_t slot_log2);
  hipStream_t stream() const { return stream_; }

  // Reverse mode (adjoint_host.cpp): a checkpointed forward of `frames` frames,
  // then the gradients of a loss of the final state.
  int adj_forward(uint32_t frames, uint32_t k_ckpt);
  int adj_ids(uint32_t* dst, size_t count);
  // the reverse passes take their lists from the recorded steps' tile lists (true) or build them
  void adj_set_lists(bool from_forward) { adj_lists_from_forward_ = from_forward; }
  int adj_backward(const float* gx, const float* gv, float* gv0, float* grho0, float* geps, float* gx0);

  // Record an error of a call made on this context (pbd_last_error).
  int report(int code, const std::string& msg) { return fail(code, msg); }
  int status() const { return status_; }
  const std::string& error() const { return error_; }
  void clear_status() {
    status_ = PBD_OK;
    error_.clear();
  }

 private:
  int fail(int code, const std::string& msg);
  int hip_check(hipError_t e, const char* what);
  std::string tune_key() const;
  int time_shape(const LaunchShape& s, uint32_t steps, double* ms);
  template <class T>
  int take(T** p, size_t count);
  int layout();
  int alloc_table();
  int ensure_batch_buffers();
  void apply_context();
  int enqueue_substep();
  int ensure_graph();
  int adj_check();
  void adj_release();
  int tape_copy(const CopySet& set);
  void stage_begin(int stage);
  void stage_end(int stage);
  int collect_timings();
  void invalidate_graph();

  pbd_params params_{};
  DevParams dev_{};
  bool dev_valid_ = false;
  uint32_t n_ = 0;
  uint32_t cap_ = 0;
  uint32_t tpb_ = 256;
  hipStream_t stream_ = nullptr;
  bool owns_stream_ = false;
  uint32_t small_max_ = kTileSmall;       // blocks of at most this many particles take one wave
  bool small_auto_ = true;                 // until a launch shape is set: default_small_max(n_)
  uint32_t small_max() const { return small_auto_ ? default_small_max(n_) : small_max_; }
  uint32_t small_tiles() const { return small_tile_limit(small_max()); }  // as the compaction makes them
  uint32_t stride_grid_ = kTileGridStride;  // workgroups of the capped tile grid
  uint32_t skin_pct_ = kListSkinPct;       // tile-list skin, percent of the list radius
  uint32_t* host_err_ = nullptr;           // the sort's error flag (pinned), unless the context lies in a region
  bool tuned_ = false;                     // autotune ran (or a cached choice was applied)
  // a caller's region the buffers are carved from (init_in_place), else null
  unsigned char* region_ = nullptr;
  size_t region_size_ = 0, region_used_ = 0;
  uint32_t region_table_ = 0;
  StepBuffers B_{};
  SortPlan sort_{};
  const uint32_t* keys_sorted_ = nullptr;
  const uint32_t* ids_sorted_ = nullptr;
  uint32_t* d_scratch_ = nullptr;  // small device scratch: [0] finite count, [1] unused
  uint32_t* tile_list_ = nullptr;   // occupied Morton blocks of the step: large tiles, then (at cap_) small ones
  uint32_t* tile_count_ = nullptr;  // [0] large, [1] small tiles
  uint32_t* tile_flag_ = nullptr;   // per Morton block: 1 + first sorted index, 0 if empty this step
  uint32_t* tile_end_ = nullptr;    // per occupied Morton block: 1 + last sorted index
  uint32_t* tile_bcount_ = nullptr;  // compaction block counts
  uint32_t* batch_solved_ = nullptr;   // collisionType 1 (allocated on first use)
  unsigned long long* batch_min_ = nullptr;
  uint32_t* batch_partner_ = nullptr;
  uint32_t batch_words_ = 0;
  const SceneParams* scene_table_ = nullptr;  // batched scenes
  const uint32_t* scene_first_ = nullptr;
  uint32_t scene_count_ = 1, slot_log2_ = 10;
  uint32_t* ph_ = nullptr;   // public phases (PBD_BUF_PHASES)
  uint32_t* phs_ = nullptr;  // phases in the step's sorted order
  bool has_solids_ = false;

  // reverse mode: checkpoints, the record of one segment and the work
  // buffers (allocated by adj_forward); rec_ is the step record being written
  struct AdjState;
  AdjState* adj_ = nullptr;
  AdjTape* rec_ = nullptr;
  bool adj_lists_from_forward_ = true;

  // graph of one substep
  hipGraph_t graph_ = nullptr;
  hipGraphExec_t graph_exec_ = nullptr;
  bool graph_valid_ = false;

  // timing
  bool timing_ = false;
  struct Pending {
    int stage;
    hipEvent_t a, b;
  };
  std::vector<Pending> pending_;
  std::vector<hipEvent_t> event_pool_;
  hipEvent_t cur_begin_ = nullptr;
  std::vector<double> stage_ms_;
  std::vector<uint64_t> stage_launches_;

  int status_ = PBD_OK;
  std::string error_;
  std::vector<void*> allocations_;
};

// Stage names used by the timers.
enum Stage {
  ST_PREDICT = 0,
  ST_CELL_RESET,
  ST_SORT,
  ST_REORDER,
  ST_TILES,
  ST_LAMBDA,
  ST_DELTA,
  ST_COLLIDE,
  ST_UPDATE,
  ST_COUNT,
  ST_OMEGA,
  ST_FINAL,
  ST_LAMBDA_CARRY,  // lambda passes that may keep the lists of an earlier pass
  ST_NUM
};
extern const char* const kStageNames[ST_NUM];

}  // namespace pbd
