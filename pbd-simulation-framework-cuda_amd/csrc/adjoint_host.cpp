// adjoint_host.cpp - host side of the reverse mode: checkpoints, segment
// recomputation with a step record, and the reverse passes (adjoint.hip).
//
// adj_forward runs `frames` frames (frames x substeps computes, one graph
// launch each) and keeps the state (positions, velocities, external forces) at
// the start of every k-th frame; the steps of the last segment run eagerly and
// write their records (AdjTape) on the way.  adj_backward walks the segments
// last first: it restores the segment's checkpoint, recomputes its steps
// eagerly while every step writes its record (skipped for the last segment
// while the forward's records are still there), and runs the reverse kernels
// of the steps last first.  The recomputation replays the same kernels on the same
// inputs, so it reproduces the forward bit for bit.
#include <algorithm>
#include <cstring>
#include <sstream>
#include <vector>

#include "fluid.hpp"

namespace pbd {

struct Fluid::AdjState {
  uint32_t n = 0, frames = 0, k = 0, sub = 0, iters = 0, stab = 0, nseg = 0, nrec = 0, table = 0;
  std::vector<void*> mem;
  std::vector<float4*> ckpt;    // per checkpoint: X | V | F (3n float4)
  std::vector<uint32_t*> ckpt_ph;  // per checkpoint: the phases in the same order (phased contexts)
  float4* final_state = nullptr;  // X | P | V | C | F after the forward
  uint32_t* final_ph = nullptr;   // phases after the forward (phased contexts)
  bool phased = false, friction = false;
  bool keep_lists = false;  // the records keep the forward's tile lists (AdjTape::NL)
  std::vector<AdjTape> tape;    // records of one segment
  AdjWork W{};
  uint32_t* ids[2] = {nullptr, nullptr};
  int ids_cur = 0;
  double* red = nullptr;  // 2 doubles
  // pinned staging of pbd_adj_backward's host arrays: dL/dx, dL/dv in, dL/dv0,
  // dL/dx0 out (n float4 each; null: the copies go to and from the caller's
  // memory directly)
  float4* pin = nullptr;
  bool valid = false;
  bool tail_recorded = false;  // the records hold the last segment (written by the forward)
  pbd_params params{};

  ~AdjState() {
    for (void* p : mem) (void)hipFree(p);
    if (pin) (void)hipHostFree(pin);
  }
  template <class T>
  bool alloc(T** p, size_t count) {
    void* q = nullptr;
    if (hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) return false;
    mem.push_back(q);
    *p = static_cast<T*>(q);
    return true;
  }
};

void Fluid::adj_release() {
  delete adj_;
  adj_ = nullptr;
}

// The reverse kernels cover the textbook step with particle collisions of
// type 0 (at most one stabilization pass) and every stage active.
int Fluid::adj_check() {
  const pbd_params& p = params_;
  if (p.kernel_variant != PBD_KERNEL_TEXTBOOK)
    return fail(PBD_ERR_UNSUPPORTED, "adjoint: only Density.kernelVariant = textbook is differentiated");
  if (p.collision_type != 0 || p.stabilization_iterations > 1)
    return fail(PBD_ERR_UNSUPPORTED, "adjoint: collisionType 0 with at most one stabilization iteration");
  if (p.solver_iterations == 0) return fail(PBD_ERR_UNSUPPORTED, "adjoint: at least one solver iteration");
  if (!p.active_apply_forces || !p.active_find_contacts || !p.active_compute_lambda ||
      !p.active_compute_delta_positions || !p.active_apply_delta_positions || !p.active_update_positions ||
      !p.active_compute_omegas || !p.active_compute_vorticity || !p.active_compute_viscosity)
    return fail(PBD_ERR_UNSUPPORTED, "adjoint: every Active.* stage but findNeighbours must be on");
  if (scene_table_) return fail(PBD_ERR_UNSUPPORTED, "adjoint: not available for batched scenes");
  if (n_ == 0) return fail(PBD_ERR_INVALID, "adjoint: no particles");
  return PBD_OK;
}

int Fluid::adj_forward(uint32_t frames, uint32_t k_ckpt) {
  if (status_ != PBD_OK) return status_;
  if (int rc = adj_check()) return rc;
  if (frames == 0 || k_ckpt == 0) return fail(PBD_ERR_INVALID, "adjoint: frames and the checkpoint interval must be > 0");
  if (int rc = sync()) return rc;
  if (!dev_valid_) {
    const char* why = nullptr;
    if (derive_device_params(params_, n_, dev_, &why) != PBD_OK) return fail(PBD_ERR_INVALID, why);
    apply_context();
    dev_valid_ = true;
  }
  const uint32_t k = std::min(k_ckpt, frames);
  const uint32_t sub = params_.substeps ? params_.substeps : 1;
  const uint32_t nseg = (frames + k - 1) / k, nrec = k * sub;
  // phases: the records hold each step's sorted phases, and with friction x at
  // every iteration's start; checkpoints keep the phases in the state's order
  const bool ph = phased();
  const bool fr = ph && params_.friction_static > 0.0f && params_.stabilization_iterations > 0;
  // a previous forward of the same shape leaves buffers of the right sizes: reuse them
  const bool reuse = adj_ && adj_->n == n_ && adj_->nseg == nseg && adj_->nrec == nrec &&
                     adj_->iters == params_.solver_iterations && adj_->table == B_.table_size &&
                     adj_->phased == ph && adj_->friction == fr && adj_->keep_lists == adj_lists_from_forward_;
  if (!reuse) {
    adj_release();
    adj_ = new AdjState();
  }
  AdjState& A = *adj_;
  A.n = n_;
  A.frames = frames;
  A.k = k;
  A.sub = sub;
  A.iters = params_.solver_iterations;
  A.stab = params_.stabilization_iterations;
  A.nseg = nseg;
  A.nrec = nrec;
  A.table = B_.table_size;
  A.params = params_;
  A.phased = ph;
  A.friction = fr;
  A.keep_lists = adj_lists_from_forward_;
  A.valid = false;
  A.tail_recorded = false;
  const size_t n = n_;
  bool ok = true;
  if (!reuse) {
    A.ckpt.assign(A.nseg, nullptr);
    A.ckpt_ph.assign(A.nseg, nullptr);
    for (uint32_t g = 0; g < A.nseg && ok; ++g) ok = A.alloc(&A.ckpt[g], 3 * n) && (!A.phased || A.alloc(&A.ckpt_ph[g], n));
    ok = ok && A.alloc(&A.final_state, 5 * n) && (!A.phased || A.alloc(&A.final_ph, n));
    A.tape.assign(A.nrec, AdjTape{});
    for (uint32_t t = 0; t < A.nrec && ok; ++t) {
      AdjTape& T = A.tape[t];
      ok = A.alloc(&T.Q, (size_t)(A.iters + 1) * n) && A.alloc(&T.LAM, (size_t)A.iters * n) && A.alloc(&T.U, n) &&
           A.alloc(&T.OM, n) && A.alloc(&T.keys, n) && A.alloc(&T.perm, n) && A.alloc(&T.cs, A.table) &&
           A.alloc(&T.ce, A.table) && A.alloc(&T.Xin, n) && A.alloc(&T.Vin, n) && A.alloc(&T.Fin, n) &&
           (!A.phased || A.alloc(&T.PH, n)) && (!A.friction || A.alloc(&T.QX, (size_t)A.iters * n));
    }
    AdjWork& W = A.W;
    W.table = A.table;
    W.stats = B_.STATS;
    ok = ok && A.alloc(&W.GX, n) && A.alloc(&W.GV, n) && A.alloc(&W.GF, n) && A.alloc(&W.Ub, n) && A.alloc(&W.Xp, n) &&
         A.alloc(&W.Eb, n) && A.alloc(&W.Ob, n) && A.alloc(&W.Pb, n) && A.alloc(&W.Xb, n) && A.alloc(&W.DPb, n) &&
         A.alloc(&W.PUb, n) && A.alloc(&W.AB, n) && A.alloc(&W.Pn, n) && A.alloc(&W.QR, n) && A.alloc(&W.acc, n) &&
         A.alloc(&W.flag, 1) && A.alloc(&A.ids[0], n) && A.alloc(&A.ids[1], n) && A.alloc(&A.red, kAdjReduceWords) &&
         (!A.friction || A.alloc(&W.XF, n)) &&
         (n_ < kAdjListMinParticles ||
          (A.alloc(&W.LE, adjoint_list_entries(n_)) && A.alloc(&W.LC, adjoint_list_counts(n_)) &&
           A.alloc(&W.redo, adjoint_redo_words(A.table))));
  }
  if (!ok) {
    adj_release();
    return fail(PBD_ERR_NOMEM, "adjoint: device allocation of checkpoints and step records failed");
  }
  // Host copies of pbd_adj_backward through pinned memory: a DMA from pageable
  // memory stages it in small pieces (the 64K scene's downloads took longer
  // than half its reverse passes).  Optional.
  if (!reuse && hipHostMalloc((void**)&A.pin, 4 * n * sizeof(float4), hipHostMallocDefault) != hipSuccess) {
    A.pin = nullptr;
    (void)hipGetLastError();
  }
  // The forward's tile lists of every recorded step, from which the reverse
  // passes take their lists (64 + 128 (iters + 1) B per particle and step).
  // Optional: without the memory the reverse passes build their lists.
  if (!reuse && A.keep_lists && n_ >= kAdjListMinParticles) {
    std::vector<void*> got;
    bool all = true;
    for (uint32_t t = 0; t < A.nrec && all; ++t) {
      void* a = nullptr;
      void* b = nullptr;
      all = hipMalloc(&a, adjoint_record_chunks(n_, A.iters) * sizeof(uint4)) == hipSuccess &&
            hipMalloc(&b, (size_t)(A.iters + 1) * n * sizeof(uint16_t)) == hipSuccess;
      for (void* q : {a, b})
        if (q) got.push_back(q);
      if (all) {
        A.tape[t].NL = static_cast<uint4*>(a);
        A.tape[t].NLC = static_cast<uint16_t*>(b);
      }
    }
    if (all) {
      A.mem.insert(A.mem.end(), got.begin(), got.end());
    } else {
      for (void* q : got) (void)hipFree(q);
      for (AdjTape& T : A.tape) {
        T.NL = nullptr;
        T.NLC = nullptr;
      }
      (void)hipGetLastError();  // the failed allocation is not an error of the step
    }
  }
  if (hip_check(launch_gather_ids(stream_, n_, nullptr, nullptr, A.ids[0]), "adjoint ids")) return status_;
  A.ids_cur = 0;
  auto save = [&](uint32_t g) {
    float4* dst = A.ckpt[g];
    CopySet set;
    set.add(dst, B_.X, n * 16).add(dst + n, B_.V, n * 16).add(dst + 2 * n, B_.F, n * 16);
    if (A.phased) set.add(A.ckpt_ph[g], ph_, n * 4);
    return tape_copy(set);
  };
  if (save(0)) return status_;
  if (int rc = ensure_graph()) return rc;
  // The last segment's steps write their records as they run (eagerly, the
  // same kernels as the graph), so the reverse pass starts without recomputing it.
  const uint32_t tail = (A.nseg - 1) * A.k;
  for (uint32_t f = 0; f < frames; ++f) {
    for (uint32_t s = 0; s < A.sub; ++s) {
      if (f >= tail) {
        rec_ = &A.tape[(f - tail) * A.sub + s];
        compute();
        rec_ = nullptr;
        if (status_ != PBD_OK) return status_;
      } else if (hip_check(hipGraphLaunch(graph_exec_, stream_), "hipGraphLaunch")) {
        return status_;
      }
      if (hip_check(launch_gather_ids(stream_, n_, ids_sorted_, A.ids[A.ids_cur], A.ids[1 - A.ids_cur]), "ids"))
        return status_;
      A.ids_cur = 1 - A.ids_cur;
    }
    if ((f + 1) % A.k == 0 && f + 1 < frames && save((f + 1) / A.k)) return status_;
  }
  A.tail_recorded = true;
  float4* fs = A.final_state;
  CopySet set;
  set.add(fs, B_.X, n * 16).add(fs + n, B_.P, n * 16).add(fs + 2 * n, B_.V, n * 16);
  set.add(fs + 3 * n, B_.C, n * 16).add(fs + 4 * n, B_.F, n * 16);
  if (A.phased) set.add(A.final_ph, ph_, n * 4);
  if (tape_copy(set)) return status_;
  A.valid = true;
  return PBD_OK;
}

int Fluid::adj_ids(uint32_t* dst, size_t count) {
  if (!adj_ || !adj_->valid) return fail(PBD_ERR_INVALID, "adjoint: run pbd_adj_forward first");
  if (count > adj_->n || (count && !dst)) return fail(PBD_ERR_INVALID, "adjoint: ids count exceeds particle count");
  if (int rc = sync()) return rc;
  if (count == 0) return PBD_OK;
  return hip_check(hipMemcpy(dst, adj_->ids[adj_->ids_cur], count * 4, hipMemcpyDeviceToHost), "adjoint ids");
}

int Fluid::adj_backward(const float* gx, const float* gv, float* gv0, float* grho0, float* geps, float* gx0) {
  if (status_ != PBD_OK) return status_;
  if (!adj_ || !adj_->valid) return fail(PBD_ERR_INVALID, "adjoint: run pbd_adj_forward first");
  AdjState& A = *adj_;
  if (A.n != n_ || std::memcmp(&A.params, &params_, sizeof(pbd_params)) != 0)
    return fail(PBD_ERR_INVALID, "adjoint: particles or parameters changed since pbd_adj_forward");
  const size_t n = n_;
  const AdjWork& W = A.W;
  hipError_t e = hipSuccess;
  // the caller's arrays are read here, before the copies run
  float4* pin = A.pin;
  const auto upload = [&](float4* dst, const float* src, float4* stage) {
    if (!pin) return hipMemcpyAsync(dst, src, n * 16, hipMemcpyHostToDevice, stream_);
    std::memcpy(stage, src, n * 16);
    return hipMemcpyAsync(dst, stage, n * 16, hipMemcpyHostToDevice, stream_);
  };
  if (gx) e = upload(W.GX, gx, pin);
  if (e == hipSuccess && gv) e = upload(W.GV, gv, pin ? pin + n : nullptr);
  CopySet zero;
  if (!gx) zero.add(W.GX, nullptr, n * 16);
  if (!gv) zero.add(W.GV, nullptr, n * 16);
  zero.add(W.GF, nullptr, n * 16).add(W.acc, nullptr, n * sizeof(double2)).add(W.flag, nullptr, 4);
  if (e == hipSuccess) e = launch_copy_set(stream_, zero);
  if (hip_check(e, "adjoint: upload of the loss adjoints")) return status_;
  for (uint32_t g = A.nseg; g-- > 0;) {
    const uint32_t nstep = (std::min(A.frames, (g + 1) * A.k) - g * A.k) * A.sub;
    if (g + 1 < A.nseg || !A.tail_recorded) {
      const float4* c = A.ckpt[g];
      CopySet set;
      set.add(B_.X, c, n * 16).add(B_.V, c + n, n * 16).add(B_.F, c + 2 * n, n * 16);
      if (A.phased) set.add(ph_, A.ckpt_ph[g], n * 4);
      if (tape_copy(set)) return status_;
      for (uint32_t t = 0; t < nstep; ++t) {
        rec_ = &A.tape[t];
        compute();
        rec_ = nullptr;
        if (status_ != PBD_OK) return status_;
      }
      A.tail_recorded = false;  // the records now hold segment g
    }
    for (uint32_t t = nstep; t-- > 0;)
      if (hip_check(launch_adjoint_step(stream_, dev_, A.iters, A.stab, A.tape[t], W), "adjoint step"))
        return status_;
  }
  if (hip_check(launch_adjoint_reduce(stream_, n_, W.acc, A.red), "adjoint reduce")) return status_;
  double red[2] = {0.0, 0.0};
  uint32_t flag = 0;
  e = hipMemcpyAsync(red, A.red, sizeof(red), hipMemcpyDeviceToHost, stream_);
  if (e == hipSuccess) e = hipMemcpyAsync(&flag, W.flag, 4, hipMemcpyDeviceToHost, stream_);
  if (e == hipSuccess && gv0)
    e = hipMemcpyAsync(pin ? (void*)(pin + 2 * n) : (void*)gv0, W.GV, n * 16, hipMemcpyDeviceToHost, stream_);
  if (e == hipSuccess && gx0)
    e = hipMemcpyAsync(pin ? (void*)(pin + 3 * n) : (void*)gx0, W.GX, n * 16, hipMemcpyDeviceToHost, stream_);
  // leave the context as pbd_adj_forward left it
  const float4* fs = A.final_state;
  CopySet set;
  set.add(B_.X, fs, n * 16).add(B_.P, fs + n, n * 16).add(B_.V, fs + 2 * n, n * 16);
  set.add(B_.C, fs + 3 * n, n * 16).add(B_.F, fs + 4 * n, n * 16);
  if (A.phased) set.add(ph_, A.final_ph, n * 4);
  if (e == hipSuccess) e = launch_copy_set(stream_, set);
  if (e == hipSuccess) e = hipStreamSynchronize(stream_);
  if (hip_check(e, "adjoint: results")) return status_;
  if (pin && gv0) std::memcpy(gv0, pin + 2 * n, n * 16);
  if (pin && gx0) std::memcpy(gx0, pin + 3 * n, n * 16);
  if (grho0) *grho0 = (float)red[0];
  if (geps) *geps = (float)red[1];
  if (flag)
    return fail(PBD_ERR_UNSUPPORTED,
                "adjoint: a neighbour list reached maxNeighboursPerParticle (the capped relation is not symmetric)");
  return PBD_OK;
}

}  // namespace pbd
