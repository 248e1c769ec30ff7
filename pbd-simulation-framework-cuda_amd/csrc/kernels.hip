// kernels.hip - gfx950 kernels of the PBF step (everything but the sort).
//
// Data layout during a step (all arrays in sorted order, float4 = 16 B):
//   Q   (p* - corner(cell), p*.w)   predicted position in cell-local coordinates
//   QX  (x  - corner(cell), x.w)    position in cell-local coordinates
//   VS  velocity
//   LAM lambda (float), DP delta p (float4), OM omega (float4)
// Working in cell-local coordinates keeps every FP32 position update at the
// resolution of the cell instead of the world box: the Jacobi updates
// p* +- dp round at ulp(0.1) rather than ulp(12.8).  The public buffers
// positions4 / predictedPositions4 / velocities4 / colors4 are read once by the
// reorder gather and written once by the final kernel.
//
// Reference kernels restated (src/app/simulation/kernel/):
//   k_predict_keys  applyForces + initializeCellIds   Forces.h:65-101, SortReorder.h:13-28
//   k_reorder       copy + reorder + computeCellInfo   SortReorder.h:53-129,160-188
//   k_lambda        computeLambda (+ neighbour counts, density)  Density.h:48-93, Collision.h:11-160
//   k_delta         computeDeltaPositions + solveCollisions + applyDeltaPositions (+ updatePositions)
//                   Density.h:104-168, Collision.h:171-285, Update.h:11-32
//   k_omega         computeOmega                       Density.h:232-269
//   k_final         computeVorticity + computeViscosity + output   Density.h:179-221,280-310
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "particle_ops.hpp"

namespace pbd {

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint32_t n) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// A step's record and the adjoint's restores move up to ten arrays between the same two
// kernels, and a step without a context clears five.  A copy of its own each took 4.8 us at
// 64K particles (1 MB: launch and latency) and a call on the host; together they are one
// launch (adjoint of two 64K substeps: 2865 to 2751 us, with the positions written to the
// record directly; a 2K step's clears: 5 launches of 2 us to one).  16 bytes a thread where
// both sides are aligned to that, the rest in words.
__global__ void k_copy_set(CopySet c) {
  const size_t stride = (size_t)gridDim.x * blockDim.x, first = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t k = 0; k < c.count; ++k) {
    const uintptr_t d = reinterpret_cast<uintptr_t>(c.dst[k]), s = reinterpret_cast<uintptr_t>(c.src[k]);
    const size_t nv = ((d | s) & 15u) == 0u ? c.bytes[k] / 16u : 0u, nw = c.bytes[k] / 4u;
    uint4* dv = static_cast<uint4*>(c.dst[k]);
    const uint4* sv = static_cast<const uint4*>(c.src[k]);
    for (size_t i = first; i < nv; i += stride) dv[i] = s ? sv[i] : make_uint4(0u, 0u, 0u, 0u);
    uint32_t* dw = static_cast<uint32_t*>(c.dst[k]);
    const uint32_t* sw = static_cast<const uint32_t*>(c.src[k]);
    for (size_t i = 4u * nv + first; i < nw; i += stride) dw[i] = s ? sw[i] : 0u;
  }
}

// ---------------------------------------------------------------------------
// Adds the digits of `passes` 8-bit passes of the lanes' keys to the
// workgroup's histogram h.  The keys arrive in the previous step's sorted
// order, so equal digits sit in runs of neighbouring lanes: the first lane of a
// run adds the run's length (valid lanes are a prefix of the wave).
__device__ __forceinline__ void hist_add(uint32_t (*h)[256], uint32_t key, bool valid, uint32_t passes) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t live = __ballot(valid);
  if (live == 0ull) return;  // uniform over the wave
  const uint32_t nlive = (uint32_t)__popcll(live);
  for (uint32_t p = 0; p < passes; ++p) {
    const uint32_t d = (key >> (8u * p)) & 255u;
    const uint32_t prev = (uint32_t)__shfl_up((int)d, 1);
    const bool head = valid && (lane == 0u || d != prev);
    const uint64_t heads = __ballot(head);
    if (head) {
      const uint64_t after = heads & ~((2ull << lane) - 1ull);
      const uint32_t end = after ? (uint32_t)(__ffsll((unsigned long long)after) - 1) : nlive;
      atomicAdd(&h[p][d], end - lane);
    }
  }
}

// applyForces + initializeCellIds, fused, and the sort's digit counts.  The
// predicted state itself is not stored: the reorder gather recomputes it with
// the same FP32 operations.
__global__ void k_predict_keys(DevParams P, const float4* __restrict__ X, const float4* __restrict__ V,
                               const float4* __restrict__ F, const float4* __restrict__ Pold,
                               uint32_t* __restrict__ keys, uint32_t* __restrict__ hist, uint32_t passes,
                               uint32_t copies) {
  __shared__ uint32_t h[4][256];
  for (uint32_t k = threadIdx.x; k < 4u * 256u; k += blockDim.x) (&h[0][0])[k] = 0u;
  __syncthreads();
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < P.n;
  uint32_t key = 0;
  if (valid) {
    const uint32_t sc = scene_of_index(P, i);
    float4 p;
    if (P.gates & G_APPLY_FORCES) {
      float4 x = X[i], v = V[i];
      predict(P, sc, x, v, F[i], p);
    } else {
      p = Pold[i];
    }
    uint32_t ix, iy, iz;
    key = cell_key(P, sc, p.x, p.y, p.z, ix, iy, iz);
    keys[i] = key;
  }
  hist_add(h, key, valid, passes);
  __syncthreads();
  uint32_t* part = hist + 1024u * (1u + blockIdx.x % copies);
  for (uint32_t k = threadIdx.x; k < passes * 256u; k += blockDim.x) {
    const uint32_t c = (&h[0][0])[k];
    if (c) atomicAdd(&part[k], c);
  }
}

// ---------------------------------------------------------------------------
// Reorder gather + cell ranges.  Cell boundaries are found per wavefront: each
// lane compares its key with the previous lane's (DPP/bpermute shuffle), lane 0
// with the previous wave's last key.
__global__ void k_reorder(DevParams P, const uint32_t* __restrict__ keys_s, const uint32_t* __restrict__ ids_s,
                          const float4* __restrict__ X, const float4* __restrict__ V, const float4* __restrict__ F,
                          const float4* __restrict__ Pold, const float4* __restrict__ C, float4* __restrict__ Q,
                          float4* __restrict__ QX, float4* __restrict__ VS, float4* __restrict__ CS,
                          uint32_t* __restrict__ cstart, uint32_t* __restrict__ cend, uint32_t tile_bits,
                          uint32_t* __restrict__ tile_start, uint32_t* __restrict__ tile_end) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  const uint32_t key = keys_s[s];
  uint32_t prev = __shfl_up(key, 1);
  if ((threadIdx.x & (warpSize - 1)) == 0) prev = s ? keys_s[s - 1] : 0xFFFFFFFFu;
  if (key != prev) {
    cstart[key] = s;
    if (s) cend[prev] = s;
    // first particle of an occupied Morton block of 2^tile_bits cells; the
    // previous block ends here
    if (tile_bits && (s == 0 || (key >> tile_bits) != (prev >> tile_bits))) {
      tile_start[key >> tile_bits] = s + 1u;
      if (s) tile_end[prev >> tile_bits] = s;
    }
  }
  if (tile_bits && s == P.n - 1u) tile_end[key >> tile_bits] = P.n;
  uint32_t j = ids_s[s];
  if (j >= P.n) j = P.n - 1;  // ids are a permutation of [0, n); the clamp only bounds a failed sort
  // the sorted key is the cell of the recomputed p* (same FP32 operations as
  // k_predict_keys); its slot names the scene
  const uint32_t sc = scene_of_key(P, key);
  float4 x = X[j], v = V[j], p;
  if (P.gates & G_APPLY_FORCES) {
    predict(P, sc, x, v, F[j], p);
  } else {
    p = Pold[j];
  }
  const float cx = frame_corner(P, frame_origin(P, sc, 0), compact10(key >> 2));
  const float cy = frame_corner(P, frame_origin(P, sc, 1), compact10(key >> 1));
  const float cz = frame_corner(P, frame_origin(P, sc, 2), compact10(key));
  Q[s] = make_float4(canonical_nan(p.x - cx), canonical_nan(p.y - cy), canonical_nan(p.z - cz), p.w);
  QX[s] = make_float4(x.x - cx, x.y - cy, x.z - cz, x.w);
  VS[s] = v;
  if (!(P.gates & G_FIND_NEIGHBOURS)) CS[s] = C[j];
  if (P.phs) P.phs[s] = P.ph[j];
}

// ---------------------------------------------------------------------------
// computeLambda.  FIRST also writes the neighbour / contact counts
// (findContacts + findNeighbours) and the density of the pass.
template <int VAR, bool FIRST>
__global__ void k_lambda(DevParams P, const float4* __restrict__ Q, const uint32_t* __restrict__ keys,
                         const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce, float* __restrict__ lam,
                         float* __restrict__ dens, uint32_t* __restrict__ ncnt, uint32_t* __restrict__ ccnt) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  lambda_particle<VAR, FIRST>(P, s, Q, keys, cs, ce, lam, dens, ncnt, ccnt);
}

// Neighbour / contact counts only (when computeLambda does not run first).
__global__ void k_count(DevParams P, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                        const uint32_t* __restrict__ ce, uint32_t* __restrict__ ncnt, uint32_t* __restrict__ ccnt) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  const CellFrame f = make_frame(P, keys[s]);
  uint32_t nc = 0;
  const uint32_t cnt =
      visit_neighbours(P, s, f, 0.0f, 0.0f, 0.0f, (P.gates & G_FIND_CONTACTS) != 0,
                       (P.gates & G_FIND_NEIGHBOURS) != 0, cs, ce, nc, [&](uint32_t, float, float, float, bool) {});
  ncnt[s] = cnt;
  ccnt[s] = nc;
}

// ---------------------------------------------------------------------------
// computeDeltaPositions (DELTA) + one collision pass (COLLIDE, gather over the
// contact cells with the pre-pass state: Jacobi) + applyDeltaPositions
// (flags & DF_APPLY) + updatePositions (flags & DF_UPDATE).  Reads Q/QX,
// writes Qo/QXo (ping-pong).  Without DELTA the stored DP is applied.
template <int VAR, bool DELTA, bool COLLIDE>
__global__ void k_delta(DevParams P, uint32_t flags, const float4* __restrict__ Q, const float4* __restrict__ QX,
                        const float* __restrict__ lam, const uint32_t* __restrict__ keys,
                        const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce, float4* __restrict__ Qo,
                        float4* __restrict__ QXo, float4* __restrict__ DP, float4* __restrict__ VS) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  delta_particle<VAR, DELTA, COLLIDE>(P, flags, s, Q, QX, lam, keys, cs, ce, Qo, QXo, DP, VS);
}

// updatePositions alone (Update.h:11-32): v = (p* - x)/dt, x = p*.
__global__ void k_update(DevParams P, const float4* __restrict__ Q, float4* __restrict__ QX, float4* __restrict__ VS) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  const float4 q = Q[s], x = QX[s];
  VS[s] = make_float4((q.x - x.x) / P.dt, (q.y - x.y) / P.dt, (q.z - x.z) / P.dt, (q.w - x.w) / P.dt);
  QX[s] = q;
}

// ---------------------------------------------------------------------------
// computeOmega: reference omega_i = sum (v_j - v_i) x grad(p_i - p_j);
// textbook omega_i = (1/rho0) sum v_ij x grad_j W_ij (SPH curl with the
// particle volume m/rho0, mass 1).  w holds |omega_i|.
template <int VAR>
__global__ void k_omega(DevParams P, const float4* __restrict__ Q, const float4* __restrict__ VS,
                        const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                        const uint32_t* __restrict__ ce, float4* __restrict__ OM) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  omega_particle<VAR>(P, s, Q, VS, keys, cs, ce, OM);
}

// ---------------------------------------------------------------------------
// computeVorticity (flags & FF_VORT) + computeViscosity (flags & FF_XSPH,
// Jacobi: reads the pre-XSPH velocities) + output of the public buffers.
// Textbook XSPH is Monaghan's form v_i += c (1/rho0) sum v_ij W_ij.
template <int VAR>
__global__ void k_final(DevParams P, uint32_t flags, const float4* __restrict__ Q, const float4* __restrict__ QX,
                        const float4* __restrict__ VS, const float4* __restrict__ OM,
                        const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
                        const uint32_t* __restrict__ ce, const float4* __restrict__ CS,
                        const uint32_t* __restrict__ ncnt, float4* __restrict__ Xo, float4* __restrict__ Po,
                        float4* __restrict__ Vo, float4* __restrict__ Co, float4* __restrict__ Fo) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  final_particle<VAR>(P, flags, s, Q, QX, VS, OM, keys, cs, ce, CS, ncnt, Xo, Po, Vo, Co, Fo);
  if (P.phs) P.ph[s] = P.phs[s];  // phases follow the particles into the sorted order
}

// Finite check of positions and velocities (failure detection).
__global__ void k_check_finite(uint32_t n, const float4* __restrict__ X, const float4* __restrict__ V,
                               uint32_t* __restrict__ bad) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4 x = X[i], v = V[i];
  const bool ok = isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(v.x) && isfinite(v.y) && isfinite(v.z);
  if (!ok) atomicAdd(bad, 1u);
}

// ---------------------------------------------------------------------------
// Host launchers
static inline uint32_t blocks_for(uint32_t n, uint32_t tpb) { return (n + tpb - 1) / tpb; }

// resetCellInfo (SortReorder.h:140-150) for the whole table in one launch:
// cstart = UINT_MAX, cend = n, and the occupied-block flags cleared, with 16-byte
// stores (the arrays come from hipMalloc, 256-byte aligned).
__global__ void k_cell_reset(uint32_t* __restrict__ cstart, uint32_t* __restrict__ cend, uint32_t ts, uint32_t n,
                             uint32_t* __restrict__ flags, uint32_t nflags, uint32_t* __restrict__ bcount,
                             uint32_t nb) {
  if (blockIdx.x == 0)
    for (uint32_t t = threadIdx.x; t < nb; t += blockDim.x) bcount[t] = 0u;
  const uint32_t q1 = ts / 4u, q2 = nflags / 4u, total = 2u * q1 + q2;
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint4 emp = make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu), cnt = make_uint4(n, n, n, n);
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    if (i < q1) reinterpret_cast<uint4*>(cstart)[i] = emp;
    else if (i < 2u * q1) reinterpret_cast<uint4*>(cend)[i - q1] = cnt;
    else reinterpret_cast<uint4*>(flags)[i - 2u * q1] = make_uint4(0u, 0u, 0u, 0u);
  }
  if (blockIdx.x == 0 && threadIdx.x < 4u) {  // tails beyond the last full 16 bytes
    const uint32_t t = threadIdx.x;
    if (4u * q1 + t < ts) {
      cstart[4u * q1 + t] = 0xFFFFFFFFu;
      cend[4u * q1 + t] = n;
    }
    if (flags && 4u * q2 + t < nflags) flags[4u * q2 + t] = 0u;
  }
}

hipError_t launch_cell_reset(hipStream_t st, uint32_t* cstart, uint32_t* cend, uint32_t ts, uint32_t n,
                             uint32_t* flags, uint32_t nflags, uint32_t* bcount) {
  if (!flags) nflags = 0;
  const uint32_t nb = (nflags + kTileCompactChunk - 1u) / kTileCompactChunk;
  const uint32_t total = 2u * (ts / 4u) + nflags / 4u + 1u;
  uint32_t b = blocks_for(total, 256);
  if (b > 4096) b = 4096;
  hipLaunchKernelGGL(k_cell_reset, dim3(b), dim3(256), 0, st, cstart, cend, ts, n, flags, nflags, bcount, nb);
  return hipGetLastError();
}

hipError_t launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t v, uint32_t n) {
  if (n == 0) return hipSuccess;
  uint32_t b = blocks_for(n, 256);
  if (b > 4096) b = 4096;
  hipLaunchKernelGGL(k_fill_u32, dim3(b), dim3(256), 0, st, p, v, n);
  return hipGetLastError();
}

hipError_t launch_copy_set(hipStream_t st, const CopySet& c) {
  size_t most = 0;
  for (uint32_t k = 0; k < c.count; ++k) {
    if (c.bytes[k] % 4u) return hipErrorInvalidValue;
    most = std::max(most, c.bytes[k]);
  }
  if (most == 0) return hipSuccess;
  const uint32_t b = (uint32_t)std::min<size_t>((most / 16u + 255u) / 256u + 1u, 4096u);
  hipLaunchKernelGGL(k_copy_set, dim3(b), dim3(256), 0, st, c);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// collisionType 1: contact batches (Collision.h:291-464, Fluid.cu:62-71).  The
// contacts of particle s are its neighbour-table row, the stencil walk of
// visit_neighbours (contacts, then shells, capped); contact c = s * cap + k.
// A batch gives every particle to the smallest unsolved contact index at it
// (the reference's in-block claim order, applied across blocks: its cross-block
// claims race).  Contacts holding both particles form a matching: each is
// marked solved and pushes its pair apart in place.
//
// Pass A: every unsolved contact offers its index to both particles; the row's
// first unsolved contact is remembered as the particle's own candidate.
__global__ void k_batch_claim(DevParams P, const float4* __restrict__ Q, const uint32_t* __restrict__ keys,
                              const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                              const uint32_t* __restrict__ solved, uint32_t words,
                              unsigned long long* __restrict__ minc, uint32_t* __restrict__ partner) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  const float4 qi = Q[s];
  const CellFrame f = make_frame(P, keys[s]);
  const uint32_t* sv = solved + (size_t)s * words;
  uint32_t k = 0, nc = 0;
  bool first = true;
  visit_neighbours(P, s, f, qi.x, qi.y, qi.z, (P.gates & G_FIND_CONTACTS) != 0, (P.gates & G_FIND_NEIGHBOURS) != 0,
                   cs, ce, nc, [&](uint32_t j, float, float, float, bool) {
                     const uint32_t kk = k++;
                     if ((sv[kk >> 5] >> (kk & 31u)) & 1u) return;
                     const unsigned long long c = (unsigned long long)s * P.cap + kk;
                     if (first) {
                       first = false;
                       partner[s] = j;
                       atomicMin(&minc[s], c);
                     }
                     atomicMin(&minc[j], c);
                   });
}

// Pass B: a particle whose smallest offer is its own candidate, and that is
// also the smallest offer at the partner, solves that contact.
__global__ void k_batch_solve(DevParams P, float4* __restrict__ Q, float4* __restrict__ QX,
                              const uint32_t* __restrict__ keys, uint32_t* __restrict__ solved, uint32_t words,
                              const unsigned long long* __restrict__ minc, const uint32_t* __restrict__ partner) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= P.n) return;
  const unsigned long long c = minc[s];
  if (c == ~0ull || c / P.cap != s) return;
  const uint32_t j = partner[s];
  if (minc[j] != c) return;
  const uint32_t k = (uint32_t)(c % P.cap);
  solved[(size_t)s * words + (k >> 5)] |= 1u << (k & 31u);  // row s is only written by its own thread
  const uint32_t ks = keys[s], kj = keys[j];
  const float4 qs = Q[s], qj = Q[j];
  // p_j - p_s with each position in its own cell frame (a contact joins two
  // particles of one scene, so one frame origin serves both)
  const uint32_t sc = scene_of_key(P, ks);
  const float ox = frame_origin(P, sc, 0), oy = frame_origin(P, sc, 1), oz = frame_origin(P, sc, 2);
  const float dx = (qj.x - qs.x) + (frame_corner(P, ox, compact10(kj >> 2)) - frame_corner(P, ox, compact10(ks >> 2)));
  const float dy = (qj.y - qs.y) + (frame_corner(P, oy, compact10(kj >> 1)) - frame_corner(P, oy, compact10(ks >> 1)));
  const float dz = (qj.z - qs.z) + (frame_corner(P, oz, compact10(kj)) - frame_corner(P, oz, compact10(ks)));
  const float len = sqrtf(dx * dx + dy * dy + dz * dz);
  const float half = (P.diameter - len) * 0.5f;
  if (half > 0.0f && len > 0.00001f) {
    // both move half the overlap times (1 - stiffness); coll_scale = -(1 - stiffness) / 2
    const float m = -2.0f * P.coll_scale * half / len;
    // p* is written back with w = 0
    Q[s] = make_float4(canonical_nan(qs.x - m * dx), canonical_nan(qs.y - m * dy), canonical_nan(qs.z - m * dz), 0.0f);
    Q[j] = make_float4(canonical_nan(qj.x + m * dx), canonical_nan(qj.y + m * dy), canonical_nan(qj.z + m * dz), 0.0f);
    const float4 xs = QX[s], xj = QX[j];
    QX[s] = make_float4(xs.x - m * dx, xs.y - m * dy, xs.z - m * dz, xs.w);
    QX[j] = make_float4(xj.x + m * dx, xj.y + m * dy, xj.z + m * dz, xj.w);
  }
}

hipError_t launch_collide_batches(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B,
                                  float4* Q, float4* QX, const uint32_t* keys, uint32_t batches, uint32_t* solved,
                                  uint32_t words, unsigned long long* minc, uint32_t* partner) {
  const dim3 g(blocks_for(P.n, tpb)), b(tpb);
  hipError_t e = launch_fill_u32(st, solved, 0u, P.n * words);
  for (uint32_t i = 0; i < batches && e == hipSuccess; ++i) {
    e = launch_fill_u32(st, reinterpret_cast<uint32_t*>(minc), 0xFFFFFFFFu, 2u * P.n);
    if (e != hipSuccess) break;
    hipLaunchKernelGGL(k_batch_claim, g, b, 0, st, P, Q, keys, B.cstart, B.cend, solved, words, minc, partner);
    hipLaunchKernelGGL(k_batch_solve, g, b, 0, st, P, Q, QX, keys, solved, words, minc, partner);
    e = hipGetLastError();
  }
  return e;
}

hipError_t launch_predict_keys(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, uint32_t* hist,
                               uint32_t passes, uint32_t copies) {
  if (P.n == 0) return hipSuccess;
  if (passes == 0u || passes > 4u || copies == 0u || copies > kSortHistCopies) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_predict_keys, dim3(blocks_for(P.n, tpb)), dim3(tpb), 0, st, P, B.X, B.V, B.F, B.P, B.keys_in,
                     hist, passes, copies);
  return hipGetLastError();
}

hipError_t launch_reorder(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B,
                          const uint32_t* keys_s, const uint32_t* ids_s, uint32_t tile_bits, uint32_t* tile_start,
                          uint32_t* tile_end) {
  hipLaunchKernelGGL(k_reorder, dim3(blocks_for(P.n, tpb)), dim3(tpb), 0, st, P, keys_s, ids_s, B.X, B.V, B.F, B.P,
                     B.C, B.Q[0], B.QX[0], B.VS, B.CS, B.cstart, B.cend, tile_bits, tile_start, tile_end);
  return hipGetLastError();
}

hipError_t launch_lambda(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, const float4* Q,
                         const uint32_t* keys_s, bool first) {
  if (wave_passes(P)) return launch_wave_lambda(st, P, B, Q, keys_s, first);
  dim3 g(blocks_for(P.n, tpb)), b(tpb);
  if (P.variant == PBD_KERNEL_TEXTBOOK) {
    if (first)
      hipLaunchKernelGGL((k_lambda<PBD_KERNEL_TEXTBOOK, true>), g, b, 0, st, P, Q, keys_s, B.cstart, B.cend, B.LAM,
                         B.DENS, B.NCNT, B.CCNT);
    else
      hipLaunchKernelGGL((k_lambda<PBD_KERNEL_TEXTBOOK, false>), g, b, 0, st, P, Q, keys_s, B.cstart, B.cend, B.LAM,
                         B.DENS, B.NCNT, B.CCNT);
  } else {
    if (first)
      hipLaunchKernelGGL((k_lambda<PBD_KERNEL_REFERENCE, true>), g, b, 0, st, P, Q, keys_s, B.cstart, B.cend, B.LAM,
                         B.DENS, B.NCNT, B.CCNT);
    else
      hipLaunchKernelGGL((k_lambda<PBD_KERNEL_REFERENCE, false>), g, b, 0, st, P, Q, keys_s, B.cstart, B.cend, B.LAM,
                         B.DENS, B.NCNT, B.CCNT);
  }
  return hipGetLastError();
}

hipError_t launch_count(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B,
                        const uint32_t* keys_s) {
  hipLaunchKernelGGL(k_count, dim3(blocks_for(P.n, tpb)), dim3(tpb), 0, st, P, keys_s, B.cstart, B.cend, B.NCNT,
                     B.CCNT);
  return hipGetLastError();
}

template <int VAR>
static void delta_dispatch(hipStream_t st, dim3 g, dim3 b, const DevParams& P, uint32_t flags, bool delta,
                           bool collide, const float4* Q, const float4* QX, const float* lam, const uint32_t* keys,
                           const uint32_t* cs, const uint32_t* ce, float4* Qo, float4* QXo, float4* DP, float4* VS) {
  if (delta && collide)
    hipLaunchKernelGGL((k_delta<VAR, true, true>), g, b, 0, st, P, flags, Q, QX, lam, keys, cs, ce, Qo, QXo, DP, VS);
  else if (delta)
    hipLaunchKernelGGL((k_delta<VAR, true, false>), g, b, 0, st, P, flags, Q, QX, lam, keys, cs, ce, Qo, QXo, DP, VS);
  else if (collide)
    hipLaunchKernelGGL((k_delta<VAR, false, true>), g, b, 0, st, P, flags, Q, QX, lam, keys, cs, ce, Qo, QXo, DP, VS);
  else
    hipLaunchKernelGGL((k_delta<VAR, false, false>), g, b, 0, st, P, flags, Q, QX, lam, keys, cs, ce, Qo, QXo, DP,
                       VS);
}

hipError_t launch_delta(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, uint32_t flags,
                        bool delta, bool collide, const float4* Q, const float4* QX, float4* Qo, float4* QXo,
                        const uint32_t* keys_s) {
  if ((delta || collide) && wave_passes(P))
    return launch_wave_delta(st, P, B, flags, delta, collide, Q, QX, Qo, QXo, keys_s);
  dim3 g(blocks_for(P.n, tpb)), b(tpb);
  if (P.variant == PBD_KERNEL_TEXTBOOK)
    delta_dispatch<PBD_KERNEL_TEXTBOOK>(st, g, b, P, flags, delta, collide, Q, QX, B.LAM, keys_s, B.cstart, B.cend, Qo,
                                        QXo, B.DP, B.VS);
  else
    delta_dispatch<PBD_KERNEL_REFERENCE>(st, g, b, P, flags, delta, collide, Q, QX, B.LAM, keys_s, B.cstart, B.cend,
                                         Qo, QXo, B.DP, B.VS);
  return hipGetLastError();
}

hipError_t launch_update(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, const float4* Q,
                         float4* QX) {
  hipLaunchKernelGGL(k_update, dim3(blocks_for(P.n, tpb)), dim3(tpb), 0, st, P, Q, QX, B.VS);
  return hipGetLastError();
}

hipError_t launch_omega(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, const float4* Q,
                        const uint32_t* keys_s) {
  if (wave_passes(P)) return launch_wave_omega(st, P, B, Q, keys_s);
  dim3 g(blocks_for(P.n, tpb)), b(tpb);
  if (P.variant == PBD_KERNEL_TEXTBOOK)
    hipLaunchKernelGGL(k_omega<PBD_KERNEL_TEXTBOOK>, g, b, 0, st, P, Q, B.VS, keys_s, B.cstart, B.cend, B.OM);
  else
    hipLaunchKernelGGL(k_omega<PBD_KERNEL_REFERENCE>, g, b, 0, st, P, Q, B.VS, keys_s, B.cstart, B.cend, B.OM);
  return hipGetLastError();
}

hipError_t launch_final(hipStream_t st, uint32_t tpb, const DevParams& P, const StepBuffers& B, uint32_t flags,
                        const float4* Q, const float4* QX, const uint32_t* keys_s) {
  if (wave_passes(P)) return launch_wave_final(st, P, B, flags, Q, QX, keys_s);
  dim3 g(blocks_for(P.n, tpb)), b(tpb);
  if (P.variant == PBD_KERNEL_TEXTBOOK)
    hipLaunchKernelGGL(k_final<PBD_KERNEL_TEXTBOOK>, g, b, 0, st, P, flags, Q, QX, B.VS, B.OM, keys_s, B.cstart,
                       B.cend, B.CS, B.NCNT, B.X, B.P, B.V, B.C, B.F);
  else
    hipLaunchKernelGGL(k_final<PBD_KERNEL_REFERENCE>, g, b, 0, st, P, flags, Q, QX, B.VS, B.OM, keys_s, B.cstart,
                       B.cend, B.CS, B.NCNT, B.X, B.P, B.V, B.C, B.F);
  return hipGetLastError();
}

hipError_t launch_check_finite(hipStream_t st, uint32_t n, const float4* X, const float4* V, uint32_t* bad) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_check_finite, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, X, V, bad);
  return hipGetLastError();
}

}  // namespace pbd
