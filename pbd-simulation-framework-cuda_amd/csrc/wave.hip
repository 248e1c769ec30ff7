// wave.hip - the neighbour passes with a wave per particle (gfx950), for scenes of the
// reference variant that are too small to fill the chip with a thread per particle.
//
// A thread that walks the 125 cells of a two-cell stencil looks up one cell after the
// other, then loads one neighbour after the other: the passes of a 13,824-particle
// scene lasted 116 to 142 us each, on 216 of 1,024 SIMDs, all of it latency.  Here
//   1. the lanes look up a cell each, in the stencil's order; a scan of the counts
//      gives every neighbour its place in the particle's list, which is the order
//      the walk visits (27 contact cells, then the shells, cut off at
//      maxNeighboursPerParticle); 256 places of it are in LDS at a time;
//   2. the lanes form the terms of 64 pairs at a time;
//   3. one lane per component of the sums adds the terms one by one, in list order
//      and with the walk's fused operations, so the sums are the walk's bit for bit.
// The 13,824-particle scene: lambda 116 -> 20 us, delta-p 123 -> 21, omega 116 -> 17,
// final 142 -> 23 us, bound by the latency of the dependent loads (keys, cells, positions)
// over three rounds of resident waves.  Compressed to 3.5 particles a cell (lists of 430):
// 321 us a step, 59,319 particles 974 us; with a thread per particle 1936 and 1952 us.  A wave issues about ten times the instructions of
// a particle's thread, so the passes go to kernels.hip above kWaveParticles.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "kernels.hpp"
#include "particle_ops.hpp"

namespace pbd {
namespace {

constexpr uint32_t kWaves = 4;          // of a workgroup, a particle each
constexpr int kWaveStencil = 2;         // stencils of up to 5 x 5 x 5 cells
constexpr uint32_t kWaveCells = 125;
constexpr uint32_t kWaveList = 256;     // neighbours a wave's list holds at a time
constexpr uint32_t kMaxTerms = 8;       // components of a pass's sums

// The stencil's cells in the walk's order: the 27 contact cells, then shell 2.
struct StencilTable {
  int8_t d[kWaveCells][4];
};
constexpr StencilTable make_stencil() {
  StencilTable t{};
  uint32_t n = 0;
  for (int x = -1; x <= 1; ++x)
    for (int y = -1; y <= 1; ++y)
      for (int z = -1; z <= 1; ++z, ++n) {
        t.d[n][0] = (int8_t)x;
        t.d[n][1] = (int8_t)y;
        t.d[n][2] = (int8_t)z;
      }
  for (int x = -2; x <= 2; ++x)
    for (int y = -2; y <= 2; ++y)
      for (int z = -2; z <= 2; ++z) {
        if (x > -2 && x < 2 && y > -2 && y < 2 && z > -2 && z < 2) continue;
        t.d[n][0] = (int8_t)x;
        t.d[n][1] = (int8_t)y;
        t.d[n][2] = (int8_t)z;
        ++n;
      }
  return t;
}
__constant__ const StencilTable kStencil = make_stencil();

struct WaveLds {
  float2 term[kMaxTerms][65];  // factors of a pair's addition to each component (65: rows on different banks)
  uint32_t j[kWaveList];
  uint8_t cell[kWaveList];
};

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The neighbour list of particle s as the lanes hold it: of cell (chunk k, lane) its
// particles st .. en - 1, from list place `at` on (s itself left out).
struct WaveCells {
  static constexpr uint32_t kChunks = (kWaveCells + 63u) / 64u;
  uint32_t st[kChunks], en[kChunks], at[kChunks], first;
};

// Looks the cells up; returns the list's length (at most P.cap), nc: how many are contacts.
__device__ __forceinline__ uint32_t wave_cells(const DevParams& P, uint32_t s, const CellFrame& f,
                                               const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                                               WaveCells& W, uint32_t& nc) {
  const uint32_t lane = threadIdx.x & 63u;
  W.first = (P.gates & G_FIND_CONTACTS) ? 0u : 27u;
  const uint32_t last = (P.gates & G_FIND_NEIGHBOURS) && P.kw > 1 ? kWaveCells : 27u;
  uint32_t base = 0u, contacts = 0u;
#pragma unroll
  for (uint32_t k = 0; k < WaveCells::kChunks; ++k) {
    const uint32_t c = W.first + 64u * k + lane;
    uint32_t st = 0u, en = 0u, cnt = 0u;
    if (c < last) {
      const int dx = kStencil.d[c][0], dy = kStencil.d[c][1], dz = kStencil.d[c][2];
      const uint32_t nx = f.ix + (uint32_t)dx, ny = f.iy + (uint32_t)dy, nz = f.iz + (uint32_t)dz;
      if (nx < P.dims[0] && ny < P.dims[1] && nz < P.dims[2]) {
        const uint32_t key = morton3(nx, ny, nz);
        const uint32_t s0 = cs[key], e0 = ce[key];
        if (s0 != 0xFFFFFFFFu) {
          st = s0;
          en = e0;
          cnt = en - st - (s >= st && s < en ? 1u : 0u);
        }
      }
    }
    uint32_t x = cnt;
#pragma unroll
    for (uint32_t o = 1; o < 64u; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    W.st[k] = st;
    W.en[k] = en;
    W.at[k] = base + x - cnt;
    if (k == 0u && W.first == 0u) contacts = __shfl(x, 26);
    base += __shfl(x, 63);
  }
  nc = min(contacts, P.cap);
  return min(base, P.cap);
}

// Entries w0 .. min(w0 + kWaveList, n) - 1 of the list to L.
__device__ __forceinline__ void wave_list(const WaveCells& W, uint32_t s, uint32_t w0, uint32_t n, WaveLds& L) {
  const uint32_t lane = threadIdx.x & 63u, end = min(n, w0 + kWaveList);
#pragma unroll
  for (uint32_t k = 0; k < WaveCells::kChunks; ++k) {
    uint32_t i = max(W.at[k], w0), j = W.st[k] + (i - W.at[k]);
    if (s >= W.st[k] && s < j) ++j;  // s is among the entries before
    for (; j < W.en[k] && i < end; ++j) {
      if (j == s) continue;
      L.j[i - w0] = j;
      L.cell[i - w0] = (uint8_t)(W.first + 64u * k + lane);
      ++i;
    }
  }
  wave_fence();
}

// Base vector of neighbour list entry i: p_s - p_j = b - q_j.
__device__ __forceinline__ float3 wave_base(const DevParams& P, const CellFrame& f, float4 q, uint32_t c) {
  const uint32_t nx = f.ix + (uint32_t)(int)kStencil.d[c][0], ny = f.iy + (uint32_t)(int)kStencil.d[c][1],
                 nz = f.iz + (uint32_t)(int)kStencil.d[c][2];
  return make_float3(q.x + (f.cx - frame_corner(P, f.ox, nx)), q.y + (f.cy - frame_corner(P, f.oy, ny)),
                     q.z + (f.cz - frame_corner(P, f.oz, nz)));
}

// The sums of N components over the first n entries of the list, kWaveList of them at a
// time: terms(i, j, r, put) forms pair i's terms, put(c, u, v) the addition of u v to
// component c (v = 1: of u, exactly); a component that it does not put gets nothing.
// Returns component (lane) of the sums.
template <uint32_t N, class Terms>
__device__ __forceinline__ float wave_sums(const DevParams& P, uint32_t s, const CellFrame& f, const WaveCells& W,
                                           const float4* __restrict__ Q, float4 q, uint32_t n, WaveLds& L,
                                           Terms terms) {
  static_assert(N <= kMaxTerms, "components");
  const uint32_t lane = threadIdx.x & 63u;
  float acc = 0.0f;
#pragma unroll 1
  for (uint32_t w0 = 0; w0 < n; w0 += kWaveList) {
    wave_list(W, s, w0, n, L);
    const uint32_t held = min(n - w0, kWaveList);
    for (uint32_t k = 0; k < held; k += 64u) {
      const uint32_t m = min(held - k, 64u);
      if (lane < m) {
        const uint32_t j = L.j[k + lane];
        const float4 qj = Q[j];
        const float3 b = wave_base(P, f, q, L.cell[k + lane]);
        terms(w0 + k + lane, j, b.x - qj.x, b.y - qj.y, b.z - qj.z,
              [&](uint32_t c, float u, float v) { L.term[c][lane] = make_float2(u, v); });
      }
      wave_fence();
      if (lane < N) {
        const float2* t = L.term[lane];
        uint32_t i = 0;
        for (; i + 8u <= m; i += 8u) {
          float2 w[8];
#pragma unroll
          for (uint32_t u = 0; u < 8u; ++u) w[u] = t[i + u];
#pragma unroll
          for (uint32_t u = 0; u < 8u; ++u) acc = fmaf(w[u].x, w[u].y, acc);
        }
        for (; i < m; ++i) acc = fmaf(t[i].x, t[i].y, acc);
      }
      wave_fence();
    }
  }
  return acc;
}

constexpr int REF = PBD_KERNEL_REFERENCE;

template <bool FIRST>
__global__ __launch_bounds__(64 * kWaves) void k_wave_lambda(DevParams P, const float4* __restrict__ Q,
                                                             const uint32_t* __restrict__ keys,
                                                             const uint32_t* __restrict__ cs,
                                                             const uint32_t* __restrict__ ce, float* __restrict__ lam,
                                                             float* __restrict__ dens, uint32_t* __restrict__ ncnt,
                                                             uint32_t* __restrict__ ccnt) {
  __shared__ WaveLds lds[kWaves];
  const uint32_t s = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (s >= P.n) return;
  WaveLds& L = lds[threadIdx.x >> 6];
  const CellFrame f = make_frame(P, keys[s]);
  const float4 q = Q[s];
  WaveCells W;
  uint32_t nc;
  const uint32_t n = wave_cells(P, s, f, cs, ce, W, nc);
  const float a = wave_sums<5>(P, s, f, W, Q, q, n, L, [&](uint32_t, uint32_t, float rx, float ry, float rz, auto put) {
    const float r2 = length_sq(rx, ry, rz);
    float hr4;
    const float g = grad_factor<REF>(P, r2, hr4);
    put(0u, w_unnorm<REF>(P, r2), 1.0f);
    put(1u, g, rx);
    put(2u, g, ry);
    put(3u, g, rz);
    put(4u, hr4, 1.0f);
  });
  LambdaAcc A;
  A.A = __shfl(a, 0);
  A.gx = __shfl(a, 1);
  A.gy = __shfl(a, 2);
  A.gz = __shfl(a, 3);
  A.B = __shfl(a, 4);
  if (lane != 0u) return;
  float rho;
  lam[s] = lambda_finish<REF>(P, A, rho, scene_eps(P, keys[s]));
  if (FIRST) {
    dens[s] = rho;
    ncnt[s] = n;
    ccnt[s] = nc;
  }
}

template <bool DELTA, bool COLLIDE>
__global__ __launch_bounds__(64 * kWaves) void k_wave_delta(
    DevParams P, uint32_t flags, const float4* __restrict__ Q, const float4* __restrict__ QX,
    const float* __restrict__ lam, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cs,
    const uint32_t* __restrict__ ce, float4* __restrict__ Qo, float4* __restrict__ QXo, float4* __restrict__ DP,
    float4* __restrict__ VS) {
  __shared__ WaveLds lds[kWaves];
  const uint32_t s = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (s >= P.n) return;
  WaveLds& L = lds[threadIdx.x >> 6];
  const CellFrame f = make_frame(P, keys[s]);
  const float4 q = Q[s];
  WaveCells W;
  uint32_t nc;
  const uint32_t all = wave_cells(P, s, f, cs, ce, W, nc);
  // without DELTA only the contacts count
  const uint32_t n = DELTA ? all : nc;
  const float li = DELTA ? lam[s] : 0.0f;
  constexpr uint32_t N = (DELTA ? 3u : 0u) + (COLLIDE ? 3u : 0u), C = DELTA ? 3u : 0u;
  const float a = wave_sums<N>(P, s, f, W, Q, q, n, L, [&](uint32_t i, uint32_t j, float rx, float ry, float rz, auto put) {
    const float r2 = length_sq(rx, ry, rz);
    if (DELTA) {
      const float w = P.wc * w_unnorm<REF>(P, r2);
      const float sc = -P.k_scorr * ipow(w * P.inv_w_dq, P.n_scorr);
      float hr4;
      const float g = grad_factor<REF>(P, r2, hr4);
      const float t = (li + lam[j] + sc) * g;
      put(0u, t, rx);
      put(1u, t, ry);
      put(2u, t, rz);
    }
    if (COLLIDE) {
      float t = 0.0f;
      if (i < nc && r2 > 0.0f) {
        const float il = rsq(r2);
        const float len = r2 * il;
        const float ov = P.diameter - len;
        if (ov > 0.0f && len > 0.00001f) t = -P.coll_scale * ov * il;
      }
      // a pair without a push adds nothing, also where its distance is not finite
      put(C, t, t == 0.0f ? 0.0f : rx);
      put(C + 1u, t, t == 0.0f ? 0.0f : ry);
      put(C + 2u, t, t == 0.0f ? 0.0f : rz);
    }
  });
  DeltaAcc A;
  if (DELTA) {
    A.ax = __shfl(a, 0);
    A.ay = __shfl(a, 1);
    A.az = __shfl(a, 2);
  }
  if (COLLIDE) {
    A.px = __shfl(a, (int)C);
    A.py = __shfl(a, (int)C + 1);
    A.pz = __shfl(a, (int)C + 2);
  }
  if (lane == 0u) delta_finish<REF, DELTA>(P, flags, s, q, QX[s], A, f.cx, f.cy, f.cz, keys[s], Qo, QXo, DP, VS);
}

__global__ __launch_bounds__(64 * kWaves) void k_wave_omega(DevParams P, const float4* __restrict__ Q,
                                                            const float4* __restrict__ VS,
                                                            const uint32_t* __restrict__ keys,
                                                            const uint32_t* __restrict__ cs,
                                                            const uint32_t* __restrict__ ce,
                                                            float4* __restrict__ OM) {
  __shared__ WaveLds lds[kWaves];
  const uint32_t s = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (s >= P.n) return;
  WaveLds& L = lds[threadIdx.x >> 6];
  const CellFrame f = make_frame(P, keys[s]);
  const float4 q = Q[s], vi = VS[s];
  WaveCells W;
  uint32_t nc;
  const uint32_t n = wave_cells(P, s, f, cs, ce, W, nc);
  const float a = wave_sums<3>(P, s, f, W, Q, q, n, L, [&](uint32_t, uint32_t j, float rx, float ry, float rz, auto put) {
    const float4 vj = VS[j];
    const float vx = vj.x - vi.x, vy = vj.y - vi.y, vz = vj.z - vi.z;
    float hr4;
    const float g = grad_factor<REF>(P, length_sq(rx, ry, rz), hr4);
    const float gx = g * rx, gy = g * ry, gz = g * rz;
    put(0u, fmaf(vy, gz, -(vz * gy)), 1.0f);
    put(1u, fmaf(vz, gx, -(vx * gz)), 1.0f);
    put(2u, fmaf(vx, gy, -(vy * gx)), 1.0f);
  });
  OmegaAcc A;
  A.ox = __shfl(a, 0);
  A.oy = __shfl(a, 1);
  A.oz = __shfl(a, 2);
  if (lane == 0u) OM[s] = omega_finish<REF, true>(P, A);
}

__global__ __launch_bounds__(64 * kWaves) void k_wave_final(
    DevParams P, uint32_t flags, const float4* __restrict__ Q, const float4* __restrict__ QX,
    const float4* __restrict__ VS, const float4* __restrict__ OM, const uint32_t* __restrict__ keys,
    const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce, const float4* __restrict__ CS,
    const uint32_t* __restrict__ ncnt, float4* __restrict__ Xo, float4* __restrict__ Po, float4* __restrict__ Vo,
    float4* __restrict__ Co, float4* __restrict__ Fo) {
  __shared__ WaveLds lds[kWaves];
  const uint32_t s = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (s >= P.n) return;
  WaveLds& L = lds[threadIdx.x >> 6];
  const bool vort = (flags & FF_VORT) != 0, xsph = (flags & FF_XSPH) != 0;
  const CellFrame f = make_frame(P, keys[s]);
  const float4 q = Q[s], vi = VS[s];
  const float4 oi = vort ? OM[s] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  WaveCells W;
  uint32_t nc, n = 0u;
  if (vort || xsph) n = wave_cells(P, s, f, cs, ce, W, nc);
  const float a = wave_sums<7>(P, s, f, W, Q, q, n, L, [&](uint32_t, uint32_t j, float rx, float ry, float rz, auto put) {
    float w = 0.0f;
    float4 dv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (xsph) {
      const float4 vj = VS[j];
      w = w_unnorm<REF>(P, length_sq(rx, ry, rz));
      dv = make_float4(vj.x - vi.x, vj.y - vi.y, vj.z - vi.z, vj.w - vi.w);
    }
    put(0u, dv.x, w);
    put(1u, dv.y, w);
    put(2u, dv.z, w);
    put(3u, dv.w, w);
    float ex = 0.0f, ey = 0.0f, ez = 0.0f;
    if (vort) {
      const float4 oj = OM[j];
      const float ol = sqrtf(length_sq(oj.x - oi.x, oj.y - oi.y, oj.z - oi.z));
      ex = ol / (-rx + 0.00000001f);
      ey = ol / (-ry + 0.00000001f);
      ez = ol / (-rz + 0.00000001f);
    }
    put(4u, ex, 1.0f);
    put(5u, ey, 1.0f);
    put(6u, ez, 1.0f);
  });
  FinalAcc A;
  A.sx = __shfl(a, 0);
  A.sy = __shfl(a, 1);
  A.sz = __shfl(a, 2);
  A.sw = __shfl(a, 3);
  A.ex = __shfl(a, 4);
  A.ey = __shfl(a, 5);
  A.ez = __shfl(a, 6);
  if (lane == 0u) final_finish<REF>(P, flags, s, q, vi, oi, A, f.cx, f.cy, f.cz, QX, CS, ncnt, Xo, Po, Vo, Co, Fo);
}

inline dim3 wave_grid(const DevParams& P) { return dim3((P.n + kWaves - 1u) / kWaves); }

}  // namespace

bool wave_passes(const DevParams& P) {
  return P.variant == PBD_KERNEL_REFERENCE && !P.phased && P.kw <= kWaveStencil && P.n <= kWaveParticles;
}

hipError_t launch_wave_lambda(hipStream_t st, const DevParams& P, const StepBuffers& B, const float4* Q,
                              const uint32_t* keys, bool first) {
  if (first)
    hipLaunchKernelGGL(k_wave_lambda<true>, wave_grid(P), dim3(64 * kWaves), 0, st, P, Q, keys, B.cstart, B.cend, B.LAM,
                       B.DENS, B.NCNT, B.CCNT);
  else
    hipLaunchKernelGGL(k_wave_lambda<false>, wave_grid(P), dim3(64 * kWaves), 0, st, P, Q, keys, B.cstart, B.cend, B.LAM,
                       B.DENS, B.NCNT, B.CCNT);
  return hipGetLastError();
}

hipError_t launch_wave_delta(hipStream_t st, const DevParams& P, const StepBuffers& B, uint32_t flags, bool delta,
                             bool collide, const float4* Q, const float4* QX, float4* Qo, float4* QXo,
                             const uint32_t* keys) {
#define PBD_WAVE_DELTA(D_, C_)                                                                                     \
  hipLaunchKernelGGL((k_wave_delta<D_, C_>), wave_grid(P), dim3(64 * kWaves), 0, st, P, flags, Q, QX, B.LAM, keys, \
                     B.cstart, B.cend, Qo, QXo, B.DP, B.VS)
  if (delta && collide) PBD_WAVE_DELTA(true, true);
  else if (delta) PBD_WAVE_DELTA(true, false);
  else if (collide) PBD_WAVE_DELTA(false, true);
  else return hipErrorInvalidValue;  // no pairs: a thread per particle
#undef PBD_WAVE_DELTA
  return hipGetLastError();
}

hipError_t launch_wave_omega(hipStream_t st, const DevParams& P, const StepBuffers& B, const float4* Q,
                             const uint32_t* keys) {
  hipLaunchKernelGGL(k_wave_omega, wave_grid(P), dim3(64 * kWaves), 0, st, P, Q, B.VS, keys, B.cstart, B.cend, B.OM);
  return hipGetLastError();
}

hipError_t launch_wave_final(hipStream_t st, const DevParams& P, const StepBuffers& B, uint32_t flags, const float4* Q,
                             const float4* QX, const uint32_t* keys) {
  hipLaunchKernelGGL(k_wave_final, wave_grid(P), dim3(64 * kWaves), 0, st, P, flags, Q, QX, B.VS, B.OM, keys, B.cstart,
                     B.cend, B.CS, B.NCNT, B.X, B.P, B.V, B.C, B.F);
  return hipGetLastError();
}

}  // namespace pbd
