// device.hpp - device (and host-twin) helpers of the PBF step kernels.
//
// Everything that decides an integer result (cell ids, sorted order, cell
// ranges, neighbour counts) is computed here with explicitly rounded FP32
// operations (no contraction) so that the GPU path and the CPU oracle agree
// bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "params.hpp"

namespace pbd {

// ---------------------------------------------------------------------------
// Morton codes (kernel/Hash.h:10-29): bit b of x goes to bit 3b+2, of y to
// 3b+1, of z to 3b.  Spread/compact by the shift-and-mask ladder.
constexpr uint32_t kMortonX = 0x24924924u;
constexpr uint32_t kMortonY = 0x12492492u;
constexpr uint32_t kMortonZ = 0x09249249u;

__host__ __device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

__host__ __device__ __forceinline__ uint32_t compact10(uint32_t v) {
  v &= 0x09249249u;
  v = (v | (v >> 2)) & 0x030C30C3u;
  v = (v | (v >> 4)) & 0x0300F00Fu;
  v = (v | (v >> 8)) & 0x030000FFu;
  v = (v | (v >> 16)) & 0x000003FFu;
  return v;
}

__host__ __device__ __forceinline__ uint32_t morton3(uint32_t x, uint32_t y, uint32_t z) {
  return (spread10(x) << 2) | (spread10(y) << 1) | spread10(z);
}

// Dilated add of a signed cell offset to one Morton component (mask m, shift sh).
__host__ __device__ __forceinline__ uint32_t dilated_add(uint32_t comp, int d, uint32_t m, uint32_t sh) {
  if (d >= 0) return ((comp | ~m) + (spread10((uint32_t)d) << sh)) & m;
  return (comp - (spread10((uint32_t)(-d)) << sh)) & m;
}

// ---------------------------------------------------------------------------
// Cell coordinate of one axis: i = (uint)clamp(floor((p - origin) * inv_cell), 0, dim - 1),
// two rounded FP32 ops then exact floor / clamp (Hash.h:21-26 generalised).
__host__ __device__ __forceinline__ uint32_t cell_coord(float p, float origin, float inv_cell, uint32_t dim) {
#pragma clang fp contract(off)
  float t = (p - origin) * inv_cell;
  float f = floorf(t);
  f = fmaxf(f, 0.0f);
  f = fminf(f, (float)(dim - 1u));
  return (uint32_t)f;
}

// The frame a scene's particles are stored in: the context's grid origin, or in
// a batched context the scene's own origin; cell coordinates enter it through
// local_mask (the coordinate inside the scene's slot).
__host__ __device__ __forceinline__ float frame_origin(const DevParams& P, uint32_t scene, int a) {
  return P.scenes ? P.scenes[scene].origin[a] : P.origin[a];
}
__host__ __device__ __forceinline__ uint32_t scene_of_key(const DevParams& P, uint32_t key) {
  return P.scenes ? key >> (3u * P.slot_log2) : 0u;
}
// Scene of particle index i before the step's keys exist (scenes are contiguous
// and in scene order in every sorted order): the last s with scene_first[s] <= i.
__host__ __device__ __forceinline__ uint32_t scene_of_index(const DevParams& P, uint32_t i) {
  if (!P.scenes) return 0u;
  uint32_t lo = 0, hi = P.n_scenes;
  while (hi - lo > 1u) {
    const uint32_t mid = (lo + hi) >> 1;
    if (P.scene_first[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Cell key of a position in the frame of `scene`: the context's grid, or the
// scene's slot of 2^slot_log2 cells per axis (key = morton(slot base + local)).
__host__ __device__ __forceinline__ uint32_t cell_key(const DevParams& P, uint32_t scene, float x, float y, float z,
                                                      uint32_t& ix, uint32_t& iy, uint32_t& iz) {
  if (!P.scenes) {
    ix = cell_coord(x, P.origin[0], P.inv_cell, P.dims[0]);
    iy = cell_coord(y, P.origin[1], P.inv_cell, P.dims[1]);
    iz = cell_coord(z, P.origin[2], P.inv_cell, P.dims[2]);
  } else {
    const SceneParams& S = P.scenes[scene];
    const uint32_t side = 1u << P.slot_log2;
    ix = (compact10(scene >> 2) << P.slot_log2) | cell_coord(x, S.origin[0], P.inv_cell, side);
    iy = (compact10(scene >> 1) << P.slot_log2) | cell_coord(y, S.origin[1], P.inv_cell, side);
    iz = (compact10(scene) << P.slot_log2) | cell_coord(z, S.origin[2], P.inv_cell, side);
  }
  return morton3(ix, iy, iz);
}

// Lower corner of a cell (local-coordinate anchor): origin + i * cell, two rounded ops.
__host__ __device__ __forceinline__ float cell_corner(float origin, float cell, uint32_t i) {
#pragma clang fp contract(off)
  return origin + (float)i * cell;
}
// The same for a cell coordinate of the grid, in the frame of its scene.
__host__ __device__ __forceinline__ float frame_corner(const DevParams& P, float origin, uint32_t i) {
  return cell_corner(origin, P.cell, i & P.local_mask);
}

// ---------------------------------------------------------------------------
// The enclosure of a particle: the context's, or in a batched context that of
// its scene.
struct Enclosure {
  float bmin[3], bmax[3], vdamp, pdamp;
};

__host__ __device__ __forceinline__ Enclosure enclosure_of(const DevParams& P, uint32_t scene) {
  Enclosure e;
  if (!P.scenes) {
    for (int a = 0; a < 3; ++a) {
      e.bmin[a] = P.bmin[a];
      e.bmax[a] = P.bmax[a];
    }
    e.vdamp = P.vdamp;
    e.pdamp = P.pdamp;
    return e;
  }
  const SceneParams& S = P.scenes[scene];
  for (int a = 0; a < 3; ++a) {
    e.bmin[a] = S.bmin[a];
    e.bmax[a] = S.bmax[a];
  }
  e.vdamp = S.vdamp;
  e.pdamp = S.pdamp;
  return e;
}

// Relaxation (Density.relaxation) and the projection box of the particle in cell `key`.
__host__ __device__ __forceinline__ float scene_eps(const DevParams& P, uint32_t key) {
  return P.scenes ? P.scenes[key >> (3u * P.slot_log2)].eps : P.eps;
}
struct ProjBox {
  float lo[3], hi[3];
};
__host__ __device__ __forceinline__ ProjBox scene_box(const DevParams& P, uint32_t key) {
  ProjBox b;
  const float* lo = P.scenes ? P.scenes[key >> (3u * P.slot_log2)].lo : P.lo;
  const float* hi = P.scenes ? P.scenes[key >> (3u * P.slot_log2)].hi : P.hi;
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = lo[a];
    b.hi[a] = hi[a];
  }
  return b;
}

// ---------------------------------------------------------------------------
// applyForces + confineToBox (Forces.h:19-101) with the reference's FP32
// operation order and no contraction:
//   v.y += (1*g)*dt;  v += f*dt;  p = x + v*dt;  clamp p per axis to the
//   enclosure inset by 0.001 (scaling that velocity component by the velocity
//   damping); if anything clamped x += pdamp*(p - x);  p.w = 1.
__host__ __device__ __forceinline__ void predict(const DevParams& P, uint32_t scene, float4& x, float4& v,
                                                 const float4 f, float4& p) {
#pragma clang fp contract(off)
  const Enclosure E = enclosure_of(P, scene);
  const float dt = P.dt;
  const float gdt = (1.0f * P.gravity) * dt;
  v.y = v.y + gdt;
  v.x = v.x + f.x * dt;
  v.y = v.y + f.y * dt;
  v.z = v.z + f.z * dt;
  v.w = v.w + f.w * dt;
  p.x = x.x + v.x * dt;
  p.y = x.y + v.y * dt;
  p.z = x.z + v.z * dt;
  p.w = x.w + v.w * dt;
  bool upd = false;
  if (p.x < E.bmin[0]) {
    v.x = E.vdamp * v.x;
    p.x = E.bmin[0] + 0.001f;
    upd = true;
  } else if (p.x > E.bmax[0]) {
    v.x = E.vdamp * v.x;
    p.x = E.bmax[0] - 0.001f;
    upd = true;
  }
  if (p.y < E.bmin[1]) {
    v.y = E.vdamp * v.y;
    p.y = E.bmin[1] + 0.001f;
    upd = true;
  } else if (p.y > E.bmax[1]) {
    v.y = E.vdamp * v.y;
    p.y = E.bmax[1] - 0.001f;
    upd = true;
  }
  if (p.z < E.bmin[2]) {
    v.z = E.vdamp * v.z;
    p.z = E.bmin[2] + 0.001f;
    upd = true;
  } else if (p.z > E.bmax[2]) {
    v.z = E.vdamp * v.z;
    p.z = E.bmax[2] - 0.001f;
    upd = true;
  }
  if (upd) {
    x.x = x.x + E.pdamp * (p.x - x.x);
    x.y = x.y + E.pdamp * (p.y - x.y);
    x.z = x.z + E.pdamp * (p.z - x.z);
    x.w = x.w + E.pdamp * (p.w - x.w);
  }
  p.w = 1.0f;
}

#ifdef __HIP_DEVICE_COMPILE__
#define PBD_DEVICE_ONLY 1
#endif

// ---------------------------------------------------------------------------
// Neighbour stencil walk (findContacts Collision.h:11-76, then findNeighbours
// Collision.h:87-160): the 27 cells around the particle's cell in (x, y, z)
// nested order -1..1, then the shells 2..kernelWidthNeighbours, every
// particle j != s of each occupied cell in sorted order, stopping at the cap.
// body(j, bx, by, bz, contact) receives the base vector b = q_s + (corner_s -
// corner_j) so that p_s - p_j = b - q_j in cell-local coordinates.
struct CellFrame {
  uint32_t ix, iy, iz;
  uint32_t kx, ky, kz;   // Morton components of the own cell
  float ox, oy, oz;      // origin of the scene's frame
  float cx, cy, cz;      // own corner
};

__device__ __forceinline__ CellFrame make_frame(const DevParams& P, uint32_t key) {
  CellFrame f;
  f.ix = compact10(key >> 2);
  f.iy = compact10(key >> 1);
  f.iz = compact10(key);
  f.kx = key & kMortonX;
  f.ky = key & kMortonY;
  f.kz = key & kMortonZ;
  const uint32_t sc = scene_of_key(P, key);
  f.ox = frame_origin(P, sc, 0);
  f.oy = frame_origin(P, sc, 1);
  f.oz = frame_origin(P, sc, 2);
  f.cx = frame_corner(P, f.ox, f.ix);
  f.cy = frame_corner(P, f.oy, f.iy);
  f.cz = frame_corner(P, f.oz, f.iz);
  return f;
}

template <class Body>
__device__ __forceinline__ void visit_cell(const DevParams& P, uint32_t s, uint32_t k, float bx, float by, float bz,
                                           bool contact, const uint32_t* __restrict__ cs,
                                           const uint32_t* __restrict__ ce, uint32_t& cnt, Body& body) {
  const uint32_t st = cs[k];
  if (st == 0xFFFFFFFFu) return;
  const uint32_t en = ce[k];
  for (uint32_t j = st; j < en; ++j) {
    if (j == s) continue;
    body(j, bx, by, bz, contact);
    if (++cnt == P.cap) return;
  }
}

// Returns the neighbour count; n_contacts receives the contact count.
template <class Body>
__device__ __forceinline__ uint32_t visit_neighbours(const DevParams& P, uint32_t s, const CellFrame& f, float qx,
                                                     float qy, float qz, bool contacts, bool shells,
                                                     const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                                                     uint32_t& n_contacts, Body body) {
  uint32_t cnt = 0;
  const uint32_t cap = P.cap;
  if (contacts) {
    for (int dx = -1; dx <= 1; ++dx) {
      const uint32_t nx = f.ix + (uint32_t)dx;
      if (nx >= P.dims[0]) continue;
      const uint32_t kx = dilated_add(f.kx, dx, kMortonX, 2);
      const float bx = qx + (f.cx - frame_corner(P, f.ox, nx));
      for (int dy = -1; dy <= 1; ++dy) {
        const uint32_t ny = f.iy + (uint32_t)dy;
        if (ny >= P.dims[1]) continue;
        const uint32_t ky = dilated_add(f.ky, dy, kMortonY, 1);
        const float by = qy + (f.cy - frame_corner(P, f.oy, ny));
        for (int dz = -1; dz <= 1; ++dz) {
          const uint32_t nz = f.iz + (uint32_t)dz;
          if (nz >= P.dims[2]) continue;
          const uint32_t kz = dilated_add(f.kz, dz, kMortonZ, 0);
          const float bz = qz + (f.cz - frame_corner(P, f.oz, nz));
          visit_cell(P, s, kx | ky | kz, bx, by, bz, true, cs, ce, cnt, body);
          if (cnt == cap) goto contacts_done;
        }
      }
    }
  }
contacts_done:
  n_contacts = cnt;
  if (shells && cnt < cap) {
    const int kw = P.kw;
    for (int sh = 2; sh <= kw; ++sh) {
      for (int dx = -sh; dx <= sh; ++dx) {
        const uint32_t nx = f.ix + (uint32_t)dx;
        if (nx >= P.dims[0]) continue;
        const uint32_t kx = dilated_add(f.kx, dx, kMortonX, 2);
        const float bx = qx + (f.cx - frame_corner(P, f.ox, nx));
        const bool ex = (dx == -sh || dx == sh);
        for (int dy = -sh; dy <= sh; ++dy) {
          const uint32_t ny = f.iy + (uint32_t)dy;
          if (ny >= P.dims[1]) continue;
          const uint32_t ky = dilated_add(f.ky, dy, kMortonY, 1);
          const float by = qy + (f.cy - frame_corner(P, f.oy, ny));
          const bool ey = ex || (dy == -sh || dy == sh);
          for (int dz = -sh; dz <= sh; ++dz) {
            if (!ey && dz != -sh && dz != sh) continue;
            const uint32_t nz = f.iz + (uint32_t)dz;
            if (nz >= P.dims[2]) continue;
            const uint32_t kz = dilated_add(f.kz, dz, kMortonZ, 0);
            const float bz = qz + (f.cz - frame_corner(P, f.oz, nz));
            visit_cell(P, s, kx | ky | kz, bx, by, bz, false, cs, ce, cnt, body);
            if (cnt == cap) return cnt;
          }
        }
      }
    }
  }
  return cnt;
}

// A NaN as the positive quiet NaN, for every position that a tile list may be built from
// (the lists read the sign of a distance test, and an operation's own NaN is negative).
__device__ __forceinline__ float canonical_nan(float x) { return x == x ? x : __uint_as_float(0x7FC00000u); }

// ---------------------------------------------------------------------------
// Kernel functions, unnormalised (coefficients wc / gc applied by the caller).
//   reference (Density.h:14-42): W ~ ((h^2 - r^2)^3)^2 on 0.001 < r < h - 0.001;
//                                grad ~ (h - r)^2 / r * r_vec on r > 1e-4, h - r > 1e-4
//   textbook:                    W ~ (h^2 - r^2)^3 on r < h;  grad ~ (h - r)^2 / r * r_vec on 0 < r < h
// r and 1/r come from the hardware reciprocal square root (v_rsq_f32, 1 ulp):
// the IEEE sqrt and divide sequences cost ~16 instructions per candidate.
__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
// |r|^2 with the fused operations spelled out, so that a path forms it alike whatever
// the compiler makes of the expressions around it.  Two orders are in use (XF: x first;
// else y first): one rounding more or less decides which side of a contact's onset a
// pair falls on, so a path keeps the order it has.
template <bool XF = false>
__device__ __forceinline__ float length_sq(float x, float y, float z) {
  return XF ? fmaf(z, z, fmaf(y, y, x * x)) : fmaf(z, z, fmaf(x, x, y * y));
}
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// Textbook terms are branch-free: max() clamps at the supports, which gives
// the same zero outside them as the r < h tests, and r2 is floored at 1e-30 so
// that 1/r stays finite for coincident particles (whose r_vec is exactly zero,
// so every g * r_vec term vanishes; (h - r)^4 is masked explicitly).
__device__ __forceinline__ float tb_inv_r(float r2) { return rsq(fmaxf(r2, 1.0e-30f)); }

template <int V>
__device__ __forceinline__ float w_unnorm(const DevParams& P, float r2) {
  if (V == PBD_KERNEL_TEXTBOOK) {
    const float t = fmaxf(P.hp2 - r2, 0.0f);
    return t * t * t;
  } else {
    const float r = r2 > 0.0f ? r2 * rsq(r2) : 0.0f;
    if (r > 0.001f && r < (P.hp - 0.001f)) {
      const float t = P.hp2 - r2;
      const float t3 = t * t * t;
      return t3 * t3;
    }
    return 0.0f;
  }
}

// grad magnitude factor g such that grad_unnorm = g * r_vec; also returns (h - r)^4 in hr4.
template <int V>
__device__ __forceinline__ float grad_factor(const DevParams& P, float r2, float& hr4) {
  if (V == PBD_KERNEL_TEXTBOOK) {
    const float ir = tb_inv_r(r2);
    const float hr = fmaxf(P.hs - fmaxf(r2, 1.0e-30f) * ir, 0.0f);
    const float hr2 = hr * hr;
    hr4 = r2 > 0.0f ? hr2 * hr2 : 0.0f;
    return hr2 * ir;
  } else {
    if (r2 > 0.0f) {
      const float ir = rsq(r2);
      const float r = r2 * ir;
      if (r > 0.0001f && (P.hs - r) > 0.0001f) {
        const float hr = P.hs - r;
        const float hr2 = hr * hr;
        hr4 = hr2 * hr2;
        return hr2 * ir;
      }
    }
  }
  hr4 = 0.0f;
  return 0.0f;
}

// x^N for a compile-time N >= 1 (square-and-multiply, N known to the compiler).
template <int N>
__device__ __forceinline__ float ipow_c(float x) {
  if (N == 1) return x;
  const float h = ipow_c<(N >= 2 ? N / 2 : 1)>(x);
  return (N & 1) ? h * h * x : h * h;
}

__device__ __forceinline__ float ipow(float x, int n) {
  bool inv = n < 0;
  unsigned e = (unsigned)(inv ? -n : n);
  float r = 1.0f;
  while (e) {
    if (e & 1u) r *= x;
    x *= x;
    e >>= 1;
  }
  return inv ? 1.0f / r : r;
}

}  // namespace pbd
