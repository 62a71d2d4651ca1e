// lbm_wale.hpp — WALE eddy viscosity of one cell from the cached velocities
// and strain (les.rs:120-211), for the closure's own pass (lbm_les.hip) and for
// the closure inside the collide-stream kernel (lbm_hydro.hip): the same
// operations in the same order, so both give the same bits.
#pragma once
#include "lbm_device.hpp"

namespace lbm {

// nu_t from the velocity gradient's parts: own velocity, strain (xy, xz, yz),
// and per axis the neighbours' kinds kp / km (0 none: non-periodic domain face;
// 1 fluid; 2 solid) and velocities pv / mv (a solid's wall velocity).  CENTRAL:
// every neighbour is fluid.  Gradient: diagonal and antisymmetric part from
// finite differences (one-sided at the half-way wall and at domain faces),
// off-diagonal symmetric part from the stress (gather_velocity_gradient,
// solver.rs:5490-5581).
template <bool CENTRAL>
__device__ __forceinline__ float wale_nut(float cw_delta_sq, const float own[3], float sxy, float sxz, float syz,
                                          const int kp[3], const int km[3], const float pv[3][3],
                                          const float mv[3][3]) {
#pragma clang fp contract(off)
  float fd[3][3];
  if (CENTRAL ||
      (kp[0] == 1 && km[0] == 1 && kp[1] == 1 && km[1] == 1 && kp[2] == 1 && km[2] == 1)) {  // the common case
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
      for (int k = 0; k < 3; ++k) fd[k][ax] = (pv[ax][k] - mv[ax][k]) * 0.5f;
  } else {
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        float v = 0.0f;
        if (kp[ax] == 1 && km[ax] == 1)
          v = (pv[ax][k] - mv[ax][k]) * 0.5f;
        else if (kp[ax] == 1 && km[ax] == 2)
          v = -(4.0f / 3.0f) * mv[ax][k] + own[k] + (1.0f / 3.0f) * pv[ax][k];
        else if (kp[ax] == 2 && km[ax] == 1)
          v = (4.0f / 3.0f) * pv[ax][k] - own[k] - (1.0f / 3.0f) * mv[ax][k];
        else if (kp[ax] == 1 && km[ax] == 0)
          v = pv[ax][k] - own[k];
        else if (kp[ax] == 0 && km[ax] == 1)
          v = own[k] - mv[ax][k];
        fd[k][ax] = v;
      }
  }
  float g[3][3];
  g[0][0] = fd[0][0];
  g[1][1] = fd[1][1];
  g[2][2] = fd[2][2];
  g[0][1] = sxy + 0.5f * (fd[0][1] - fd[1][0]);
  g[1][0] = sxy + 0.5f * (fd[1][0] - fd[0][1]);
  g[0][2] = sxz + 0.5f * (fd[0][2] - fd[2][0]);
  g[2][0] = sxz + 0.5f * (fd[2][0] - fd[0][2]);
  g[1][2] = syz + 0.5f * (fd[1][2] - fd[2][1]);
  g[2][1] = syz + 0.5f * (fd[2][1] - fd[1][2]);
  // WALE invariants
  float s2 = 0.0f, g2[3][3];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const float sv = 0.5f * (g[p][q] + g[q][p]);
      s2 = s2 + sv * sv;
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < 3; ++k) acc = acc + g[p][k] * g[k][q];
      g2[p][q] = acc;
    }
  const float tr = g2[0][0] + g2[1][1] + g2[2][2];
  float sd2 = 0.0f;
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      float sd = 0.5f * (g2[p][q] + g2[q][p]);
      if (p == q) sd = sd - tr / 3.0f;
      sd2 = sd2 + sd * sd;
    }
  // the three powers from square roots (s2^2.5 = s2^2 sqrt(s2),
  // sd2^1.5 = sd2 sqrt(sd2), sd2^1.25 = sd2 sqrt(sqrt(sd2))): a few ulp from
  // the correctly rounded powers, at a fraction of a general powf's cost
  const float rs = sqrtf(s2), rd = sqrtf(sd2);
  const float denom = s2 * s2 * rs + sd2 * sqrtf(rd);
  return denom > 0.0f ? cw_delta_sq * (sd2 * rd) / denom : 0.0f;
}

__device__ __forceinline__ float wale_omega(float nu0, float nut) { return 1.0f / (3.0f * (nu0 + nut) + 0.5f); }

// What the closure inside the step reads for one cell: the six axis
// neighbours' velocities (x+ x- y+ y- z+ z-), the own one and the strain.  All
// are issued at construction; the own velocity only where a wall can be near.
template <bool PLAIN>
struct WaleLoads {
  float v[6][3], own[3], s[3];
  __device__ __forceinline__ WaleLoads(const WaleStep& w, const Dom& d, uint32_t i) {
    const int64_t sy = d.nx, sz = (int64_t)d.nx * d.ny;
    const int64_t off[6] = {1, -1, sy, -sy, sz, -sz};
#pragma unroll
    for (int n = 0; n < 6; ++n)
#pragma unroll
      for (int k = 0; k < 3; ++k) v[n][k] = (w.vel + (int64_t)k * (int64_t)w.ps + off[n])[i];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s[k] = (w.strain + k * w.ps)[i];
      own[k] = PLAIN ? 0.0f : (w.vel + k * w.ps)[i];
    }
  }
  // omega_plus of fluid cell i with mask word m on a closed domain: the link
  // bit of the direction that would come from a neighbour (1: x-, 2: x+,
  // 3: y-, ...) says that it is solid
  __device__ __forceinline__ float omega(const WaleStep& w, const Dom& d, const float* wall_u, uint32_t i,
                                         uint32_t m) {
    int kp[3], km[3];
    float pv[3][3], mv[3][3];
    const int64_t off[6] = {1, -1, (int64_t)d.nx, -(int64_t)d.nx, (int64_t)d.nx * d.ny, -(int64_t)d.nx * d.ny};
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      km[ax] = kp[ax] = 1;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        pv[ax][k] = v[2 * ax][k];
        mv[ax][k] = v[2 * ax + 1][k];
      }
    }
    if constexpr (!PLAIN) {
      if (m & 0x7Eu) {
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          if ((m >> (2 * ax + 1)) & 1u) km[ax] = 2;
          if ((m >> (2 * ax + 2)) & 1u) kp[ax] = 2;
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            if (km[ax] == 2) mv[ax][k] = wall_u ? wall_u[3 * (size_t)((int64_t)i + off[2 * ax + 1]) + k] : 0.0f;
            if (kp[ax] == 2) pv[ax][k] = wall_u ? wall_u[3 * (size_t)((int64_t)i + off[2 * ax]) + k] : 0.0f;
          }
        }
      }
    }
    const float raw = wale_nut<PLAIN>(w.cw_delta_sq, own, s[0], s[1], s[2], kp, km, pv, mv);
    return wale_omega(w.nu0, w.nut_max >= 0.0f && raw > w.nut_max ? w.nut_max : raw);
  }
};
}  // namespace lbm
