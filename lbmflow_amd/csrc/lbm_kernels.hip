// lbm_kernels.hip — CDNA4 (gfx950) kernels around lbm-core's
// lattice-Boltzmann step (the collide-stream itself is lbm_hydro.hip): masks,
// device geometry, staging, moments and f64 reductions.
//
// Storage: q-major planes f[q*ps + cell] of the deviation f - w_q in fp32,
// or scaled by 1/w_q in fp16 / bf16.  Arithmetic is fp32, reductions are
// fp64; the whole file is compiled with -ffp-contract=off.
#include <algorithm>
#include <type_traits>

#include "lbm_device.hpp"

namespace lbm {

// clear the force field at the listed cells of all domains
__global__ void k_clear_batch(const HydroArgs* __restrict__ tab, const uint32_t* __restrict__ cells, uint32_t n) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  float* F = const_cast<float*>(tab[cells[2 * (size_t)k + 1]].F_cur);
  const size_t i = cells[2 * (size_t)k];
  F[3 * i] = 0.0f;
  F[3 * i + 1] = 0.0f;
  F[3 * i + 2] = 0.0f;
}

// moments readback (moments_row with the cached-moment force F_u + F_mom)
template <int Q, typename S>
__global__ void k_moments(Dom d, const S* f, const uint32_t* mask, const float* F_mom, HydroParams p, int odd,
                          uint32_t i0, uint32_t cnt, float* rho, float* ux, float* uy, float* uz) {
  // cells i0 .. i0 + cnt - 1, written at 0 .. cnt - 1
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= cnt) return;
  const uint32_t i = i0 + k;
  const uint32_t m = mask[i];
  if (m & kMaskSolid) {
    rho[k] = 1.0f;
    ux[k] = uy[k] = uz[k] = 0.0f;
    return;
  }
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  const Nbr nb(d, x, y, z);
  float fv[Q];
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    fv[q] = read_pop<Q, S, q>(f, d.ps, nb, i, m, odd != 0);
  });
  // the field is zero off the force list, whose fluid cells carry kMaskForced
  float Fm[3] = {p.F[0], p.F[1], p.F[2]};
  bool fon = p.force_on != 0;
  if (F_mom && (m & kMaskForced)) {
    for (int c = 0; c < 3; ++c) Fm[c] = p.F[c] + F_mom[3 * (size_t)i + c];
    fon = true;
  }
  float r, a, b, c;
  moments<Q>(fv, Fm, fon, r, a, b, c);
  rho[k] = r;
  ux[k] = a;
  uy[k] = b;
  uz[k] = c;
}

// stage in (dir 0: host layout -> device, parity reset to even) /
// stage out (dir 1: device -> host layout, de-permuted by parity).
// Cells i0 .. i0 + cnt - 1; the host layout holds Q planes of cnt.
template <int Q, typename S>
__global__ void k_stage(Dom d, S* f, float* h, const uint32_t* mask, int dir, int odd, uint32_t i0, uint32_t cnt) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= cnt) return;
  const uint32_t i = i0 + k;
  if (dir == 0) {
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      pop_st<S, Q, q>(f + (size_t)q * d.ps, i, h[(size_t)q * cnt + k]);
    });
    return;
  }
  const uint32_t m = mask[i];
  const bool solid = (m & kMaskSolid) != 0;
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  const Nbr nb(d, x, y, z);
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    h[(size_t)q * cnt + k] = solid ? 0.0f : read_pop<Q, S, q>(f, d.ps, nb, i, m, odd != 0);
  });
}

// Solver::init_with, solver.rs:2474-2623 (pass 2): feq of every cell plus
// the gradient non-equilibrium part on fluid cells.
template <int Q, typename S>
__global__ void k_init_with(Dom d, S* f, const uint32_t* mask, const float* rho, const float* u, float tau) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N) return;
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  const float r = rho[i];
  const float own[3] = {u[3 * (size_t)i], u[3 * (size_t)i + 1], u[3 * (size_t)i + 2]};
  // equilibrium(), kernels.rs:103-121
  const float three = 3.0f, f45 = 4.5f, f15 = 1.5f, half = 0.5f;
  float usq = own[0] * own[0];
  usq = usq + own[1] * own[1];
  usq = usq + own[2] * own[2];
  const float drho = r - 1.0f;
  float fv[Q];
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const float cu = cdot<q>(own[0], own[1], own[2]);
    fv[q] = lat_wf(Q, q) * (drho + r * (three * cu + f45 * cu * cu - f15 * usq));
  });
  const bool solid = (mask[i] & kMaskSolid) != 0;
  if (!solid) {
    const uint32_t n3[3] = {d.nx, d.ny, d.nz};
    const uint32_t c3[3] = {x, y, z};
    float grad[3][3];
    for (int ax = 0; ax < 3; ++ax) {
      float pv[3], mv[3];
      bool hp = false, hm = false;
      for (int sgn = -1; sgn <= 1; sgn += 2) {
        int64_t g[3] = {(int64_t)x, (int64_t)y, (int64_t)z};
        g[ax] += sgn;
        bool ok = true;
        if (g[ax] < 0 || g[ax] >= (int64_t)n3[ax]) {
          if (d.per[ax])
            g[ax] = (g[ax] + n3[ax]) % n3[ax];
          else
            ok = false;
        }
        if (ok) {
          const uint32_t j = (uint32_t)((g[2] * d.ny + g[1]) * d.nx + g[0]);
          if (mask[j] & kMaskSolid) ok = false;
          if (ok) {
            float* dst = sgn > 0 ? pv : mv;
            dst[0] = u[3 * (size_t)j];
            dst[1] = u[3 * (size_t)j + 1];
            dst[2] = u[3 * (size_t)j + 2];
          }
        }
        (sgn > 0 ? hp : hm) = ok;
      }
      (void)c3;
      for (int b = 0; b < 3; ++b) {
        if (hp && hm)
          grad[ax][b] = (pv[b] - mv[b]) * half;
        else if (hp)
          grad[ax][b] = pv[b] - own[b];
        else if (hm)
          grad[ax][b] = own[b] - mv[b];
        else
          grad[ax][b] = 0.0f;
      }
    }
    float div = grad[0][0];
    div = div + grad[1][1];
    div = div + grad[2][2];
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr float c0 = lat_c(q, 0), c1 = lat_c(q, 1), c2 = lat_c(q, 2);
      float ccgu = c0 * c0 * grad[0][0];
      ccgu = ccgu + c0 * c1 * (grad[0][1] + grad[1][0]);
      ccgu = ccgu + c0 * c2 * (grad[0][2] + grad[2][0]);
      ccgu = ccgu + c1 * c1 * grad[1][1];
      ccgu = ccgu + c1 * c2 * (grad[1][2] + grad[2][1]);
      ccgu = ccgu + c2 * c2 * grad[2][2];
      const float fneq = -lat_wf(Q, q) * r * tau * (three * ccgu - div);
      fv[q] = fv[q] + fneq;
    });
  }
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    pop_st<S, Q, q>(f + (size_t)q * d.ps, i, fv[q]);
  });
}

// f64 reductions (reduce_impl, backend.rs:920-970): one partial per block,
// fixed tree inside the block, partials summed in block order on the host.
template <int Q, typename S>
__global__ __launch_bounds__(256) void k_reduce(Dom d, const S* f, const uint32_t* mask, const float* F_cur,
                                                HydroParams p, int odd, int kind, int axis, double* partials) {
  __shared__ double sm[4];
  double acc = 0.0;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < d.N; i += gridDim.x * 256) {
    const uint32_t m = mask[i];
    if (m & kMaskSolid) continue;
    if (kind == 0) {
      acc += 1.0;
      continue;
    }
    uint32_t x, y, z;
    cell_xyz(d, i, x, y, z);
    const Nbr nb(d, x, y, z);
    double s = 0.0, mom = 0.0;
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      const double v = (double)read_pop<Q, S, q>(f, d.ps, nb, i, m, odd != 0);
      s += v;
      if (kind == 2) {
        const int c = axis == 0 ? lat_c(q, 0) : (axis == 1 ? lat_c(q, 1) : lat_c(q, 2));
        mom += (double)c * v;
      }
    });
    if (kind == 1) {
      acc += s;
    } else {
      double fa = (double)p.F[axis];
      if (F_cur) fa = fa + ((double)F_cur[3 * (size_t)i + axis] + 0.0);
      acc += mom + 0.5 * fa;
    }
  }
  block_sum256<1>(&acc, sm);
  if (threadIdx.x == 0) partials[blockIdx.x] = acc;
}

// The previous step's post-collision populations f*_q(j) (what the
// reference's second buffer holds between steps: fields.rs ftmp, the
// checkpoint's STALE_STASH section), recovered from the current state by
// undoing the streaming: f*_q(j) = f_q(j + c_q) when j + c_q is fluid; the
// reflected population f_opp(q)(j), less the moving-wall term 6 w rho
// (c_opp . u_wall) (rho of the current state), when j + c_q is solid; 0 for
// solid cells and where j + c_q lies beyond a non-periodic face (a slot the
// next stream overwrites).  Exact copies on resting walls.
template <int Q, typename S>
__global__ void k_poststate(Dom d, const S* f, const uint32_t* mask, const float* wall_u, int odd, float* out) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= d.N) return;
  const uint32_t m = mask[j];
  if (m & kMaskSolid) {
    for (int q = 0; q < Q; ++q) out[(size_t)q * d.N + j] = 0.0f;
    return;
  }
  uint32_t x, y, z;
  cell_xyz(d, j, x, y, z);
  const Nbr nb(d, x, y, z);
  float rho = 1.0f;
  if (wall_u && (m & kMaskMoving)) {
    float dr = 0.0f;
    sfor<0, Q>([&](auto qc) { dr = dr + read_pop<Q, S, decltype(qc)::value>(f, d.ps, nb, j, m, odd != 0); });
    rho = 1.0f + dr;
  }
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int o = lat_opp(q);
    constexpr int cx = lat_c(q, 0), cy = lat_c(q, 1), cz = lat_c(q, 2);
    float v = 0.0f;
    if (q != 0 && ((m >> o) & 1u)) {  // j + c_q solid: reflected into f_opp(j)
      v = read_pop<Q, S, o>(f, d.ps, nb, j, m, odd != 0);
      if (wall_u && (m & kMaskMoving)) {
        const uint32_t t = j + (uint32_t)nb.template off<cx, cy, cz>();
        const float* wu = wall_u + 3 * (size_t)t;
        v = v - 6.0f * lat_wf(Q, o) * rho * cdot<o>(wu[0], wu[1], wu[2]);
      }
    } else {
      const int64_t tx = (int64_t)x + cx, ty = (int64_t)y + cy, tz = (int64_t)z + cz;
      const bool out_x = (tx < 0 || tx >= (int64_t)d.nx) && !d.per[0];
      const bool out_y = (ty < 0 || ty >= (int64_t)d.ny) && !d.per[1];
      const bool out_z = (tz < 0 || tz >= (int64_t)d.nz) && !d.per[2];
      if (!(out_x || out_y || out_z)) {
        const uint32_t t = j + (uint32_t)nb.template off<cx, cy, cz>();
        uint32_t ux, uy, uz;
        cell_xyz(d, t, ux, uy, uz);
        const Nbr nt(d, ux, uy, uz);
        v = read_pop<Q, S, q>(f, d.ps, nt, t, mask[t], odd != 0);
      }
    }
    out[(size_t)q * d.N + j] = v;
  });
}

// masks: links in the pull convention plus cell flags
template <int Q>
__global__ void k_build_mask(Dom d, const uint8_t* solid, const float* wall_u, uint32_t* mask,
                             unsigned int* err) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N) return;
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  if (solid[i]) {
    // bit q: the odd-step store target of direction q (i + c_q, wrapped or
    // linear, as either addressing of the collide-stream kernel reaches it)
    // is a fluid cell, which writes that slot itself
    const Nbr nb(d, x, y, z);
    uint32_t m = kMaskSolid;
    sfor<1, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int cx = lat_c(q, 0), cy = lat_c(q, 1), cz = lat_c(q, 2);
      const uint32_t jw = i + (uint32_t)nb.template off<cx, cy, cz>();
      const int64_t jl = (int64_t)i + cx + cy * (int64_t)d.nx + cz * (int64_t)d.nx * d.ny;
      const bool fluid_target = !solid[jw] || (jl >= 0 && jl < (int64_t)d.N && !solid[jl]);
      if (fluid_target) m |= 1u << q;
    });
    mask[i] = m;
    return;
  }
  const bool edge = (!d.per[0] && (x == 0 || x == d.nx - 1)) || (!d.per[1] && (y == 0 || y == d.ny - 1)) ||
                    (!d.per[2] && (z == 0 || z == d.nz - 1));
  if (edge) atomicAdd(err, 1u);
  const Nbr nb(d, x, y, z);
  uint32_t m = 0;
  sfor<1, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const uint32_t s = i + (uint32_t)nb.template off<-lat_c(q, 0), -lat_c(q, 1), -lat_c(q, 2)>();
    if (solid[s]) {
      m |= 1u << q;
      if (wall_u && (wall_u[3 * (size_t)s] != 0.0f || wall_u[3 * (size_t)s + 1] != 0.0f ||
                     wall_u[3 * (size_t)s + 2] != 0.0f))
        m |= kMaskMoving;
    }
  });
  mask[i] = m;
}

// flags per 64-cell x-segment: bit 0 some cell for the main kernel, bit 1
// all 64 cells plain fluid (mask word 0), bits 2/3 lanes 0-31 / 32-63 all
// solid (or past the row end)
// Linear tiles (`linear`): tile t is cells 64t .. 64t + 63 of the linear
// index, across row ends, with the same four flags.
__global__ void k_tile_flags(Dom d, const uint32_t* mask, uint8_t* flags, int linear) {
  const uint32_t nseg = (d.nx + 63) / 64;
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t c0, c1;
  if (linear) {
    if (t >= (d.N + 63) / 64) return;
    c0 = t * 64;
    c1 = min(c0 + 64, d.N);
  } else {
    if (t >= nseg * d.ny * d.nz) return;
    const uint32_t row = t / nseg, seg = t - row * nseg;
    c0 = row * d.nx + seg * 64;
    c1 = row * d.nx + min(seg * 64 + 64, d.nx);
  }
  bool any = false, plain = c1 - c0 == 64, dead[2] = {true, true};
  for (uint32_t c = c0; c < c1; ++c) {
    const uint32_t m = mask[c];
    if (!(m & (kMaskSolid | kMaskForced))) any = true;
    if (m != 0u) plain = false;
    if (!(m & kMaskSolid)) dead[(c - c0) >> 5] = false;
  }
  flags[t] = (uint8_t)((any ? 1 : 0) | (plain ? 2 : 0) | (dead[0] ? 4 : 0) | (dead[1] ? 8 : 0));
}

__global__ void k_mark_forced(const uint32_t* flist, uint32_t n, uint32_t* mask) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t i = flist[k];
  if (!(mask[i] & kMaskSolid)) mask[i] |= kMaskForced;
}

// apply_cylindrical_tank_mask + apply_baffle_mask (geometry.rs:657-723),
// f64 with the same expressions (no contraction in this file).
__global__ void k_tank(Dom d, double dx, double diameter, double height, int baffles, double bw, double bt,
                       uint8_t* solid) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N) return;
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  const double radius = 0.5 * diameter;
  const double cx = 0.5 * (double)d.nx * dx, cy = 0.5 * (double)d.ny * dx;
  const double z_m = ((double)z + 0.5) * dx;
  const double pxm = ((double)x + 0.5) * dx, pym = ((double)y + 0.5) * dx;
  const double r = sqrt((pxm - cx) * (pxm - cx) + (pym - cy) * (pym - cy));
  const bool rim = x == 0 || y == 0 || z == 0 || x + 1 == d.nx || y + 1 == d.ny || z + 1 == d.nz;
  const bool outside = r >= radius || z_m >= height;
  bool s = rim || outside;
  if (baffles == 4 && !rim && !(z_m >= height)) {
    const double rx = pxm - cx, ry = pym - cy;
    const double rb = sqrt(rx * rx + ry * ry);
    const double radial_inner = radius - bw;
    if (!(rb >= radius || rb < radial_inner)) {
      if (fabs(ry) <= 0.5 * bt || fabs(rx) <= 0.5 * bt) s = true;
    }
  }
  if (s) solid[i] = 1;
}

// build_wall_rims, solver.rs:1357-1406: one launch per face in the
// reference's order; the faster wall keeps the corner.
__global__ void k_rim_face(Dom d, int face, double speed, float u0, float u1, float u2, uint8_t* solid,
                           float* wall_u, double* best) {
  const int a = face / 2;
  const int t1 = a == 0 ? 1 : 0, t2 = a == 2 ? 1 : 2;
  const uint32_t n3[3] = {d.nx, d.ny, d.nz};
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n3[t1] * n3[t2]) return;
  uint32_t pos[3];
  pos[a] = (face % 2 == 0) ? 0 : n3[a] - 1;
  pos[t1] = k % n3[t1];
  pos[t2] = k / n3[t1];
  const uint32_t i = (pos[2] * d.ny + pos[1]) * d.nx + pos[0];
  solid[i] = 1;
  // best[] holds the squared speed of the velocity stored so far (-1 = none)
  if (speed > best[i]) {
    best[i] = speed;
    wall_u[3 * (size_t)i + 0] = u0;
    wall_u[3 * (size_t)i + 1] = u1;
    wall_u[3 * (size_t)i + 2] = u2;
  }
}

__global__ void k_fill(float* p, size_t n, float v) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_copy_list(const uint32_t* flist, uint32_t n, float* dst, const float* src) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const size_t i = flist[k];
  dst[3 * i] = src ? src[3 * i] : 0.0f;
  dst[3 * i + 1] = src ? src[3 * i + 1] : 0.0f;
  dst[3 * i + 2] = src ? src[3 * i + 2] : 0.0f;
}

// STREAM copy (b[i] = a[i]) with 16-byte accesses: the measured HBM ceiling
// and the calibration run for the byte counters.
__global__ __launch_bounds__(256) void k_stream_copy(const float4* __restrict__ a, float4* __restrict__ b, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) b[i] = a[i];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
Tiling make_tiling(const Dom& d, uint32_t tx_pref) {
  Tiling t;
  uint32_t tx = tx_pref ? tx_pref : 256;
  while (tx > 64 && tx / 2 >= d.nx) tx /= 2;
  t.tx = tx;
  t.ty = 256 / tx;
  t.bx = (d.nx + t.tx - 1) / t.tx;
  t.by = (d.ny + t.ty - 1) / t.ty;
  t.nblocks = t.bx * t.by * d.nz;
  return t;
}

static inline uint32_t blocks_for(size_t n, uint32_t bs = 256) { return (uint32_t)((n + bs - 1) / bs); }
// The collide-stream launchers of each lattice, storage and collision
// (lbm_hydro.hip).
template <int Q, int KIND>
static hipError_t hydro_kind(int storage, int odd, const HydroArgs& a, hipStream_t s, bool list) {
  if (storage == kF32) return hydro_launch<Q, kF32, KIND>(odd, a, s, list);
  if (storage == kF16) return hydro_launch<Q, kF16, KIND>(odd, a, s, list);
  return hydro_launch<Q, kBF16, KIND>(odd, a, s, list);
}
template <int Q>
static hipError_t hydro_any(int storage, int collision, int odd, const HydroArgs& a, hipStream_t s, bool list) {
  return collision == 2 ? hydro_kind<Q, 1>(storage, odd, a, s, list) : hydro_kind<Q, 0>(storage, odd, a, s, list);
}

hipError_t launch_hydro(int Q, int storage, int collision, int odd, const HydroArgs& a, hipStream_t s) {
  if (Q == 19) return hydro_any<19>(storage, collision, odd, a, s, false);
  if (Q == 27) return hydro_any<27>(storage, collision, odd, a, s, false);
  return hipErrorInvalidValue;
}

hipError_t launch_hydro_list(int Q, int storage, int collision, int odd, const HydroArgs& a, hipStream_t s) {
  if (Q == 19) return hydro_any<19>(storage, collision, odd, a, s, true);
  if (Q == 27) return hydro_any<27>(storage, collision, odd, a, s, true);
  return hipErrorInvalidValue;
}

template <int Q, int KIND>
static hipError_t batch_kind(int storage, int odd, const HydroArgs* tab, const uint32_t* ent, uint32_t nent,
                             uint32_t grid, const uint32_t* cells, uint32_t ncells, hipStream_t s) {
  if (storage == kF32) return batch_launch<Q, kF32, KIND>(odd, tab, ent, nent, grid, cells, ncells, s);
  if (storage == kF16) return batch_launch<Q, kF16, KIND>(odd, tab, ent, nent, grid, cells, ncells, s);
  return batch_launch<Q, kBF16, KIND>(odd, tab, ent, nent, grid, cells, ncells, s);
}
template <int Q>
static hipError_t batch_any(int storage, int collision, int odd, const HydroArgs* tab, const uint32_t* ent,
                            uint32_t nent, uint32_t grid, const uint32_t* cells, uint32_t ncells, hipStream_t s) {
  return collision == 2 ? batch_kind<Q, 1>(storage, odd, tab, ent, nent, grid, cells, ncells, s)
                        : batch_kind<Q, 0>(storage, odd, tab, ent, nent, grid, cells, ncells, s);
}

hipError_t launch_hydro_batch(int Q, int storage, int collision, int odd, const HydroArgs* tab, const uint32_t* ent,
                              uint32_t nent, uint32_t grid, hipStream_t s) {
  if (grid == 0) return hipErrorInvalidValue;
  if (Q == 19) return batch_any<19>(storage, collision, odd, tab, ent, nent, grid, nullptr, 0, s);
  if (Q == 27) return batch_any<27>(storage, collision, odd, tab, ent, nent, grid, nullptr, 0, s);
  return hipErrorInvalidValue;
}

hipError_t launch_hydro_list_batch(int Q, int storage, int collision, int odd, const HydroArgs* tab,
                                   const uint32_t* cells, uint32_t n, hipStream_t s) {
  if (Q == 19) return batch_any<19>(storage, collision, odd, tab, nullptr, 0, 0, cells, n, s);
  if (Q == 27) return batch_any<27>(storage, collision, odd, tab, nullptr, 0, 0, cells, n, s);
  return hipErrorInvalidValue;
}

// The open-face and volume-source launchers of each lattice and storage
// (lbm_open.hip).
hipError_t launch_open_faces(int Q, int storage, const FaceArgs& a, hipStream_t s) {
  if (storage == kF32) return Q == 19 ? open_launch<19, kF32>(a, s) : open_launch<27, kF32>(a, s);
  if (storage == kF16) return Q == 19 ? open_launch<19, kF16>(a, s) : open_launch<27, kF16>(a, s);
  return Q == 19 ? open_launch<19, kBF16>(a, s) : open_launch<27, kBF16>(a, s);
}

hipError_t launch_volume_source(int Q, int storage, const SourceArgs& a, hipStream_t s) {
  if (storage == kF32) return Q == 19 ? source_launch<19, kF32>(a, s) : source_launch<27, kF32>(a, s);
  if (storage == kF16) return Q == 19 ? source_launch<19, kF16>(a, s) : source_launch<27, kF16>(a, s);
  return Q == 19 ? source_launch<19, kBF16>(a, s) : source_launch<27, kBF16>(a, s);
}

// fluid cells of non-periodic faces that no open face covers
__global__ void k_uncovered(Dom d, const uint8_t* solid, uint32_t open_bits, unsigned int* count) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N || solid[i]) return;
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  const uint32_t c[3] = {x, y, z}, n[3] = {d.nx, d.ny, d.nz};
  bool bad = false;
  for (int ax = 0; ax < 3; ++ax) {
    if (d.per[ax]) continue;
    if (c[ax] == 0 && !((open_bits >> (2 * ax)) & 1u)) bad = true;
    if (c[ax] == n[ax] - 1 && !((open_bits >> (2 * ax + 1)) & 1u)) bad = true;
  }
  if (bad) atomicAdd(count, 1u);
}

hipError_t launch_uncovered(const Dom& d, const uint8_t* solid, uint32_t open_bits, unsigned int* count,
                            hipStream_t s) {
  hipLaunchKernelGGL(k_uncovered, dim3((d.N + 255) / 256), dim3(256), 0, s, d, solid, open_bits, count);
  return hipGetLastError();
}

hipError_t launch_clear_batch(const HydroArgs* tab, const uint32_t* cells, uint32_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_clear_batch, dim3(blocks_for(n)), dim3(256), 0, s, tab, cells, n);
  return hipGetLastError();
}

hipError_t launch_build_mask(int Q, const Dom& d, const uint8_t* solid, const float* wall_u, uint32_t* mask,
                             unsigned int* err, hipStream_t s) {
  if (Q == 19)
    hipLaunchKernelGGL((k_build_mask<19>), dim3(blocks_for(d.N)), dim3(256), 0, s, d, solid, wall_u, mask, err);
  else
    hipLaunchKernelGGL((k_build_mask<27>), dim3(blocks_for(d.N)), dim3(256), 0, s, d, solid, wall_u, mask, err);
  return hipGetLastError();
}

hipError_t launch_tile_flags(const Dom& d, const uint32_t* mask, uint8_t* flags, int linear, hipStream_t s) {
  const size_t nt = linear ? (size_t)(d.N + 63) / 64 : (size_t)((d.nx + 63) / 64) * d.ny * d.nz;
  hipLaunchKernelGGL(k_tile_flags, dim3(blocks_for(nt)), dim3(256), 0, s, d, mask, flags, linear);
  return hipGetLastError();
}

hipError_t launch_mark_forced(const uint32_t* flist, uint32_t n, uint32_t* mask, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mark_forced, dim3(blocks_for(n)), dim3(256), 0, s, flist, n, mask);
  return hipGetLastError();
}

template <typename S>
static hipError_t stage_s(int Q, int dir, int odd, const Dom& d, void* f, float* h, const uint32_t* mask, uint32_t i0,
                          uint32_t cnt, hipStream_t s) {
  if (Q == 19)
    hipLaunchKernelGGL((k_stage<19, S>), dim3(blocks_for(cnt)), dim3(256), 0, s, d, (S*)f, h, mask, dir, odd, i0, cnt);
  else
    hipLaunchKernelGGL((k_stage<27, S>), dim3(blocks_for(cnt)), dim3(256), 0, s, d, (S*)f, h, mask, dir, odd, i0, cnt);
  return hipGetLastError();
}

hipError_t launch_stage(int Q, int storage, int dir, int odd, const Dom& d, void* f, float* h, const uint32_t* mask,
                        uint32_t i0, uint32_t cnt, hipStream_t s) {
  if (storage == kF32) return stage_s<float>(Q, dir, odd, d, f, h, mask, i0, cnt, s);
  if (storage == kF16) return stage_s<_Float16>(Q, dir, odd, d, f, h, mask, i0, cnt, s);
  return stage_s<bf16s>(Q, dir, odd, d, f, h, mask, i0, cnt, s);
}

template <typename S>
static hipError_t init_s(int Q, const Dom& d, void* f, const uint32_t* mask, const float* rho, const float* u,
                         float tau, hipStream_t s) {
  if (Q == 19)
    hipLaunchKernelGGL((k_init_with<19, S>), dim3(blocks_for(d.N)), dim3(256), 0, s, d, (S*)f, mask, rho, u, tau);
  else
    hipLaunchKernelGGL((k_init_with<27, S>), dim3(blocks_for(d.N)), dim3(256), 0, s, d, (S*)f, mask, rho, u, tau);
  return hipGetLastError();
}

hipError_t launch_init_with(int Q, int storage, const Dom& d, void* f, const uint32_t* mask, const float* rho,
                            const float* u, float tau, hipStream_t s) {
  if (storage == kF32) return init_s<float>(Q, d, f, mask, rho, u, tau, s);
  if (storage == kF16) return init_s<_Float16>(Q, d, f, mask, rho, u, tau, s);
  return init_s<bf16s>(Q, d, f, mask, rho, u, tau, s);
}

template <typename S>
static hipError_t moments_s(int Q, int odd, const Dom& d, const void* f, const uint32_t* mask, const float* F_mom,
                            HydroParams p, uint32_t i0, uint32_t cnt, float* rho, float* ux, float* uy, float* uz,
                            hipStream_t s) {
  if (Q == 19)
    hipLaunchKernelGGL((k_moments<19, S>), dim3(blocks_for(cnt)), dim3(256), 0, s, d, (const S*)f, mask, F_mom, p,
                       odd, i0, cnt, rho, ux, uy, uz);
  else
    hipLaunchKernelGGL((k_moments<27, S>), dim3(blocks_for(cnt)), dim3(256), 0, s, d, (const S*)f, mask, F_mom, p,
                       odd, i0, cnt, rho, ux, uy, uz);
  return hipGetLastError();
}

template <typename S>
static hipError_t poststate_s(int Q, int odd, const Dom& d, const void* f, const uint32_t* mask, const float* wall_u,
                              float* out, hipStream_t s) {
  if (Q == 19)
    hipLaunchKernelGGL((k_poststate<19, S>), dim3(blocks_for(d.N)), dim3(256), 0, s, d, (const S*)f, mask, wall_u, odd,
                       out);
  else
    hipLaunchKernelGGL((k_poststate<27, S>), dim3(blocks_for(d.N)), dim3(256), 0, s, d, (const S*)f, mask, wall_u, odd,
                       out);
  return hipGetLastError();
}

hipError_t launch_poststate(int Q, int storage, int odd, const Dom& d, const void* f, const uint32_t* mask,
                            const float* wall_u, float* out, hipStream_t s) {
  if (storage == kF32) return poststate_s<float>(Q, odd, d, f, mask, wall_u, out, s);
  if (storage == kF16) return poststate_s<_Float16>(Q, odd, d, f, mask, wall_u, out, s);
  return poststate_s<bf16s>(Q, odd, d, f, mask, wall_u, out, s);
}

hipError_t launch_moments(int Q, int storage, int odd, const Dom& d, const void* f, const uint32_t* mask,
                          const float* F_mom, HydroParams p, uint32_t i0, uint32_t cnt, float* rho, float* ux,
                          float* uy, float* uz, hipStream_t s) {
  if (storage == kF32) return moments_s<float>(Q, odd, d, f, mask, F_mom, p, i0, cnt, rho, ux, uy, uz, s);
  if (storage == kF16) return moments_s<_Float16>(Q, odd, d, f, mask, F_mom, p, i0, cnt, rho, ux, uy, uz, s);
  return moments_s<bf16s>(Q, odd, d, f, mask, F_mom, p, i0, cnt, rho, ux, uy, uz, s);
}

template <typename S>
static hipError_t reduce_s(int Q, int odd, const Dom& d, const void* f, const uint32_t* mask, const float* F,
                           HydroParams p, int kind, int axis, double* partials, uint32_t np, hipStream_t s) {
  if (Q == 19)
    hipLaunchKernelGGL((k_reduce<19, S>), dim3(np), dim3(256), 0, s, d, (const S*)f, mask, F, p, odd, kind, axis,
                       partials);
  else
    hipLaunchKernelGGL((k_reduce<27, S>), dim3(np), dim3(256), 0, s, d, (const S*)f, mask, F, p, odd, kind, axis,
                       partials);
  return hipGetLastError();
}

hipError_t launch_reduce(int Q, int storage, int odd, const Dom& d, const void* f, const uint32_t* mask,
                         const float* F, HydroParams p, int kind, int axis, double* partials, uint32_t np,
                         hipStream_t s) {
  if (storage == kF32) return reduce_s<float>(Q, odd, d, f, mask, F, p, kind, axis, partials, np, s);
  if (storage == kF16) return reduce_s<_Float16>(Q, odd, d, f, mask, F, p, kind, axis, partials, np, s);
  return reduce_s<bf16s>(Q, odd, d, f, mask, F, p, kind, axis, partials, np, s);
}

hipError_t launch_tank(const Dom& d, double dx, double diameter, double height, int baffles, double bw, double bt,
                       uint8_t* solid, hipStream_t s) {
  hipLaunchKernelGGL(k_tank, dim3(blocks_for(d.N)), dim3(256), 0, s, d, dx, diameter, height, baffles, bw, bt,
                     solid);
  return hipGetLastError();
}

__global__ void k_filld(double* p, size_t n, double v) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

hipError_t launch_rims(const Dom& d, const int is_wall[6], const double u[18], uint8_t* solid, float* wall_u,
                       double* best, hipStream_t s) {
  hipLaunchKernelGGL(k_filld, dim3(blocks_for(d.N)), dim3(256), 0, s, best, (size_t)d.N, -1.0);
  const int order[6] = {2, 3, 0, 1, 4, 5};  // YNeg, YPos, XNeg, XPos, ZNeg, ZPos
  const uint32_t n3[3] = {d.nx, d.ny, d.nz};
  for (int k = 0; k < 6; ++k) {
    const int face = order[k];
    if (!is_wall[face]) continue;
    const int a = face / 2;
    const int t1 = a == 0 ? 1 : 0, t2 = a == 2 ? 1 : 2;
    const float u0 = (float)u[3 * face], u1 = (float)u[3 * face + 1], u2 = (float)u[3 * face + 2];
    double speed = (double)u0 * (double)u0 + (double)u1 * (double)u1;
    speed += (double)u2 * (double)u2;
    const size_t cnt = (size_t)n3[t1] * n3[t2];
    hipLaunchKernelGGL(k_rim_face, dim3(blocks_for(cnt)), dim3(256), 0, s, d, face, speed, u0, u1, u2, solid,
                       wall_u, best);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Copy n elements of T, each lane one naturally aligned element per
// iteration, starting OFF elements past 256-byte-aligned bases: the access
// widths and line offsets of the collide-stream kernels (4-byte planes, and
// their x-shifted neighbour rows that put a wave across three lines; 2-byte
// planes of 16-bit storage) next to the 16-byte copy, for calibrating the
// memory counters per access form.
template <typename T, int OFF>
__global__ __launch_bounds__(256) void k_access_copy(const T* __restrict__ a, T* __restrict__ b, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    b[OFF + i] = a[OFF + i];
}

hipError_t launch_access_copy(int width, int offset_elems, const void* a, void* b, size_t n, hipStream_t s) {
  const uint32_t grid = (uint32_t)std::min<size_t>((n + 255) / 256, 256 * 8 * 64);
  if (width == 16 && offset_elems == 0)
    hipLaunchKernelGGL((k_access_copy<uint4, 0>), dim3(grid), dim3(256), 0, s, (const uint4*)a, (uint4*)b, n);
  else if (width == 4 && offset_elems == 0)
    hipLaunchKernelGGL((k_access_copy<uint32_t, 0>), dim3(grid), dim3(256), 0, s, (const uint32_t*)a, (uint32_t*)b, n);
  else if (width == 4 && offset_elems == 1)
    hipLaunchKernelGGL((k_access_copy<uint32_t, 1>), dim3(grid), dim3(256), 0, s, (const uint32_t*)a, (uint32_t*)b, n);
  else if (width == 2 && offset_elems == 0)
    hipLaunchKernelGGL((k_access_copy<uint16_t, 0>), dim3(grid), dim3(256), 0, s, (const uint16_t*)a, (uint16_t*)b, n);
  else if (width == 2 && offset_elems == 1)
    hipLaunchKernelGGL((k_access_copy<uint16_t, 1>), dim3(grid), dim3(256), 0, s, (const uint16_t*)a, (uint16_t*)b, n);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_stream_copy(const void* a, void* b, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  const uint32_t grid = (uint32_t)std::min<size_t>((n + 255) / 256, 256 * 8 * 64);
  hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, s, (const float4*)a, (float4*)b, n);
  return hipGetLastError();
}

// Into pinned memory, 16 bytes per lane where both ends allow it (dst is a slot
// or a place in it, src any array): bound by the host link.
template <typename T>
__global__ __launch_bounds__(256) void k_to_host(T* dst, const T* src, size_t n) {
  const size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_to_host(void* dst, const void* src, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (((uintptr_t)dst | (uintptr_t)src | n) % 16 == 0) {
    const size_t v = n / 16;
    hipLaunchKernelGGL((k_to_host<uint4>), dim3((unsigned)std::min<size_t>((v + 255) / 256, 512)), dim3(256), 0, s,
                       (uint4*)dst, (const uint4*)src, v);
  } else {
    const size_t v = n / 4;
    hipLaunchKernelGGL((k_to_host<uint32_t>), dim3((unsigned)std::min<size_t>((v + 255) / 256, 2048)), dim3(256), 0,
                       s, (uint32_t*)dst, (const uint32_t*)src, v);
  }
  return hipGetLastError();
}

hipError_t launch_fill_f32(float* p, size_t n, float v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill, dim3(blocks_for(n)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_copy_force_list(const uint32_t* flist, uint32_t n, float* dst, const float* src, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_copy_list, dim3(blocks_for(n)), dim3(256), 0, s, flist, n, dst, src);
  return hipGetLastError();
}

}  // namespace lbm
