// lbm_les.hip — WALE large-eddy closure (Nicoud & Ducros 1999) as a
// producer of the per-cell omega_plus field the collide-stream kernels read.
//
// Two cell-parallel passes per update (WaleLes::update, les.rs:120-211):
//   k_wale_local  reads the cell's Q populations once and writes the cached
//     velocity of the current state (moments_row) and the off-diagonal
//     strain from the non-equilibrium stress (strain_rate_at,
//     solver.rs:5393-5447) into a 6 x N work buffer;
//   k_wale        takes the velocity gradient g = du_i/dx_j: diagonal from
//     finite differences of the cached velocity, off-diagonal S + the
//     antisymmetric part of the finite differences
//     (gather_velocity_gradient, solver.rs:5490-5581), then
//     nu_t = (Cw Delta)^2 (Sd:Sd)^(3/2) / ((S:S)^(5/2) + (Sd:Sd)^(5/4)),
//     clipped to nu_t_max when asked, omega = 1/(3 (nu0 + nu_t) + 1/2).
//     The second pass marches (x, y) columns along z with the z - 1, z,
//     z + 1 velocities in registers, so each velocity is read from memory
//     once; x and y neighbours come from the tile's own rows in L2.
// On closed domains the per-step closure does without the second pass: the
// collide-stream kernel takes the same gradient and nu_t of each cell it
// updates (lbm_wale.hpp).
// Bytes per fluid cell: Q S + 4 (mask) + 24 in the first pass; 4 + 24 + the
// neighbours' velocities (mostly from L2) + 4 in the second, 24 + 4 inside the
// step.  Per solid cell 4 in the first pass (nothing is stored), 8 in the second.
#include <cstdlib>
#include <type_traits>

#include "lbm_device.hpp"
#include "lbm_internal.hpp"
#include "lbm_scalar.hpp"
#include "lbm_wale.hpp"

#pragma clang fp contract(off)

namespace lbm {

// what the second pass computes with and writes
struct WaleOut {
  float cw_delta_sq;  // (Cw Delta)^2
  float nu0;          // laminar viscosity
  float nut_max;      // < 0: no clip
  float* omega;       // N: omega_plus
  float* nut;         // N or null: nu_t (after the clip)
  uint32_t* stats;    // null or [clipped cells, bits of the largest raw nu_t]
};

// NT: the first pass loads its populations non-temporally (wale_nt).
template <int Q, typename S, int q, bool NT>
__device__ __forceinline__ float read_pop_once(const S* base, size_t ps, const Nbr& nb, uint32_t i, uint32_t m,
                                               bool odd) {
  if constexpr (NT) {
    const bool own = !odd || ((m >> q) & 1u);
    const uint32_t j = own ? i : i + (uint32_t)nb.template off<-lat_c(q, 0), -lat_c(q, 1), -lat_c(q, 2)>();
    using Raw = std::conditional_t<sizeof(S) == 4, float, uint16_t>;
    const Raw raw = __builtin_nontemporal_load((const Raw*)(base + (size_t)(own ? q : lat_opp(q)) * ps + j));
    const S v = __builtin_bit_cast(S, raw);
    return pop_ld<S, Q, q>(&v, 0);
  } else {
    return read_pop<Q, S, q>(base, ps, nb, i, m, odd);
  }
}

// Pass 1, per cell: the cached moments (moments_row with the force the state
// was produced under, as the moment readback computes them) and the
// off-diagonal strain from the same populations, read once.
// A solid cell's values are never read (a solid neighbour contributes its
// wall velocity).  With QS the pass takes the previous step's passive-scalar
// step along (no axis wraps then): it collides with exactly these velocities,
// so its own read of the populations (Q S bytes per cell) is saved.
// Blocks in the plain order: against stretches and runs per XCD (xcd_remap) the
// best or within 1 % of it at every size measured, 3 to 7 % better for large
// fp32 domains (512^3 tank 8.52 -> 7.93 ms per step with the loads of wale_nt).
template <int Q, typename S, bool WRAP, int QS, bool NT>
__global__ __launch_bounds__(256) void k_wale_local(WaleFields a, ScalarStepArgs sc) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.d.N) return;
  float* const vel = a.work;
  float* const strain = a.work + 3 * a.ps;
  const uint32_t m = a.mask[i];
  if (m & kMaskSolid) return;
  uint32_t x = 0, y = 0, z = 0;
  if constexpr (WRAP) cell_xyz(a.d, i, x, y, z);
  const Nbr nb = WRAP ? Nbr(a.d, x, y, z) : Nbr(a.d);
  float hv[QS > 0 ? QS : 1], fv[Q];
  if constexpr (QS > 0) scalar_load<QS>(sc, i, hv);
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    fv[q] = read_pop_once<Q, S, q, NT>((const S*)a.f, a.d.ps, nb, i, m, a.odd != 0);
  });
  float Fm[3] = {a.p.F[0], a.p.F[1], a.p.F[2]};
  bool fon = a.p.force_on != 0;
  if (a.F_mom && (m & kMaskForced)) {
    for (int c = 0; c < 3; ++c) Fm[c] = a.p.F[c] + a.F_mom[3 * (size_t)i + c];
    fon = true;
  }
  float r, u0, u1, u2;
  moments<Q>(fv, Fm, fon, r, u0, u1, u2);
  vel[i] = u0;
  vel[a.ps + i] = u1;
  vel[2 * a.ps + i] = u2;
  if constexpr (QS > 0) scalar_push<QS>(sc, nb, i, m, hv, u0, u1, u2);
  // Pi_neq = sum_q c c (f_q - feq_q), deviation-form equilibrium
  // (kernels.rs:103-121); terms with a zero factor add exact zeros in the
  // reference's sums and are dropped.
  const float usq = u0 * u0 + u1 * u1 + u2 * u2;
  const float drho = r - 1.0f;
  float pxy = 0.0f, pxz = 0.0f, pyz = 0.0f;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int cx = lat_c(q, 0), cy = lat_c(q, 1), cz = lat_c(q, 2);
    const float cu = cdot<q>(u0, u1, u2);
    const float feq = lat_wf(Q, q) * (drho + r * (3.0f * cu + 4.5f * cu * cu - 1.5f * usq));
    const float fn = fv[q] - feq;
    if constexpr (cx * cy == 1) pxy = pxy + fn;
    if constexpr (cx * cy == -1) pxy = pxy - fn;
    if constexpr (cx * cz == 1) pxz = pxz + fn;
    if constexpr (cx * cz == -1) pxz = pxz - fn;
    if constexpr (cy * cz == 1) pyz = pyz + fn;
    if constexpr (cy * cz == -1) pyz = pyz - fn;
  });
  // Guo-force correction of the stress, + (u_a F_b + u_b F_a)/2 off the
  // diagonal, F = uniform force + current field
  float F0 = a.p.F[0], F1 = a.p.F[1], F2 = a.p.F[2];
  if (a.F_cur && (m & kMaskForced)) {  // the field is zero off the force list
    F0 = F0 + a.F_cur[3 * (size_t)i + 0];
    F1 = F1 + a.F_cur[3 * (size_t)i + 1];
    F2 = F2 + a.F_cur[3 * (size_t)i + 2];
  }
  pxy = pxy + 0.5f * (u0 * F1 + u1 * F0);
  pxz = pxz + 0.5f * (u0 * F2 + u2 * F0);
  pyz = pyz + 0.5f * (u1 * F2 + u2 * F1);
  // S = -Pi / (2 cs^2 rho tau), tau = 1/omega_p (the global rate)
  const float scale = -(1.0f / ((2.0f / 3.0f) * r * a.tau_eff));
  strain[i] = pxy * scale;
  strain[a.ps + i] = pxz * scale;
  strain[2 * a.ps + i] = pyz * scale;
}

// One neighbour of a finite difference: kind 0 none (non-periodic domain
// face), 1 fluid (v = its cached velocity), 2 solid (v = its wall velocity).
__device__ __forceinline__ int wale_nbr(const WaleFields& a, bool none, uint32_t j, uint32_t mj, const float* uj,
                                        float v[3]) {
  if (none) {
    v[0] = v[1] = v[2] = 0.0f;
    return 0;
  }
  if (mj & kMaskSolid) {
    if (a.wall_u) {
      v[0] = a.wall_u[3 * (size_t)j + 0];
      v[1] = a.wall_u[3 * (size_t)j + 1];
      v[2] = a.wall_u[3 * (size_t)j + 2];
    } else {
      v[0] = v[1] = v[2] = 0.0f;
    }
    return 2;
  }
  v[0] = uj[0];
  v[1] = uj[1];
  v[2] = uj[2];
  return 1;
}

// Pass 2: a block is a 64 x 4 tile of (x, y) columns, each thread marches
// its column over `zlen` cells keeping the mask and cached velocity of
// z - 1, z, z + 1 in registers, so every velocity is read from HBM about
// once; the x and y neighbours come from the rows the tile's own threads
// load (L2).  Each step of the march waits for its loads, so the march is
// kept short enough for the grid to hold many waves (wale_zlen).
constexpr uint32_t kWaleTileX = 64, kWaleTileY = 4;
static_assert(kWaleTileX * kWaleTileY == 256 && kWaleTileX == 64, "one wave per tile row, 256-thread blocks");

__global__ __launch_bounds__(256) void k_wale(WaleFields a, WaleOut o, uint32_t zlen) {
  const float* const vel = a.work;
  const float* const strain = a.work + 3 * a.ps;
  const uint32_t nx = a.d.nx, ny = a.d.ny, nz = a.d.nz;
  const uint32_t x = blockIdx.x * kWaleTileX + (threadIdx.x & (kWaleTileX - 1));
  const uint32_t y = blockIdx.y * kWaleTileY + threadIdx.x / kWaleTileX;
  const uint32_t z0 = blockIdx.z * zlen;
  const uint32_t z1 = min(z0 + zlen, nz);
  const size_t N = a.ps;
  const uint32_t plane = nx * ny;
  uint32_t cnt = 0u, mx = 0u;
  if (x < nx && y < ny && z0 < nz) {
    uint32_t i = (z0 * ny + y) * nx + x;
    const uint32_t iwrap = (nz - 1) * plane;  // z = 0 <-> z = nz - 1
    uint32_t jm = z0 == 0 ? i + iwrap : i - plane;
    uint32_t mm = a.mask[jm], mc = a.mask[i];
    float um[3] = {vel[jm], vel[N + jm], vel[2 * N + jm]};
    float uc[3] = {vel[i], vel[N + i], vel[2 * N + i]};
    for (uint32_t z = z0; z < z1; ++z) {
      const uint32_t jp = z == nz - 1 ? i - iwrap : i + plane;
      const uint32_t mp = a.mask[jp];
      const float up[3] = {vel[jp], vel[N + jp], vel[2 * N + jp]};
      float nut_raw = 0.0f;
      if (!(mc & kMaskSolid)) {
        const Nbr nb(a.d, x, y, z);
        int kp[3], km[3];
        float pv[3][3], mv[3][3];
        {
          const uint32_t j1 = i + (uint32_t)nb.xp, j2 = i + (uint32_t)nb.xm;
          const float u1[3] = {vel[j1], vel[N + j1], vel[2 * N + j1]};
          const float u2[3] = {vel[j2], vel[N + j2], vel[2 * N + j2]};
          kp[0] = wale_nbr(a, x == nx - 1 && !a.d.per[0], j1, a.mask[j1], u1, pv[0]);
          km[0] = wale_nbr(a, x == 0 && !a.d.per[0], j2, a.mask[j2], u2, mv[0]);
        }
        {
          const uint32_t j1 = i + (uint32_t)nb.yp, j2 = i + (uint32_t)nb.ym;
          const float u1[3] = {vel[j1], vel[N + j1], vel[2 * N + j1]};
          const float u2[3] = {vel[j2], vel[N + j2], vel[2 * N + j2]};
          kp[1] = wale_nbr(a, y == ny - 1 && !a.d.per[1], j1, a.mask[j1], u1, pv[1]);
          km[1] = wale_nbr(a, y == 0 && !a.d.per[1], j2, a.mask[j2], u2, mv[1]);
        }
        kp[2] = wale_nbr(a, z == nz - 1 && !a.d.per[2], jp, mp, up, pv[2]);
        km[2] = wale_nbr(a, z == 0 && !a.d.per[2], jm, mm, um, mv[2]);
        nut_raw = wale_nut<false>(o.cw_delta_sq, uc, strain[i], strain[N + i], strain[2 * N + i], kp, km, pv, mv);
      }
      const bool clipped = o.nut_max >= 0.0f && nut_raw > o.nut_max;
      const float nut = clipped ? o.nut_max : nut_raw;
      o.omega[i] = wale_omega(o.nu0, nut);
      if (o.nut) o.nut[i] = nut;
      cnt += clipped ? 1u : 0u;
      mx = max(mx, __float_as_uint(nut_raw));
      // slide the window one cell up
      jm = i;
      mm = mc;
      um[0] = uc[0];
      um[1] = uc[1];
      um[2] = uc[2];
      i = jp;
      mc = mp;
      uc[0] = up[0];
      uc[1] = up[1];
      uc[2] = up[2];
    }
  }
  if (o.stats) {
    // block totals: clipped count and the largest raw nu_t (non-negative, so
    // its bit pattern orders like the value)
    __shared__ uint32_t s_cnt[4], s_max[4];
#pragma unroll
    for (int l = 32; l > 0; l >>= 1) {
      cnt += __shfl_xor(cnt, l);
      mx = max(mx, (uint32_t)__shfl_xor(mx, l));
    }
    const uint32_t w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      s_cnt[w] = cnt;
      s_max[w] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint32_t c = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
      const uint32_t b = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
      if (c) atomicAdd(&o.stats[0], c);
      if (b) atomicMax(&o.stats[1], b);
    }
  }
}

// March length of the second pass: the longest power of two up to 64 that
// still gives the grid 65,536 blocks, at least 4 (measured best: 4 cells at
// 256^3, 8 at 512^3; 64 cost 4.6 % and 1.5 % of the whole step there);
// LBM_WALE_ZLEN overrides it (tuning).  Any length gives the same values.
static uint32_t wale_zlen(const Dom& d) {
  if (const char* e = getenv("LBM_WALE_ZLEN")) {
    const long v = strtol(e, nullptr, 10);
    if (v >= 1 && v <= 1024) return (uint32_t)v;
  }
  const uint64_t cols = (uint64_t)((d.nx + kWaleTileX - 1) / kWaleTileX) * ((d.ny + kWaleTileY - 1) / kWaleTileY);
  uint32_t z = 64;
  while (z > 4 && cols * ((d.nz + z - 1) / z) < 65536) z >>= 1;
  return z;
}

// Whether the first pass's population loads are non-temporal: they keep the
// velocity planes in the caches for the pass that follows, which pays while the
// populations are a few times the last-level cache.  Below that they would be
// found in it by the step; far above, ordinary loads stream better.  ms per
// step with the closure, plain loads -> non-temporal, by bytes of populations:
//   tanks D3Q27 fp32 128^3 (0.23 GB) 0.175 -> 0.182, 200^3 (0.86) 0.650 -> 0.613,
//     256^3 (1.81) 1.170 -> 1.167, 320^3 2.17 -> 2.29, 512^3 7.93 -> 8.34;
//     fp16 128^3 (0.11) 0.145 -> 0.157, 200^3 (0.43) 0.446 -> 0.437, 320^3 (1.77)
//     1.45 -> 1.52, 512^3 5.17 -> 5.42
//   periodic D3Q27 fp32 192^3 (0.76) 0.581 -> 0.527, D3Q19 bf16 256^3 (0.64) 0.681
//     -> 0.668, open D3Q19 384 x 128 x 128 fp32 (0.48) 0.421 -> 0.366, fp16 (0.24)
//     0.276 -> 0.262
// LBM_WALE_NT=0 or 1 overrides it (tuning); any choice gives the same values.
static bool wale_nt(int Q, size_t elem, const Dom& d) {
  if (const char* e = getenv("LBM_WALE_NT"))
    if (*e) return e[0] == '1';
  const size_t bytes = (size_t)Q * elem * d.N;
  return bytes > 230000000 && bytes < 1500000000;
}

template <int Q, typename S, bool NT>
static void local_n(const WaleFields& a, const ScalarStepArgs* sc, hipStream_t s) {
  const dim3 grid((a.d.N + 255) / 256), block(256);
  const ScalarStepArgs none{};
  if (sc)
    hipLaunchKernelGGL((k_wale_local<Q, S, false, 7, NT>), grid, block, 0, s, a, *sc);
  else if (a.d.per[0] || a.d.per[1] || a.d.per[2] || a.open)
    hipLaunchKernelGGL((k_wale_local<Q, S, true, 0, NT>), grid, block, 0, s, a, none);
  else
    hipLaunchKernelGGL((k_wale_local<Q, S, false, 0, NT>), grid, block, 0, s, a, none);
}

template <int Q, typename S>
static void local_q(const WaleFields& a, const ScalarStepArgs* sc, hipStream_t s) {
  wale_nt(Q, sizeof(S), a.d) ? local_n<Q, S, true>(a, sc, s) : local_n<Q, S, false>(a, sc, s);
}

hipError_t launch_wale_local(int Q, int storage, const WaleFields& a, const ScalarStepArgs* sc, hipStream_t s) {
  if (a.d.N == 0) return hipSuccess;
  if (storage == kF32)
    Q == 19 ? local_q<19, float>(a, sc, s) : local_q<27, float>(a, sc, s);
  else if (storage == kF16)
    Q == 19 ? local_q<19, _Float16>(a, sc, s) : local_q<27, _Float16>(a, sc, s);
  else
    Q == 19 ? local_q<19, bf16s>(a, sc, s) : local_q<27, bf16s>(a, sc, s);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_wale_solid(uint32_t n, const uint32_t* mask, float nu0, float* omega) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && (mask[i] & kMaskSolid)) omega[i] = wale_omega(nu0, 0.0f);
}

hipError_t launch_wale_solid(uint32_t n, const uint32_t* mask, float nu0, float* omega, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_wale_solid, dim3((n + 255) / 256), dim3(256), 0, s, n, mask, nu0, omega);
  return hipGetLastError();
}

__global__ void k_zero_u32(uint32_t* p, uint32_t n) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = 0u;
}

hipError_t launch_wale_omega(const WaleFields& a, float cw_delta_sq, float nu0, float nut_max, float* omega,
                             float* nut, uint32_t* stats, hipStream_t s) {
  if (a.d.N == 0) return hipSuccess;
  if (stats) {
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, stats, 2u);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const uint32_t zlen = wale_zlen(a.d);
  const dim3 tiles((a.d.nx + kWaleTileX - 1) / kWaleTileX, (a.d.ny + kWaleTileY - 1) / kWaleTileY,
                   (a.d.nz + zlen - 1) / zlen);
  hipLaunchKernelGGL(k_wale, tiles, dim3(256), 0, s, a, WaleOut{cw_delta_sq, nu0, nut_max, omega, nut, stats}, zlen);
  return hipGetLastError();
}

}  // namespace lbm
