// lbm_adjoint.hip — reverse-mode (discrete adjoint) kernel of one D3Q19
// TRT/BGK collide-stream step with half-way bounce-back and Guo forcing.
//
// Forward map of one step at a fluid cell i (collision.rs:123-202 with the
// stale-moment force of solver.rs:2805-2822, stream_row kernels.rs:547-622):
//   rho = 1 + sum f,  m = sum c f,  u = (m + F_mom/2)/rho
//   feq_q = w_q (rho - 1 + rho (3 cu + 4.5 cu^2 - 1.5 u.u))
//   S_q   = w_q (3 (c_q.F - u.F) + 9 cu c_q.F)          (F = F_cur)
//   f*_q  = f_q - w+ (f+ - feq+) - w- (f- - feq-) + (1 - w+/2) S+ + (1 - w-/2) S-
//   f'_q(i) = f*_q(i - c_q), or f*_opp(q)(i) when i - c_q is solid.
// Forced cells (the force list) carry F_mom and F_cur; every other cell has
// no force.  w+ may vary per cell (omega field); w- is global.
//
// The kernel is the transposed Jacobian of that map at the forward state:
// given lam' (adjoint of f' at step n+1) it pulls lam* = adjoint of f*
// through the streaming (lam*_q(i) = lam'_q(i + c_q), or lam'_opp(q)(i)
// across a wall link) and returns the adjoint of f (lam), of w+ (added to
// omega_bar), of F_cur (Fbar) and of F_mom (Gout) at forced cells.  All
// adjoint arithmetic is f64; the forward state is the stored fp32 (or
// 16-bit) populations, read in the parity-dependent AA layout.
#include <algorithm>

#include "lbm_device.hpp"
#include "lbm_internal.hpp"

namespace lbm {

struct AdjArgs {
  Dom d;
  const void* f;
  const uint32_t* mask;
  const float* omega;  // per-cell omega_plus or null
  const float* F_cur;  // N x 3 or null
  const float* F_mom;  // N x 3 or null
  HydroParams p;
  const double* lam_in;  // Q x N: adjoint of the populations after the step
  double* lam_out;       // Q x N: adjoint of the populations before it
  double* omega_bar;     // N: accumulated adjoint of omega_plus
  double* Fbar;          // N x 3: adjoint of F_cur (forced cells; others untouched)
  double* Gout;          // N x 3: adjoint of F_mom (forced cells; others untouched)
  const uint32_t* flist;  // the force list (forced cells), or none
  uint32_t nlist;
  uint32_t deal;
};

// Bound by HBM: 2 x 152 bytes of adjoint populations, 76 of populations, 16 of
// omega_bar per fluid cell.  Per pair of opposite directions everything the
// transposed Jacobian needs of feq and S is a multiple of Lp = lam*_a + lam*_b
// and Lm = lam*_a - lam*_b, so the direct part, the feq and the S adjoints are
// never stored: what lives through the kernel is lam* (19 f64) and f (19 fp32).
// The form that held all three took 296 VGPRs, one wave per SIMD, and 240 us
// on the 128^3 tank; this one 168, three waves, and 155 us (0.53 GB, 3.4 TB/s).
// Solid cells are skipped and their adjoint is left undefined: what a fluid
// cell pulls from one is always replaced by its own reflected value.
// FORCED cells (those of the force list) take the source's terms as well, in a
// launch of their own over the list: in one kernel that rare branch sets the
// register count.
template <typename S, bool ODD, bool WRAP, bool FORCED>
__device__ __forceinline__ void adj_cell(const AdjArgs& a, uint32_t i, uint32_t m) {
  constexpr int Q = 19;
  const size_t N = a.d.N;
  uint32_t x = 0, y = 0, z = 0;
  if constexpr (WRAP) cell_xyz(a.d, i, x, y, z);
  const Nbr nb = WRAP ? Nbr(a.d, x, y, z) : Nbr(a.d);
  // forward state, and the adjoint of the post-collision populations pulled
  // through the streaming
  float f[Q];
  double ls[Q];
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    f[q] = read_pop<Q, S, q>((const S*)a.f, a.d.ps, nb, i, m, ODD);
  });
  // (plane bases are uniform, the per-lane part is one 32-bit byte offset:
  // lbm_adjoint_torque refuses domains whose f64 planes reach 4 GiB)
  const uint32_t at = i * 8u;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int cx = lat_c(q, 0), cy = lat_c(q, 1), cz = lat_c(q, 2);
    if constexpr (WRAP) {
      const uint32_t j = i + (uint32_t)nb.template off<cx, cy, cz>();
      ls[q] = a.lam_in[(size_t)q * N + j];
    } else {
      const int64_t shift = cx + cy * (int64_t)a.d.nx + cz * (int64_t)a.d.nx * a.d.ny;
      ls[q] = *(const double*)((const char*)(a.lam_in + (int64_t)(q * N) + shift) + at);
    }
  });
  if (m & kMaskLinks)  // reflected ones: i + c_q is solid
    sfor<1, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int o = lat_opp(q);
      if ((m >> o) & 1u) ls[q] = *(const double*)((const char*)(a.lam_in + o * N) + at);
    });
  double Fm[3] = {0.0, 0.0, 0.0}, Fc[3] = {0.0, 0.0, 0.0};
  if constexpr (FORCED)
    for (int c = 0; c < 3; ++c) {
      Fm[c] = (double)a.F_mom[3 * (size_t)i + c];
      Fc[c] = (double)a.F_cur[3 * (size_t)i + c];
    }
  const double op = a.omega ? (double)a.omega[i] : (double)a.p.omega_p;
  const double cp = 1.0 - 0.5 * op;
  const double om = (double)a.p.omega_m, cm = (double)a.p.cm;
  // moments
  double r = 1.0, u[3] = {0.0, 0.0, 0.0};
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const double fq = (double)f[q];
    r += fq;
    if constexpr (lat_c(q, 0) != 0) u[0] += (double)lat_c(q, 0) * fq;
    if constexpr (lat_c(q, 1) != 0) u[1] += (double)lat_c(q, 1) * fq;
    if constexpr (lat_c(q, 2) != 0) u[2] += (double)lat_c(q, 2) * fq;
  });
  for (int c = 0; c < 3; ++c) u[c] = (u[c] + 0.5 * Fm[c]) / r;
  const double usq = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
  const double uf = u[0] * Fc[0] + u[1] * Fc[1] + u[2] * Fc[2];
  // feq back to rho and u: with eb_a +- eb_b = op Lp, om Lm,
  //   rho: w (op Lp (1 + 4.5 cu^2 - 1.5 u.u) + om Lm 3 cu)
  //   u:   w r (op Lp (9 cu c - 3 u) + 3 om Lm c)
  const double w0 = (double)lat_wf(Q, 0);
  const double sym = 1.0 - 1.5 * usq;
  double rb = op * ls[0] * w0 * sym;
  double lpw = op * ls[0] * w0;  // sum w op Lp: the -3 u part of the u adjoint
  double ub[3] = {0.0, 0.0, 0.0};
  double obar = ls[0] * -((double)f[0] - w0 * (r - 1.0 - r * 1.5 * usq));
  sfor<0, (Q - 1) / 2>([&](auto kc) {
    constexpr int qa = 2 * decltype(kc)::value + 1;
    constexpr int qb = qa + 1;
    const double w = (double)lat_wf(Q, qa);
    double cu = 0.0;
    if constexpr (lat_c(qa, 0) != 0) cu += (double)lat_c(qa, 0) * u[0];
    if constexpr (lat_c(qa, 1) != 0) cu += (double)lat_c(qa, 1) * u[1];
    if constexpr (lat_c(qa, 2) != 0) cu += (double)lat_c(qa, 2) * u[2];
    const double Lp = ls[qa] + ls[qb];
    const double P = w * op * Lp, M = w * om * (ls[qa] - ls[qb]);
    const double cu2 = 4.5 * cu * cu;
    rb += P * (sym + cu2) + M * (3.0 * cu);
    lpw += P;
    const double t = P * (9.0 * cu) + 3.0 * M;
    if constexpr (lat_c(qa, 0) != 0) ub[0] += (double)lat_c(qa, 0) * t;
    if constexpr (lat_c(qa, 1) != 0) ub[1] += (double)lat_c(qa, 1) * t;
    if constexpr (lat_c(qa, 2) != 0) ub[2] += (double)lat_c(qa, 2) * t;
    const double ep = w * (r - 1.0 + r * (cu2 - 1.5 * usq));
    obar -= Lp * (0.5 * ((double)f[qa] + (double)f[qb]) - ep);
  });
  for (int c = 0; c < 3; ++c) ub[c] = r * (ub[c] - 3.0 * lpw * u[c]);
  // Each phase recomputes its pair sums from lam*: kept from one phase to the
  // next (as the compiler would) they cost 54 registers.
  auto fresh = [](double* v) {
#pragma unroll
    for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(v[q]));
  };
  fresh(ls);
  if constexpr (FORCED) {
    // the source back to u and F_cur, and its share of omega_bar: with
    // sb_a +- sb_b = cp Lp, cm Lm
    double fcb[3] = {0.0, 0.0, 0.0};
    const double s0 = cp * ls[0] * w0;
    obar += ls[0] * -0.5 * (w0 * (-3.0 * uf));
    for (int c = 0; c < 3; ++c) {
      ub[c] += -3.0 * s0 * Fc[c];
      fcb[c] += -3.0 * s0 * u[c];
    }
    sfor<0, (Q - 1) / 2>([&](auto kc) {
      constexpr int qa = 2 * decltype(kc)::value + 1;
      constexpr int qb = qa + 1;
      const double w = (double)lat_wf(Q, qa);
      const double c3[3] = {(double)lat_c(qa, 0), (double)lat_c(qa, 1), (double)lat_c(qa, 2)};
      const double cu = c3[0] * u[0] + c3[1] * u[1] + c3[2] * u[2];
      const double cf = c3[0] * Fc[0] + c3[1] * Fc[1] + c3[2] * Fc[2];
      const double Lp = ls[qa] + ls[qb];
      const double P = w * cp * Lp, M = w * cm * (ls[qa] - ls[qb]);
      for (int c = 0; c < 3; ++c) {
        ub[c] += P * (-3.0 * Fc[c] + 9.0 * c3[c] * cf);
        fcb[c] += P * (-3.0 * u[c] + 9.0 * cu * c3[c]) + 3.0 * M * c3[c];
      }
      obar -= 0.5 * Lp * (w * (-3.0 * uf + 9.0 * cu * cf));
    });
    for (int c = 0; c < 3; ++c) {
      a.Fbar[3 * (size_t)i + c] = fcb[c];
      a.Gout[3 * (size_t)i + c] = ub[c] / (2.0 * r);
    }
  }
  // u = (m + F_mom/2)/rho
  double mb[3];
  for (int c = 0; c < 3; ++c) {
    mb[c] = ub[c] / r;
    rb += -ub[c] * u[c] / r;
  }
  fresh(ls);
  auto out = [&](int q) { return (double*)((char*)(a.lam_out + (size_t)q * N) + at); };
  *out(0) = ls[0] * (1.0 - op) + rb;
  sfor<0, (Q - 1) / 2>([&](auto kc) {
    constexpr int qa = 2 * decltype(kc)::value + 1;
    constexpr int qb = qa + 1;
    const double ep = 0.5 * op * (ls[qa] + ls[qb]), em = 0.5 * om * (ls[qa] - ls[qb]);
    double cmb = 0.0;
    if constexpr (lat_c(qa, 0) != 0) cmb += (double)lat_c(qa, 0) * mb[0];
    if constexpr (lat_c(qa, 1) != 0) cmb += (double)lat_c(qa, 1) * mb[1];
    if constexpr (lat_c(qa, 2) != 0) cmb += (double)lat_c(qa, 2) * mb[2];
    *out(qa) = ls[qa] - ep - em + rb + cmb;
    *out(qb) = ls[qb] - ep + em + rb - cmb;
  });
  a.omega_bar[i] += obar;
}

template <typename S, bool ODD, bool WRAP>
__global__ __launch_bounds__(256, 3) void k_adj_collide_stream(AdjArgs a) {
  const uint32_t i = xcd_remap(blockIdx.x, gridDim.x, a.deal) * 256 + threadIdx.x;
  if (i >= a.d.N) return;
  const uint32_t m = a.mask[i];
  if ((m & kMaskSolid) || (a.nlist && (m & kMaskForced))) return;
  adj_cell<S, ODD, WRAP, false>(a, i, m);
}

template <typename S, bool ODD>
__global__ __launch_bounds__(64) void k_adj_list(AdjArgs a) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.nlist) return;
  const uint32_t i = a.flist[k];
  const uint32_t m = a.mask[i];
  if (!(m & kMaskSolid)) adj_cell<S, ODD, true, true>(a, i, m);
}

template <typename S>
static hipError_t adj_s(int odd, const AdjArgs& a, hipStream_t s) {
  const dim3 grid((a.d.N + 255) / 256), block(256);
  const bool wrap = a.d.per[0] || a.d.per[1] || a.d.per[2];
  if (odd && wrap)
    hipLaunchKernelGGL((k_adj_collide_stream<S, true, true>), grid, block, 0, s, a);
  else if (odd)
    hipLaunchKernelGGL((k_adj_collide_stream<S, true, false>), grid, block, 0, s, a);
  else if (wrap)
    hipLaunchKernelGGL((k_adj_collide_stream<S, false, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((k_adj_collide_stream<S, false, false>), grid, block, 0, s, a);
  if (a.nlist) {
    const dim3 lg((a.nlist + 63) / 64), lb(64);
    if (odd)
      hipLaunchKernelGGL((k_adj_list<S, true>), lg, lb, 0, s, a);
    else
      hipLaunchKernelGGL((k_adj_list<S, false>), lg, lb, 0, s, a);
  }
  return hipGetLastError();
}

hipError_t launch_adj_collide_stream(int storage, int odd, const Dom& d, const void* f, const uint32_t* mask,
                                     const float* omega, const float* F_cur, const float* F_mom,
                                     const HydroParams& p, const uint32_t* flist, uint32_t nlist, const double* lam_in,
                                     double* lam_out, double* omega_bar, double* Fbar, double* Gout,
                                     hipStream_t s) {
  // One stretch per XCD below 1 GB of the pass's bytes (about 400 per cell),
  // short runs above (xcd_remap).  us per pass of a tank, stretch -> dealt, medians
  // of four processes: 96^3 64.2 -> 63.5, 112^3 104.3 -> 107.0, 128^3 (0.84 GB) 155
  // -> 165, 144^3 (1.19 GB) 223.5 -> 218.4, 160^3 301 -> 292, 192^3 499 -> 483,
  // 224^3 777 -> 753, 256^3 1132 -> 1157 (1130 +- 30 either way).
  const uint32_t deal = (size_t)d.N * 400 < 1000000000 ? kXcdStretch : 5u;
  AdjArgs a{d, f, mask, omega, F_cur, F_mom, p, lam_in, lam_out, omega_bar, Fbar, Gout,
            flist, F_cur && F_mom ? nlist : 0u, deal};
  if (storage == kF32) return adj_s<float>(odd, a, s);
  if (storage == kF16) return adj_s<_Float16>(odd, a, s);
  return adj_s<bf16s>(odd, a, s);
}

// dJ/dnu from the adjoint of omega_plus = 1 / (3 nu + 1/2): times -3 omega_plus^2
__global__ void k_nu_bar(uint32_t n, const double* omega_bar, const float* omega, float omega_p, double* out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double op = omega ? (double)omega[i] : (double)omega_p;
  out[i] = omega_bar[i] * (-3.0 * op * op);
}

// the listed cells' vec3 of F into buf (dir 0) or back (dir 1)
__global__ void k_list_pack(const uint32_t* flist, uint32_t n, float* F, float* buf, int dir) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const size_t i = flist[k];
  for (int c = 0; c < 3; ++c) {
    if (dir == 0)
      buf[3 * (size_t)k + c] = F[3 * i + c];
    else
      F[3 * i + c] = buf[3 * (size_t)k + c];
  }
}

hipError_t launch_list_pack(const uint32_t* flist, uint32_t n, float* F, float* buf, int dir, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_list_pack, dim3((n + 255) / 256), dim3(256), 0, s, flist, n, F, buf, dir);
  return hipGetLastError();
}

hipError_t launch_nu_bar(uint32_t n, const double* omega_bar, const float* omega, float omega_p, double* out,
                         hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_nu_bar, dim3((n + 255) / 256), dim3(256), 0, s, n, omega_bar, omega, omega_p, out);
  return hipGetLastError();
}

__global__ void k_fill_d(double* p, size_t n, double v) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) p[k] = v;
}

hipError_t launch_fill_f64(double* p, size_t n, double v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  // one work-item per double would pass the 2^32 work-items a launch may have
  // from 148 M cells on (29 doubles per cell are zeroed at once)
  const size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_fill_d, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

}  // namespace lbm
