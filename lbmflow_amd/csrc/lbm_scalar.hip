// lbm_scalar.hip — passive-scalar advection-diffusion distributions on the
// device (solver.rs:2113-2205, scalar.rs:6-15): BGK collide toward
// h_eq = w C (1 + c.u/cs^2) with the cached concentration and the post-step
// hydro velocity, streaming with half-way bounce-back at solids, C = sum h.
// The hydro lattice (reference) and D3Q7 (cs^2 = 1/4) are both supported.
//
// A step is one pass over the fluid cells: the cell's velocity from its
// populations, its Qs scalar populations in, the collided ones pushed into
// the other buffer.  That is what the step cannot do without (Q S + 4 bytes of
// populations and mask, 8 Qs of scalar); the concentration, which the next
// collide takes as the sum of what it reads anyway, is written once per call.
// The reference's form -- moments to memory, collide in place, pull stream
// with C -- moves 8 Qs + 36 bytes per cell more in two more passes.  Per step:
// 512^3 tank, fp16 populations, D3Q7 4.77 -> 2.51 ms (114 bytes per fluid cell
// at 3.9 TB/s); 128^3 the same 73 -> 33.5 us; 96^3 on D3Q19 fp32 61 -> 31 us.
#include <algorithm>
#include <cmath>

#include "lbm_aux.hpp"
#include "lbm_scalar.hpp"

namespace lbm {

namespace {
inline uint32_t nblk(size_t n, uint32_t bs = 256) { return (uint32_t)((n + bs - 1) / bs); }
}  // namespace

struct ScalarState {
  int Qs = 7;
  double D = 0.0;
  float omega = 1.0f;
  float* h = nullptr;
  float* h2 = nullptr;
  float* C = nullptr;
  size_t ps = 0;  // plane stride of h and h2
  double* partials = nullptr;
  uint32_t npartials = 1024;
  // C was given (set or restored) and is not the sum of h
  bool c_given = false;
  // C is older than h (inside a span)
  bool c_stale = false;
  // h2 holds the reference's ping-pong partner (the last step's
  // post-collision populations) rather than this path's older h
  bool partner = true;
  // solid cells of h / h2 may be nonzero; a step zeroes its target's
  bool dirty = false, dirty2 = false;
};

// What a kernel needs to take a cell's velocity (the moment readback's:
// moments_row with the force the state was made under).
struct VelArgs {
  Dom d;
  const void* f;
  const uint32_t* mask;
  const float* F_mom;
  HydroParams p;
  int odd;
  uint32_t deal;
};

template <int Q, typename S, int Qs, bool WRAP>
__global__ __launch_bounds__(256) void k_scalar_step(VelArgs a, ScalarStepArgs s) {
  const uint32_t i = xcd_remap(blockIdx.x, gridDim.x, a.deal) * 256 + threadIdx.x;
  if (i >= a.d.N) return;
  const uint32_t m = a.mask[i];
  if (m & kMaskSolid) return;
  uint32_t x = 0, y = 0, z = 0;
  if constexpr (WRAP) cell_xyz(a.d, i, x, y, z);
  const Nbr nb = WRAP ? Nbr(a.d, x, y, z) : Nbr(a.d);
  float hv[Qs], fv[Q];
  scalar_load<Qs>(s, i, hv);
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    fv[q] = read_pop<Q, S, q>((const S*)a.f, a.d.ps, nb, i, m, a.odd != 0);
  });
  // the field is zero off the force list, whose fluid cells carry kMaskForced
  float Fm[3] = {a.p.F[0], a.p.F[1], a.p.F[2]};
  bool fon = a.p.force_on != 0;
  if (a.F_mom && (m & kMaskForced)) {
    for (int c = 0; c < 3; ++c) Fm[c] = a.p.F[c] + a.F_mom[3 * (size_t)i + c];
    fon = true;
  }
  float r, ux, uy, uz;
  moments<Q>(fv, Fm, fon, r, ux, uy, uz);
  scalar_push<Qs>(s, nb, i, m, hv, ux, uy, uz);
}

template <int Qs>
__global__ __launch_bounds__(256) void k_scalar_set(Dom d, const float* conc, const float* mom, float* h, size_t ps,
                                                    float* C) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N) return;
  const float c = conc[i];
  const float ux = mom[d.N + i], uy = mom[2 * (size_t)d.N + i], uz = mom[3 * (size_t)d.N + i];
  C[i] = c;
  sfor<0, Qs>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    h[q * ps + i] = heq_q<Qs, q>(c, ux, uy, uz);
  });
}

// C = sum of h in direction order, 0 at solids
__global__ __launch_bounds__(256) void k_scalar_conc(Dom d, const uint32_t* mask, const float* h, size_t ps, int Qs,
                                                     float* C) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N) return;
  float c = 0.0f;
  if (!(mask[i] & kMaskSolid))
    for (int q = 0; q < Qs; ++q) c = c + h[q * ps + i];
  C[i] = c;
}

__global__ __launch_bounds__(256) void k_scalar_zero_solid(Dom d, const uint32_t* mask, float* h, size_t ps, int Qs) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N || !(mask[i] & kMaskSolid)) return;
  for (int q = 0; q < Qs; ++q) h[q * ps + i] = 0.0f;
}

// The reference's ping-pong partner after a step, its post-collision
// populations, from the streamed ones: h*_q(i) = h_q(i + c_q), or the
// reflected h_opp(q)(i) when i + c_q is solid (exact copies).  Solid cells of
// the partner keep what they hold.
template <int Qs>
__global__ __launch_bounds__(256) void k_scalar_partner(Dom d, const uint32_t* mask, const float* h, float* h2,
                                                        size_t ps) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.N) return;
  const uint32_t m = mask[i];
  if (m & kMaskSolid) return;
  uint32_t x, y, z;
  cell_xyz(d, i, x, y, z);
  const Nbr nb(d, x, y, z);
  sfor<0, Qs>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int o = lat_opp(q);
    const bool back = q != 0 && ((m >> o) & 1u);
    const uint32_t j = back ? i : i + (uint32_t)nb.template off<lat_c(q, 0), lat_c(q, 1), lat_c(q, 2)>();
    h2[q * ps + i] = h[(back ? o : q) * ps + j];
  });
}

// Two-pass CV over fluid cells (qoi::scalar_cv, qoi.rs:507-532), for the
// whole fluid (parts = 1) or the three compartments of compartment_cv
// (qoi.rs:699-739, parts = 3): a fluid cell of plane z is "top" when
// (z + 0.5)/nz >= 2/3, else "near_impeller" when an impeller height is given
// and |(z + 0.5) - z_imp| <= nz/6, else "bulk" (f64, the reference's
// expressions).  Pass 0 sums counts and values per compartment, pass 1 the
// squared deviations from the compartment means.  Per block: 6 doubles
// (count, sum per compartment; pass 1 fills the first 3 with the variances).
__global__ __launch_bounds__(256) void k_cv_pass(Dom d, const uint32_t* mask, const float* C, int pass, int parts,
                                                 int has_imp, double imp_z, double m0, double m1, double m2,
                                                 double* partials) {
  __shared__ double lds[4 * 6];
  double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  const double nz = (double)d.nz;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < d.N; i += gridDim.x * 256) {
    if (mask[i] & kMaskSolid) continue;
    int k = 0;
    if (parts == 3) {
      const double zc = (double)(i / (d.nx * d.ny)) + 0.5;
      if (zc / nz >= 2.0 / 3.0)
        k = 0;
      else if (has_imp && fabs(zc - imp_z) <= nz / 6.0)
        k = 2;
      else
        k = 1;
    }
    const double v = (double)C[i];
    if (pass == 0) {
      acc[2 * k] += 1.0;
      acc[2 * k + 1] += v;
    } else {
      const double dv = v - (k == 0 ? m0 : (k == 1 ? m1 : m2));
      acc[k] += dv * dv;
    }
  }
  block_sum256<6>(acc, lds);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < 6; ++k) partials[6 * blockIdx.x + k] = acc[k];
}

ScalarState* scalar_create(const FieldsView& v, double diffusivity, int Qs, std::string* err) {
  ScalarState* s = new ScalarState();
  s->Qs = Qs;
  s->D = diffusivity;
  // omega = T(1/(3D + 1/2)) on the hydro lattice (solver.rs:2131);
  // D3Q7 maps tau = D/cs^2 + 1/2 = 4D + 1/2.
  s->omega = Qs == 7 ? (float)(1.0 / (4.0 * diffusivity + 0.5)) : (float)(1.0 / (3.0 * diffusivity + 0.5));
  const size_t N = v.d.N;
  // planes an odd multiple of 256 elements apart, like the populations', so
  // that they do not all start in the same HBM channel
  s->ps = (N + 255) / 256 * 256;
  if (s->ps / 256 % 2 == 0) s->ps += 256;
  const size_t bytes = (size_t)Qs * s->ps * 4;
  hipError_t e = gpu_malloc(&s->h, bytes, v.rb);
  if (e == hipSuccess) e = gpu_malloc(&s->h2, bytes, v.rb);
  if (e == hipSuccess) e = gpu_malloc(&s->C, N * 4, v.rb);
  if (e == hipSuccess) e = gpu_malloc(&s->partials, 6 * s->npartials * sizeof(double), v.rb);
  if (e == hipSuccess) e = hipMemsetAsync(s->h, 0, bytes, v.stream);
  if (e == hipSuccess) e = hipMemsetAsync(s->h2, 0, bytes, v.stream);
  if (e == hipSuccess) e = hipMemsetAsync(s->C, 0, N * 4, v.stream);
  if (e != hipSuccess) {
    *err = std::string("scalar allocation failed: ") + hipGetErrorString(e);
    scalar_destroy(s);
    return nullptr;
  }
  return s;
}

void scalar_destroy(ScalarState* s) {
  if (!s) return;
  for (void* p : {(void*)s->h, (void*)s->h2, (void*)s->C, (void*)s->partials})
    if (p) (void)hipFree(p);
  delete s;
}

bool scalar_steady(const ScalarState* s) { return !s->c_given && !s->dirty && !s->dirty2; }

const void* scalar_current(const ScalarState* s) { return s->h; }

void scalar_replayed(ScalarState* s) {
  s->c_stale = true;
  s->partner = false;
}

int scalar_finish(const FieldsView& v, ScalarState* s) {
  if (!s->c_stale) return LBM_OK;
  hipLaunchKernelGGL(k_scalar_conc, dim3(nblk(v.d.N)), dim3(256), 0, v.stream, v.d, v.mask, s->h, s->ps, s->Qs, s->C);
  AUXCHK(v, hipGetLastError());
  s->c_stale = false;
  return LBM_OK;
}

static int restore_partner(const FieldsView& v, ScalarState* s) {
  if (s->partner) return LBM_OK;
  const dim3 g(nblk(v.d.N)), b(256);
  if (s->Qs == 7)
    hipLaunchKernelGGL((k_scalar_partner<7>), g, b, 0, v.stream, v.d, v.mask, s->h, s->h2, s->ps);
  else if (s->Qs == 19)
    hipLaunchKernelGGL((k_scalar_partner<19>), g, b, 0, v.stream, v.d, v.mask, s->h, s->h2, s->ps);
  else
    hipLaunchKernelGGL((k_scalar_partner<27>), g, b, 0, v.stream, v.d, v.mask, s->h, s->h2, s->ps);
  AUXCHK(v, hipGetLastError());
  s->partner = true;
  return LBM_OK;
}

int scalar_settle(const FieldsView& v, ScalarState* s) {
  int rc = scalar_finish(v, s);
  if (!rc) rc = restore_partner(v, s);
  if (rc) return rc;
  s->dirty = s->dirty2 = true;
  return LBM_OK;
}

int scalar_set(const FieldsView& v, ScalarState* s, const float* conc) {
  const size_t N = v.d.N;
  int rc = restore_partner(v, s);
  if (rc) return rc;
  float *dc = nullptr, *mom = nullptr;
  AUXCHK(v, gpu_malloc(&dc, N * 4, v.rb));
  hipError_t e = gpu_malloc(&mom, 4 * N * 4, v.rb);
  if (e == hipSuccess) e = hipMemcpyAsync(dc, conc, N * 4, hipMemcpyHostToDevice, v.stream);
  if (e == hipSuccess)
    e = launch_moments(v.Q, v.storage, v.parity, v.d, v.f, v.mask, v.F_mom, v.hp, 0, v.d.N, mom, mom + N,
                       mom + 2 * N, mom + 3 * N, v.stream);
  if (e == hipSuccess) {
    const dim3 g(nblk(N)), b(256);
    if (s->Qs == 7)
      hipLaunchKernelGGL((k_scalar_set<7>), g, b, 0, v.stream, v.d, dc, mom, s->h, s->ps, s->C);
    else if (s->Qs == 19)
      hipLaunchKernelGGL((k_scalar_set<19>), g, b, 0, v.stream, v.d, dc, mom, s->h, s->ps, s->C);
    else
      hipLaunchKernelGGL((k_scalar_set<27>), g, b, 0, v.stream, v.d, dc, mom, s->h, s->ps, s->C);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(v.stream);
  (void)hipFree(dc);
  if (mom) (void)hipFree(mom);
  AUXCHK(v, e);
  s->c_given = s->dirty = true;
  s->c_stale = false;
  return LBM_OK;
}

// checkpoint access: the distribution h (current), its ping-pong partner h2
// (after a step: the post-collision populations), the concentration, and
// the lattice size and diffusivity
int scalar_info(const ScalarState* s, int* Qs, double* D) {
  *Qs = s->Qs;
  *D = s->D;
  return LBM_OK;
}

int scalar_get_state(const FieldsView& v, ScalarState* s, float* h, float* h2, float* C) {
  const size_t w = (size_t)v.d.N * 4, pitch = s->ps * 4;
  int rc = scalar_finish(v, s);
  if (!rc) rc = restore_partner(v, s);
  if (rc) return rc;
  AUXCHK(v, hipMemcpy2DAsync(h, w, s->h, pitch, w, (size_t)s->Qs, hipMemcpyDeviceToHost, v.stream));
  AUXCHK(v, hipMemcpy2DAsync(h2, w, s->h2, pitch, w, (size_t)s->Qs, hipMemcpyDeviceToHost, v.stream));
  AUXCHK(v, hipMemcpyAsync(C, s->C, w, hipMemcpyDeviceToHost, v.stream));
  AUXCHK(v, hipStreamSynchronize(v.stream));
  return LBM_OK;
}

int scalar_put_state(const FieldsView& v, ScalarState* s, const float* h, const float* h2, const float* C) {
  const size_t w = (size_t)v.d.N * 4, pitch = s->ps * 4;
  AUXCHK(v, hipMemcpy2DAsync(s->h, pitch, h, w, w, (size_t)s->Qs, hipMemcpyHostToDevice, v.stream));
  AUXCHK(v, hipMemcpy2DAsync(s->h2, pitch, h2, w, w, (size_t)s->Qs, hipMemcpyHostToDevice, v.stream));
  AUXCHK(v, hipMemcpyAsync(s->C, C, w, hipMemcpyHostToDevice, v.stream));
  AUXCHK(v, hipStreamSynchronize(v.stream));
  s->c_given = s->partner = s->dirty = s->dirty2 = true;
  s->c_stale = false;
  return LBM_OK;
}

int scalar_gather(const FieldsView& v, ScalarState* s, float* conc) {
  int rc = scalar_finish(v, s);
  if (rc) return rc;
  const hipError_t read_back = v.rb->read(v.device, v.stream, 1, [&](int, std::vector<Readback::Seg>& segs) {
    segs.push_back({conc, s->C, (size_t)v.d.N * 4});
    return hipSuccess;
  });
  AUXCHK(v, read_back);
  return LBM_OK;
}

template <int Q, typename S, int Qs>
static void scalar_step_q(const VelArgs& a, const ScalarStepArgs& st, hipStream_t s) {
  const dim3 g(nblk(a.d.N)), b(256);
  if (a.d.per[0] || a.d.per[1] || a.d.per[2])
    hipLaunchKernelGGL((k_scalar_step<Q, S, Qs, true>), g, b, 0, s, a, st);
  else
    hipLaunchKernelGGL((k_scalar_step<Q, S, Qs, false>), g, b, 0, s, a, st);
}

template <typename S>
static void scalar_step_s(int Q, int Qs, const VelArgs& a, const ScalarStepArgs& st, hipStream_t s) {
  if (Q == 19 && Qs == 7) return scalar_step_q<19, S, 7>(a, st, s);
  if (Q == 19) return scalar_step_q<19, S, 19>(a, st, s);
  if (Qs == 7) return scalar_step_q<27, S, 7>(a, st, s);
  return scalar_step_q<27, S, 27>(a, st, s);
}

// This step's buffers and concentration; the state moves on to the next.
int scalar_turn(const FieldsView& v, ScalarState* s, ScalarStepArgs* st) {
  if (s->dirty2) {
    hipLaunchKernelGGL(k_scalar_zero_solid, dim3(nblk(v.d.N)), dim3(256), 0, v.stream, v.d, v.mask, s->h2, s->ps,
                       s->Qs);
    AUXCHK(v, hipGetLastError());
    s->dirty2 = false;
  }
  *st = ScalarStepArgs{s->h, s->h2, s->c_given ? s->C : nullptr, s->ps, s->omega};
  s->c_given = s->partner = false;
  s->c_stale = true;
  std::swap(s->h, s->h2);
  std::swap(s->dirty, s->dirty2);
  return LBM_OK;
}

int scalar_step(const FieldsView& v, ScalarState* s) {
  ScalarStepArgs st;
  int rc = scalar_turn(v, s, &st);
  if (rc) return rc;
  // One stretch per XCD while the last-level cache holds most of what the pass
  // reads, short runs beyond (xcd_remap).  Whole step of a closed cavity, stretch
  // -> dealt ms: D3Q7 144^3 fp16 D3Q27 (257 MB read) 0.144 -> 0.147, fp32 D3Q19
  // (322) 0.162 -> 0.167, 160^3 (352, 442) 0.214 -> 0.209 and 0.265 -> 0.253;
  // hydro lattice 128^3 (327, 348) 0.173 -> 0.178 and 0.216 -> 0.220, 144^3 (466,
  // 495) 0.276 -> 0.266 and 0.302 -> 0.292; 320^3 and more within 1 %.
  const size_t reads = ((size_t)v.Q * (v.storage == kF32 ? 4 : 2) + 4 + 4 * (size_t)s->Qs) * v.d.N;
  const VelArgs a{v.d, v.f, v.mask, v.F_mom, v.hp, v.parity, reads < 350000000 ? kXcdStretch : 5u};
  if (v.storage == kF32)
    scalar_step_s<float>(v.Q, s->Qs, a, st, v.stream);
  else if (v.storage == kF16)
    scalar_step_s<_Float16>(v.Q, s->Qs, a, st, v.stream);
  else
    scalar_step_s<bf16s>(v.Q, s->Qs, a, st, v.stream);
  AUXCHK(v, hipGetLastError());
  return LBM_OK;
}

// Both passes of k_cv_pass; results per compartment (parts = 1 or 3).
static int cv_parts(const FieldsView& v, ScalarState* s, int parts, int has_imp, double imp_z, double* cv,
                    int* defined, int64_t* counts) {
  int frc = scalar_finish(v, s);
  if (frc) return frc;
  const uint32_t np = std::min<uint32_t>(s->npartials, nblk(v.d.N));
  std::vector<double> h(6 * (size_t)np);
  auto run = [&](int pass, const double* mean) -> int {
    hipLaunchKernelGGL(k_cv_pass, dim3(np), dim3(256), 0, v.stream, v.d, v.mask, s->C, pass, parts, has_imp, imp_z,
                       mean[0], mean[1], mean[2], s->partials);
    AUXCHK(v, hipGetLastError());
    AUXCHK(v, hipMemcpyAsync(h.data(), s->partials, h.size() * sizeof(double), hipMemcpyDeviceToHost, v.stream));
    AUXCHK(v, hipStreamSynchronize(v.stream));
    return LBM_OK;
  };
  const double zero[3] = {0.0, 0.0, 0.0};
  int rc = run(0, zero);
  if (rc) return rc;
  double n[3] = {0, 0, 0}, sum[3] = {0, 0, 0}, mean[3] = {0, 0, 0};
  for (uint32_t b = 0; b < np; ++b)
    for (int k = 0; k < parts; ++k) {
      n[k] += h[6 * (size_t)b + 2 * k];
      sum[k] += h[6 * (size_t)b + 2 * k + 1];
    }
  bool any = false;
  for (int k = 0; k < parts; ++k) {
    counts[k] = (int64_t)n[k];
    defined[k] = 0;
    cv[k] = 0.0;
    if (n[k] == 0.0) continue;
    mean[k] = sum[k] / n[k];
    if (mean[k] == 0.0) continue;
    defined[k] = 1;
    any = true;
  }
  if (!any) return LBM_OK;
  rc = run(1, mean);
  if (rc) return rc;
  double var[3] = {0, 0, 0};
  for (uint32_t b = 0; b < np; ++b)
    for (int k = 0; k < parts; ++k) var[k] += h[6 * (size_t)b + k];
  for (int k = 0; k < parts; ++k)
    if (defined[k]) cv[k] = std::sqrt(var[k] / n[k]) / std::fabs(mean[k]);
  return LBM_OK;
}

int scalar_cv(const FieldsView& v, ScalarState* s, double* cv, int* defined) {
  int64_t count = 0;
  return cv_parts(v, s, 1, 0, 0.0, cv, defined, &count);
}

int scalar_compartment_cv(const FieldsView& v, ScalarState* s, int has_imp, double imp_z, double cv[3],
                          int defined[3], int64_t counts[3]) {
  return cv_parts(v, s, 3, has_imp, imp_z, cv, defined, counts);
}

}  // namespace lbm
