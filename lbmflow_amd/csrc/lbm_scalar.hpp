// lbm_scalar.hpp — one cell's passive-scalar step, inlined by the kernels
// that have the cell's velocity in registers (lbm_scalar.hip, lbm_les.hip).
#pragma once
#include "lbm_device.hpp"

namespace lbm {

// h_eq of scalar_equilibrium (scalar.rs:6-15) for the hydro lattice; the
// D3Q7 form uses 1/cs^2 = 4.
template <int Qs, int q>
__device__ __forceinline__ float heq_q(float conc, float ux, float uy, float uz) {
  const float cu = cdot<q>(ux, uy, uz);
  constexpr float k = Qs == 7 ? 4.0f : 3.0f;
  return lat_wf(Qs, q) * conc * (1.0f + k * cu);
}

template <int Qs>
__device__ __forceinline__ void scalar_load(const ScalarStepArgs& s, uint32_t i, float* hv) {
  sfor<0, Qs>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    hv[q] = s.h[q * s.ps + i];
  });
}

// Collide and push of fluid cell i (mask word m) with velocity u.  The
// concentration is the sum of h in direction order, the value the previous
// step's stream would have stored.  A population heading into a solid comes
// back into the cell's own opposite slot, every other one goes to cell
// i + c_q, so each slot of a fluid cell has exactly one writer and a solid
// cell's slots none.
template <int Qs>
__device__ __forceinline__ void scalar_push(const ScalarStepArgs& s, const Nbr& nb, uint32_t i, uint32_t m,
                                            const float* hv, float ux, float uy, float uz) {
  float c = 0.0f;
  if (s.C)
    c = s.C[i];
  else
    sfor<0, Qs>([&](auto qc) { c = c + hv[decltype(qc)::value]; });
  sfor<0, Qs>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int o = lat_opp(q);
    const float v = hv[q] - s.omega * (hv[q] - heq_q<Qs, q>(c, ux, uy, uz));
    const bool back = q != 0 && ((m >> o) & 1u);
    const uint32_t j = back ? i : i + (uint32_t)nb.template off<lat_c(q, 0), lat_c(q, 1), lat_c(q, 2)>();
    s.h2[(back ? o : q) * s.ps + j] = v;
  });
}

}  // namespace lbm
