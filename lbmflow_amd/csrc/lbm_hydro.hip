// lbm_hydro.hip — CDNA4 (gfx950) fused in-place (AA-pattern) collide-stream
// kernels: TRT/BGK and the factorised central-moment collision, half-way
// bounce-back, moving walls, Guo forcing, for one domain or a batch.
//
// The file is compiled once per lattice, population storage and collision
// (LBM_Q = 19 | 27, LBM_STORAGE = 0 f32 | 1 f16 | 2 bf16, LBM_KIND = 0 TRT/BGK |
// 1 central moments), so the twelve object files build in parallel;
// lbm_kernels.hip selects among them at launch.
//
// Storage: q-major planes f[q*ps + cell] of the deviation f - w_q in fp32,
// or scaled by 1/w_q in fp16 / bf16.  Arithmetic is fp32.  Reductions are
// fp64.  The whole file is compiled with -ffp-contract=off so the TRT path
// keeps the reference's separately rounded multiply/add sequence
// (collision.rs:123-202) and reproduces the CpuScalar f32 trajectory
// bit for bit; the central-moment path opts into contraction locally, per
// source expression (contract(on)), so every kernel that inlines it rounds
// identically (the batched launch reproduces the single-domain one).
//
// AA pattern (in-place streaming, one buffer):
//   even step  cell i reads f_q from slot (i, q), writes the post-collision
//              value moving along c_q to slot (i, opp q);
//   odd step   cell i reads f_q from slot (i - c_q, opp q), writes the value
//              moving along c_q to slot (i + c_q, q).
// A post-collision population heading into a solid neighbour s = i + c_q is
// reflected immediately: on even steps it is written to the solid's slot
// (s, q) -- where the odd step's uniform read of i looks for the incoming
// opp(q) population -- and on odd steps to (i, opp q), where the next even
// step reads it.  Each slot is read and written by exactly one cell per
// step, so cells are independent and no second buffer is needed.
#include <type_traits>

#include "lbm_device.hpp"
#include "lbm_wale.hpp"

namespace lbm {

// ---------------------------------------------------------------------------
// TRT/BGK with Guo forcing: TrtGuo::relax (collision.rs:123-202) with the
// equilibrium of SecondOrderEq::feq (81-102) and GuoForcing::source
// (104-121).  Same operand order, no contraction.
// ---------------------------------------------------------------------------
template <int Q, bool HALVE>
__device__ __forceinline__ void collide_trt(float* fv, float r, float ux, float uy, float uz, const float Fc[3],
                                            bool fon, float op, float cp, const HydroParams& p) {
  float usq = ux * ux;
  usq = usq + uy * uy;
  usq = usq + uz * uz;
  float uf = 0.0f;
  if (fon) {
    uf = ux * Fc[0];
    uf = uf + uy * Fc[1];
    uf = uf + uz * Fc[2];
  }
  const float drho = r - 1.0f;
  const float f15_usq = 1.5f * usq;
  // rest population
  {
    constexpr float w0 = lat_wf(Q, 0);
    const float cu0 = 0.0f * ux;  // cu of the rest velocity is a signed zero
    const float feq0 = w0 * (drho + r * ((3.0f * cu0 + (4.5f * cu0) * cu0) - f15_usq));
    float f0 = fv[0];
    float relaxed = f0 - op * (f0 - feq0);
    if (fon) {
      const float src0 = w0 * (3.0f * (0.0f - uf) + (9.0f * cu0) * 0.0f);
      relaxed = relaxed + cp * src0;
    }
    fv[0] = relaxed;
  }
  // Pairs (q, q+1), q odd, ascending (lattice.rs PAIRS).  Every value is the
  // reference's: cu of the opposite direction is -cu, so the even products are
  // shared and the odd ones change sign.  HALVE (fp32 storage) halves the pair
  // sums where the reference does; without it the factor 1/2 goes into the
  // rates, op (f+ - feq+) = (op/2) ((f_a + f_b) - (e_a + e_b)), the same bits
  // short of the denormal range, which a front running into fluid at rest does
  // reach in fp32.  VALU instructions per wave, D3Q19 fp32 486 -> 462, D3Q27
  // bf16 with force 1158 -> 1000, which is time where 16-bit storage is
  // VALU-bound (201 x 147 x 173 periodic D3Q27 bf16 with a force, even / odd:
  // 0.189 / 0.221 -> 0.170 / 0.199 ms with the hardware's bf16 rounding).
  const float hop = HALVE ? op : 0.5f * op, hom = HALVE ? p.omega_m : 0.5f * p.omega_m;
  const float hcp = HALVE ? cp : 0.5f * cp, hcm = HALVE ? p.cm : 0.5f * p.cm;
  auto halve = [](float v) { return HALVE ? 0.5f * v : v; };
  sfor<0, (Q - 1) / 2>([&](auto kc) {
    constexpr int qa = 2 * decltype(kc)::value + 1;
    constexpr int qb = qa + 1;
    constexpr float w = lat_wf(Q, qa);
    const float cu = cdot<qa>(ux, uy, uz);
    const float three_cu = 3.0f * cu;
    const float f45_cu2 = (4.5f * cu) * cu;
    const float ea = w * (drho + r * ((f45_cu2 + three_cu) - f15_usq));
    const float eb = w * (drho + r * ((f45_cu2 - three_cu) - f15_usq));
    const float fa = fv[qa], fb = fv[qb];
    const float rp = hop * (halve(fa + fb) - halve(ea + eb));
    const float rm = hom * (halve(fa - fb) - halve(ea - eb));
    float va = (fa - rp) - rm;
    float vb = (fb - rp) + rm;
    if (fon) {
      const float cf = cdot<qa>(Fc[0], Fc[1], Fc[2]);
      const float second = (9.0f * cu) * cf;
      const float sa = w * (3.0f * (cf - uf) + second);
      const float sb = w * (3.0f * (-cf - uf) + second);
      const float cp_sp = hcp * halve(sa + sb);
      const float cm_sm = hcm * halve(sa - sb);
      va = va + (cp_sp + cm_sm);
      vb = vb + (cp_sp - cm_sm);
    }
    fv[qa] = va;
    fv[qb] = vb;
  });
}

// ---------------------------------------------------------------------------
// Central-moment collision (collide_row_central_moment, kernels.rs:406-533)
// in non-equilibrium form.  With feq the deviation equilibrium and
// K = central moments of (f - feq), S = central moments of the Guo source,
// the reference's post-collision populations are feq + B(d), where B is the
// inverse central-moment transform and
//   order 0,1:       d = K + S
//   order 2, a!=b:   d = (1-os) K + (1-os/2) S
//   order 2, a==b:   d = (1-os)(K_aa - K_bulk) + S_bulk/2 + (1-os/2)(S_aa - S_bulk)
//   order >= 3:      d = S/2
// (the reference relaxes the trace and all orders >= 3 at rate 1).  The
// D3Q27 transforms factorise into three passes of 1-D three-point lines
// (tensor-product basis, exponents 0..2 per axis), so no 27x27 matrix
// is ever formed.  Working on f - feq keeps the fp32 arithmetic on small
// numbers; the rounding difference to the reference's f64 internals stays
// well below the 1e-6 population gate.
// ---------------------------------------------------------------------------
constexpr int gidx(int cx, int cy, int cz) { return (cx + 1) * 9 + (cy + 1) * 3 + (cz + 1); }

// forward 1-D central line: (g-, g0, g+) -> (k0, k1, k2)
__device__ __forceinline__ void fwd_line(float& a0, float& a1, float& a2, float u) {
#pragma clang fp contract(on)
  const float gm = a0, g0 = a1, gp = a2;
  const float s = gp + gm, t = gp - gm;
  const float k0 = s + g0;
  const float k1 = t - u * k0;
  const float k2 = (s - 2.0f * u * t) + u * u * k0;
  a0 = k0;
  a1 = k1;
  a2 = k2;
}
// inverse 1-D central line: (k0, k1, k2) -> (g-, g0, g+)
__device__ __forceinline__ void inv_line(float& a0, float& a1, float& a2, float u) {
#pragma clang fp contract(on)
  const float k0 = a0, k1 = a1, k2 = a2;
  const float m1 = k1 + u * k0;
  const float m2 = (k2 + 2.0f * u * k1) + u * u * k0;
  a0 = 0.5f * (m2 - m1);
  a1 = k0 - m2;
  a2 = 0.5f * (m1 + m2);
}

// Full 27-point transforms on G[(a*9 + b*3 + c)], a/b/c = x/y/z index 0..2.
__device__ __forceinline__ void fwd27(float* G, float ux, float uy, float uz) {
#pragma unroll
  for (int ab = 0; ab < 9; ++ab) fwd_line(G[ab * 3 + 0], G[ab * 3 + 1], G[ab * 3 + 2], uz);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int c = 0; c < 3; ++c) fwd_line(G[a * 9 + 0 + c], G[a * 9 + 3 + c], G[a * 9 + 6 + c], uy);
#pragma unroll
  for (int bc = 0; bc < 9; ++bc) fwd_line(G[bc], G[9 + bc], G[18 + bc], ux);
}
__device__ __forceinline__ void inv27(float* G, float ux, float uy, float uz) {
#pragma unroll
  for (int bc = 0; bc < 9; ++bc) inv_line(G[bc], G[9 + bc], G[18 + bc], ux);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int c = 0; c < 3; ++c) inv_line(G[a * 9 + 0 + c], G[a * 9 + 3 + c], G[a * 9 + 6 + c], uy);
#pragma unroll
  for (int ab = 0; ab < 9; ++ab) inv_line(G[ab * 3 + 0], G[ab * 3 + 1], G[ab * 3 + 2], uz);
}

// deviation equilibrium of all 27 directions (same formula as the TRT
// path, here with contraction allowed)
__device__ __forceinline__ void feq27(float* feq, float r, float ux, float uy, float uz) {
#pragma clang fp contract(on)
  const float usq = ux * ux + uy * uy + uz * uz;
  const float drho = r - 1.0f;
  const float b = drho - r * 1.5f * usq;
  sfor<0, 27>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const float cu = cdot<q>(ux, uy, uz);
    feq[q] = lat_wf(27, q) * (b + r * cu * (3.0f + 4.5f * cu));
  });
}

__device__ __forceinline__ float cm_rate(float os_base, float ux, float uy, float uz) {
#pragma clang fp contract(on)
  const float usq = ux * ux + uy * uy + uz * uz;
  return fminf(os_base * (1.0f - 0.16f * usq), 2.0f);
}

// General form (any force): full transforms of f - feq and of the source.
__device__ __forceinline__ void collide_cm27_general(float* fv, float r, float ux, float uy, float uz,
                                                     const float F[3], bool fon, float os_base) {
#pragma clang fp contract(on)
  float feq[27];
  feq27(feq, r, ux, uy, uz);
  float K[27], S[27];
  sfor<0, 27>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int g = gidx(lat_c(q, 0), lat_c(q, 1), lat_c(q, 2));
    K[g] = fv[q] - feq[q];
  });
  fwd27(K, ux, uy, uz);
  if (fon) {
    const float uf = ux * F[0] + uy * F[1] + uz * F[2];
    sfor<0, 27>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int g = gidx(lat_c(q, 0), lat_c(q, 1), lat_c(q, 2));
      const float cu = cdot<q>(ux, uy, uz);
      const float cf = cdot<q>(F[0], F[1], F[2]);
      S[g] = lat_wf(27, q) * (3.0f * (cf - uf) + 9.0f * cu * cf);
    });
    fwd27(S, ux, uy, uz);
  } else {
#pragma unroll
    for (int g = 0; g < 27; ++g) S[g] = 0.0f;
  }
  const float os = cm_rate(os_base, ux, uy, uz);
  const float a1 = 1.0f - os, a2 = 1.0f - 0.5f * os;
  const int ixx = 2 * 9, iyy = 2 * 3, izz = 2;
  const float kb = (K[ixx] + K[iyy] + K[izz]) * (1.0f / 3.0f);
  const float sb = (S[ixx] + S[iyy] + S[izz]) * (1.0f / 3.0f);
  float D[27];
#pragma unroll
  for (int g = 0; g < 27; ++g) {
    const int ex = g / 9, ey = (g / 3) % 3, ez = g % 3;
    const int order = ex + ey + ez;
    if (order <= 1)
      D[g] = K[g] + S[g];
    else if (order == 2 && (ex == 2 || ey == 2 || ez == 2))
      D[g] = a1 * (K[g] - kb) + 0.5f * sb + a2 * (S[g] - sb);
    else if (order == 2)
      D[g] = a1 * K[g] + a2 * S[g];
    else
      D[g] = 0.5f * S[g];
  }
  inv27(D, ux, uy, uz);
  sfor<0, 27>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int g = gidx(lat_c(q, 0), lat_c(q, 1), lat_c(q, 2));
    fv[q] = feq[q] + D[g];
  });
}

// D3Q19 central moments.  The basis is the reference's (central_basis,
// kernels.rs:162-183): exponents (ex, ey, ez) in {0,1,2}^3, x outermost,
// without the eight with all three positive.  It is not a tensor product, so
// the transforms are the raw-moment matrix R (entries c^e in {-1, 0, 1}),
// the binomial shift by -u / +u (kernels.rs:332-370) and the inverse
// P = R^-1, whose entries (0, +-1/4, +-1/2, +-1) are exact in fp32.  All three
// are compile-time tables; zero terms vanish when the loops unroll.
struct Cm19Tables {
  int e[19][3];
  int idx[3][3][3];  // exponent -> moment, -1 when not in the basis
  double P[19][19];
};

constexpr int cm19_phi(int q, int m, const Cm19Tables& t) {
  int v = 1;
  for (int a = 0; a < 3; ++a)
    for (int k = 0; k < t.e[m][a]; ++k) v *= lat_c(q, a);
  return v;
}

constexpr Cm19Tables make_cm19() {
  Cm19Tables t{};
  for (int a = 0; a < 3; ++a)
    for (int b = 0; b < 3; ++b)
      for (int c = 0; c < 3; ++c) t.idx[a][b][c] = -1;
  int n = 0;
  for (int ax = 0; ax <= 2; ++ax)
    for (int ay = 0; ay <= 2; ++ay)
      for (int az = 0; az <= 2; ++az) {
        if (ax > 0 && ay > 0 && az > 0) continue;
        t.e[n][0] = ax;
        t.e[n][1] = ay;
        t.e[n][2] = az;
        t.idx[ax][ay][az] = n;
        ++n;
      }
  // Gauss-Jordan inverse of R (partial pivoting), exact here: R is integer
  // with a power-of-two-denominator inverse
  double A[19][38] = {};
  for (int m = 0; m < 19; ++m) {
    for (int q = 0; q < 19; ++q) A[m][q] = cm19_phi(q, m, t);
    A[m][19 + m] = 1.0;
  }
  for (int col = 0; col < 19; ++col) {
    int piv = col;
    for (int r = col + 1; r < 19; ++r)
      if ((A[r][col] < 0 ? -A[r][col] : A[r][col]) > (A[piv][col] < 0 ? -A[piv][col] : A[piv][col])) piv = r;
    for (int j = 0; j < 38; ++j) {
      const double tmp = A[col][j];
      A[col][j] = A[piv][j];
      A[piv][j] = tmp;
    }
    const double inv = 1.0 / A[col][col];
    for (int j = 0; j < 38; ++j) A[col][j] *= inv;
    for (int r = 0; r < 19; ++r) {
      if (r == col || A[r][col] == 0.0) continue;
      const double f = A[r][col];
      for (int j = 0; j < 38; ++j) A[r][j] -= f * A[col][j];
    }
  }
  for (int q = 0; q < 19; ++q)
    for (int m = 0; m < 19; ++m) t.P[q][m] = A[q][19 + m];
  return t;
}
inline constexpr Cm19Tables kCm19 = make_cm19();

constexpr int binom2(int n, int k) { return (k == 0 || k == n) ? 1 : 2; }  // n <= 2

// u^k for k in 0..2
__device__ __forceinline__ float pow2u(float u, int k) { return k == 0 ? 1.0f : (k == 1 ? u : u * u); }

// central moments (shift by -u) of the raw moments R, or raw moments (shift
// by +u) of central moments: out[m] = sum_{k <= e_m} C(e,k) s^(e-k) in[idx(k)]
template <bool TO_CENTRAL>
__device__ __forceinline__ void cm19_shift(const float* in, float* out, float ux, float uy, float uz) {
#pragma clang fp contract(on)
  const float sx = TO_CENTRAL ? -ux : ux, sy = TO_CENTRAL ? -uy : uy, sz = TO_CENTRAL ? -uz : uz;
  sfor<0, 19>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    constexpr int ex = kCm19.e[m][0], ey = kCm19.e[m][1], ez = kCm19.e[m][2];
    float acc = in[m];  // k = e: coefficient 1
    sfor<0, (ex + 1) * (ey + 1) * (ez + 1)>([&](auto kc) {
      constexpr int kk = decltype(kc)::value;
      constexpr int kx = kk / ((ey + 1) * (ez + 1)), ky = (kk / (ez + 1)) % (ey + 1), kz = kk % (ez + 1);
      if constexpr (!(kx == ex && ky == ey && kz == ez)) {
        constexpr int j = kCm19.idx[kx][ky][kz];
        constexpr float coef = (float)(binom2(ex, kx) * binom2(ey, ky) * binom2(ez, kz));
        acc = acc + coef * (pow2u(sx, ex - kx) * pow2u(sy, ey - ky) * pow2u(sz, ez - kz)) * in[j];
      }
    });
    out[m] = acc;
  });
}

// raw moments of a population vector: R[m] = sum_q c_q^e_m v_q
__device__ __forceinline__ void cm19_raw(const float* v, float* R) {
  sfor<0, 19>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    float acc = 0.0f;
    sfor<0, 19>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int c = cm19_phi(q, m, kCm19);
      if constexpr (c == 1) acc = acc + v[q];
      if constexpr (c == -1) acc = acc - v[q];
    });
    R[m] = acc;
  });
}

// D3Q19 central-moment collision, general form (any force): feq + B(d) as
// for D3Q27, with the matrix transforms above.
__device__ __forceinline__ void collide_cm19_general(float* fv, float r, float ux, float uy, float uz,
                                                     const float F[3], bool fon, float os_base) {
#pragma clang fp contract(on)
  const float usq = ux * ux + uy * uy + uz * uz;
  const float b = (r - 1.0f) - r * 1.5f * usq;
  float feq[19], G[19], K[19], Sm[19];
  sfor<0, 19>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const float cu = cdot<q>(ux, uy, uz);
    feq[q] = lat_wf(19, q) * (b + r * cu * (3.0f + 4.5f * cu));
    G[q] = fv[q] - feq[q];
  });
  cm19_raw(G, Sm);
  cm19_shift<true>(Sm, K, ux, uy, uz);
  if (fon) {
    const float uf = ux * F[0] + uy * F[1] + uz * F[2];
    sfor<0, 19>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      const float cu = cdot<q>(ux, uy, uz);
      const float cf = cdot<q>(F[0], F[1], F[2]);
      G[q] = lat_wf(19, q) * (3.0f * (cf - uf) + 9.0f * cu * cf);
    });
    float Rs[19];
    cm19_raw(G, Rs);
    cm19_shift<true>(Rs, Sm, ux, uy, uz);
  } else {
#pragma unroll
    for (int m = 0; m < 19; ++m) Sm[m] = 0.0f;
  }
  const float os = cm_rate(os_base, ux, uy, uz);
  const float a1 = 1.0f - os, a2 = 1.0f - 0.5f * os;
  constexpr int ixx = kCm19.idx[2][0][0], iyy = kCm19.idx[0][2][0], izz = kCm19.idx[0][0][2];
  const float kb = (K[ixx] + K[iyy] + K[izz]) * (1.0f / 3.0f);
  const float sb = (Sm[ixx] + Sm[iyy] + Sm[izz]) * (1.0f / 3.0f);
  float D[19];
  sfor<0, 19>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    constexpr int ex = kCm19.e[m][0], ey = kCm19.e[m][1], ez = kCm19.e[m][2];
    constexpr int order = ex + ey + ez;
    if constexpr (order <= 1)
      D[m] = K[m] + Sm[m];
    else if constexpr (order == 2 && (ex == 2 || ey == 2 || ez == 2))
      D[m] = a1 * (K[m] - kb) + 0.5f * sb + a2 * (Sm[m] - sb);
    else if constexpr (order == 2)
      D[m] = a1 * K[m] + a2 * Sm[m];
    else
      D[m] = 0.5f * Sm[m];
  });
  cm19_shift<false>(D, K, ux, uy, uz);
  sfor<0, 19>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    float acc = feq[q];
    sfor<0, 19>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      constexpr float pc = (float)kCm19.P[q][m];
      if constexpr (pc != 0.0f) acc = acc + pc * K[m];
    });
    fv[q] = acc;
  });
}

// Force-free D3Q27 central-moment collision straight from the populations.
// The ten raw moments of order <= 2 of f - w (partial sums z, y, x) give rho
// and u, and -- because the second-order equilibrium reproduces those moments
// exactly (sum w = 1, sum w c_a c_b = delta/3, sum w c_a^2 c_b^2 = 1/9 for
// a != b, 1/3 for a == b) -- also the non-equilibrium raw moments:
//   N_0 = R_0 - (rho - 1),  N_a = R_a - rho u_a,
//   N_aa = R_aa - (rho - 1)/3 - rho u_a^2,  N_ab = R_ab - rho u_a u_b.
// Writing N_0 and N_a out (instead of dropping them as zero) keeps the
// rounding of rho and u exactly as mass- and momentum-conserving as the
// reference's f64 path.  Returns rho for the moving-wall bounce-back term.
__device__ __forceinline__ float collide_cm27_free_direct(float* fv, float os_base) {
#pragma clang fp contract(on)
  float Z0[9], Z1[9], Z2[9];
  sfor<0, 9>([&](auto abc) {
    constexpr int ab = decltype(abc)::value;
    constexpr int cx = ab / 3 - 1, cy = ab % 3 - 1;
    // populations of this (cx, cy) line with cz = -1, 0, +1
    constexpr int qm = [] {
      for (int q = 0; q < 27; ++q)
        if (lat_c(q, 0) == cx && lat_c(q, 1) == cy && lat_c(q, 2) == -1) return q;
      return -1;
    }();
    constexpr int q0 = [] {
      for (int q = 0; q < 27; ++q)
        if (lat_c(q, 0) == cx && lat_c(q, 1) == cy && lat_c(q, 2) == 0) return q;
      return -1;
    }();
    constexpr int qp = [] {
      for (int q = 0; q < 27; ++q)
        if (lat_c(q, 0) == cx && lat_c(q, 1) == cy && lat_c(q, 2) == 1) return q;
      return -1;
    }();
    Z2[ab] = fv[qp] + fv[qm];
    Z1[ab] = fv[qp] - fv[qm];
    Z0[ab] = Z2[ab] + fv[q0];
  });
  float Y00[3], Y10[3], Y20[3], Y01[3], Y11[3], Y02[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float* z0 = Z0 + 3 * a;
    const float* z1 = Z1 + 3 * a;
    const float* z2 = Z2 + 3 * a;
    Y20[a] = z0[2] + z0[0];
    Y10[a] = z0[2] - z0[0];
    Y00[a] = Y20[a] + z0[1];
    Y11[a] = z1[2] - z1[0];
    Y01[a] = (z1[2] + z1[0]) + z1[1];
    Y02[a] = (z2[2] + z2[0]) + z2[1];
  }
  const float R200 = Y00[2] + Y00[0], R100 = Y00[2] - Y00[0], R000 = R200 + Y00[1];
  const float R110 = Y10[2] - Y10[0], R010 = (Y10[2] + Y10[0]) + Y10[1];
  const float R020 = (Y20[2] + Y20[0]) + Y20[1];
  const float R101 = Y01[2] - Y01[0], R001 = (Y01[2] + Y01[0]) + Y01[1];
  const float R011 = (Y11[2] + Y11[0]) + Y11[1];
  const float R002 = (Y02[2] + Y02[0]) + Y02[1];
  const float r = 1.0f + R000;
  const float inv = 1.0f / r;
  const float ux = R100 * inv, uy = R010 * inv, uz = R001 * inv;
  const float dr = r - 1.0f;
  const float third_dr = dr * (1.0f / 3.0f);
  const float rux = r * ux, ruy = r * uy, ruz = r * uz;
  // non-equilibrium raw moments
  const float N000 = R000 - dr;
  const float N100 = R100 - rux, N010 = R010 - ruy, N001 = R001 - ruz;
  const float N200 = R200 - (third_dr + rux * ux);
  const float N020 = R020 - (third_dr + ruy * uy);
  const float N002 = R002 - (third_dr + ruz * uz);
  const float N110 = R110 - rux * uy, N101 = R101 - rux * uz, N011 = R011 - ruy * uz;
  // central moments of the non-equilibrium part
  const float K000 = N000;
  const float K100 = N100 - ux * N000, K010 = N010 - uy * N000, K001 = N001 - uz * N000;
  const float K200 = (N200 - 2.0f * ux * N100) + ux * ux * N000;
  const float K020 = (N020 - 2.0f * uy * N010) + uy * uy * N000;
  const float K002 = (N002 - 2.0f * uz * N001) + uz * uz * N000;
  const float K110 = ((N110 - ux * N010) - uy * N100) + ux * uy * N000;
  const float K101 = ((N101 - ux * N001) - uz * N100) + ux * uz * N000;
  const float K011 = ((N011 - uy * N001) - uz * N010) + uy * uz * N000;
  const float os = cm_rate(os_base, ux, uy, uz);
  const float a1 = 1.0f - os;
  const float kb = (K200 + K020 + K002) * (1.0f / 3.0f);
  const float d200 = a1 * (K200 - kb), d020 = a1 * (K020 - kb), d002 = a1 * (K002 - kb);
  const float d110 = a1 * K110, d101 = a1 * K101, d011 = a1 * K011;
  float X[27];
#pragma unroll
  for (int g = 0; g < 27; ++g) X[g] = 0.0f;
  const float ux2 = ux * ux, uy2 = uy * uy, uz2 = uz * uz;
  auto inv3 = [](float k0, float k1, float k2, float u, float u2, float& gm, float& g0, float& gp) {
    const float m1 = k1 + u * k0;
    const float m2 = (k2 + 2.0f * u * k1) + u2 * k0;
    gm = 0.5f * (m2 - m1);
    g0 = k0 - m2;
    gp = 0.5f * (m1 + m2);
  };
  auto inv2 = [](float k0, float k1, float u, float u2, float& gm, float& g0, float& gp) {
    const float m1 = k1 + u * k0;
    const float m2 = 2.0f * u * k1 + u2 * k0;
    gm = 0.5f * (m2 - m1);
    g0 = k0 - m2;
    gp = 0.5f * (m1 + m2);
  };
  auto inv1 = [](float k0, float u, float u2, float& gm, float& g0, float& gp) {
    const float m1 = u * k0;
    const float m2 = u2 * k0;
    gm = 0.5f * (m2 - m1);
    g0 = k0 - m2;
    gp = 0.5f * (m1 + m2);
  };
  inv3(K000, K100, d200, ux, ux2, X[0], X[9], X[18]);
  inv2(K010, d110, ux, ux2, X[3], X[12], X[21]);
  inv2(K001, d101, ux, ux2, X[1], X[10], X[19]);
  inv1(d020, ux, ux2, X[6], X[15], X[24]);
  inv1(d002, ux, ux2, X[2], X[11], X[20]);
  inv1(d011, ux, ux2, X[4], X[13], X[22]);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float* L = X + 9 * a;
    float g_m, g_0, g_p;
    inv3(L[0], L[3], L[6], uy, uy2, g_m, g_0, g_p);
    L[0] = g_m;
    L[3] = g_0;
    L[6] = g_p;
    inv2(L[1], L[4], uy, uy2, g_m, g_0, g_p);
    L[1] = g_m;
    L[4] = g_0;
    L[7] = g_p;
    inv1(L[2], uy, uy2, g_m, g_0, g_p);
    L[2] = g_m;
    L[5] = g_0;
    L[8] = g_p;
  }
#pragma unroll
  for (int ab = 0; ab < 9; ++ab) {
    float g_m, g_0, g_p;
    inv3(X[ab * 3 + 0], X[ab * 3 + 1], X[ab * 3 + 2], uz, uz2, g_m, g_0, g_p);
    X[ab * 3 + 0] = g_m;
    X[ab * 3 + 1] = g_0;
    X[ab * 3 + 2] = g_p;
  }
  // f' = feq + B(d).  Opposite directions share feq but for the sign of the
  // linear term: feq_{q, opp q} = s -+ t, s = w (b + 4.5 r cu^2), t = 3 w r cu.
  const float usq = ux2 + uy2 + uz2;
  const float b = dr - r * 1.5f * usq;
  const float r45 = 4.5f * r, r3 = 3.0f * r;
  fv[0] = lat_wf(27, 0) * b + X[gidx(0, 0, 0)];
  sfor<0, 13>([&](auto kc) {
    constexpr int qa = 2 * decltype(kc)::value + 1;
    constexpr int qb = qa + 1;
    constexpr int ga = gidx(lat_c(qa, 0), lat_c(qa, 1), lat_c(qa, 2));
    constexpr int gb = gidx(lat_c(qb, 0), lat_c(qb, 1), lat_c(qb, 2));
    constexpr float w = lat_wf(27, qa);
    const float cu = cdot<qa>(ux, uy, uz);
    const float sym = w * (b + r45 * (cu * cu));
    const float lin = (w * r3) * cu;
    fv[qa] = (sym + lin) + X[ga];
    fv[qb] = (sym - lin) + X[gb];
  });
  return r;
}

// ---------------------------------------------------------------------------
// one cell: load (parity), moments, collide, bounce-back-aware store
// ---------------------------------------------------------------------------
// Population slot addressing.  Plane bases are wave-uniform (scalar
// registers); the per-lane part of every address is one 32-bit byte offset,
// so the loads and stores use the scalar-base + 32-bit-offset form.  When no
// axis wraps, the neighbour shift is uniform as well and folds into the
// scalar base: all Q accesses of a cell share one offset register.
template <typename S, bool WRAP>
struct Slots {
  char* base;
  size_t plane_bytes;
  int64_t sy, sz;  // element strides of y and z
  uint32_t voff;   // i * sizeof(S)
  uint32_t i;
  Nbr nb;
  __device__ __forceinline__ Slots(const HydroArgs& a, uint32_t i_, uint32_t x, uint32_t y, uint32_t z)
      : base((char*)a.f),
        plane_bytes((size_t)a.d.ps * sizeof(S)),
        sy(a.d.nx),
        sz((int64_t)a.d.nx * a.d.ny),
        voff(i_ * (uint32_t)sizeof(S)),
        i(i_),
        nb(a.d, x, y, z) {}
  // slot of plane p at cell i + (cx, cy, cz)
  template <int p, int cx, int cy, int cz>
  __device__ __forceinline__ S* at() const {
    if constexpr (!WRAP) {
      const int64_t shift = ((int64_t)cx + cy * sy + cz * sz) * (int64_t)sizeof(S);
      return (S*)(base + p * plane_bytes + shift + voff);
    } else {
      const uint32_t o = (i + (uint32_t)nb.template off<cx, cy, cz>()) * (uint32_t)sizeof(S);
      return (S*)(base + p * plane_bytes + o);
    }
  }
};

template <typename S, int Q, int q>
__device__ __forceinline__ float slot_ld(const S* p) {
  float v = Store<S>::ld(p, 0);
  if constexpr (Store<S>::kScaled) v = v * lat_wf(Q, q);
  return v;
}
template <typename S, int Q, int q>
__device__ __forceinline__ void slot_st(S* p, float v) {
  if constexpr (Store<S>::kScaled) v = v * lat_inv_w(Q, q);
  Store<S>::st(p, 0, v);
}

// Bounce-back layout.  A population reflected off the wall at i + c_q is
// stored where the plain AA store of direction q would put it in the cell's
// own slots: even steps write slot opp(q) of cell i (the plain target), odd
// steps write slot opp(q) of cell i instead of slot q of i + c_q.  The odd
// step then reads a wall-link direction q (i - c_q solid) from the cell's
// own slot q, not from the solid upstream cell.  So no fluid cell ever reads
// or writes a solid cell's slots, and a solid cell inside an active tile can
// rewrite its own slots freely: even steps do, which turns every store of an
// active tile into whole cache lines (partial lines cost the memory a
// read-modify-write).
//
// PLAIN: the whole tile is fluid with mask word 0 (no wall link, no force
// list, no moving wall), known from the tile list; the mask is not read.
// WALE: the relaxation rate comes from the closure (lbm_wale.hpp), taken here
// from the neighbours' cached velocities and written to the omega field.
template <int Q, typename S, int KIND, bool ODD, bool FON, bool WRAP, bool FILL, bool PLAIN = false,
          bool WALE = false>
__device__ __forceinline__ void cell_step(const HydroArgs& a, uint32_t i, uint32_t x, uint32_t y, uint32_t z,
                                          const uint32_t* mask_ptr, uint32_t skip, const float Fm[3],
                                          const float Fc[3], uint32_t xlo = 0u, uint32_t xhi = 0u,
                                          uint32_t xr = 0xFFFFFFFFu) {
  constexpr bool fon = FON;
  const Slots<S, WRAP> sl(a, i, x, y, z);
  // The mask word and the Q populations are loaded together: the loads do
  // not wait for the solid test (the buffer's guard bands keep a solid face
  // cell's neighbour addresses inside the allocation); only the stores are
  // predicated on it.
  const uint32_t m = PLAIN ? 0u : *mask_ptr;
  float fv[Q];
  [[maybe_unused]] float wale_om = 0.0f;
  auto slot = [&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int o = lat_opp(q);
    if constexpr (!ODD)
      return (const S*)sl.template at<q, 0, 0, 0>();
    else
      return (const S*)sl.template at<o, -lat_c(q, 0), -lat_c(q, 1), -lat_c(q, 2)>();
  };
  if constexpr (WALE) {
    // The closure's loads go first and the rate is computed while the
    // populations are still on their way, so it costs the step neither a
    // latency nor a register of its peak.  The fence keeps every load ahead of
    // the first use: without it the scheduler meets the register limit by
    // waiting for each 16-bit load before the next (512^3 fp16 odd step 5.11
    // ms against 3.24).
    WaleLoads<PLAIN> wl(a.wale, a.d, i);
    S raw[Q];
    sfor<0, Q>([&](auto qc) { raw[decltype(qc)::value] = *slot(qc); });
    __builtin_amdgcn_sched_barrier(0);
    if (!(m & kMaskSolid)) wale_om = wl.omega(a.wale, a.d, a.wall_u, i, m);
    sfor<0, Q>([&](auto qc) { fv[decltype(qc)::value] = slot_ld<S, Q, decltype(qc)::value>(&raw[decltype(qc)::value]); });
  } else {
    sfor<0, Q>([&](auto qc) { fv[decltype(qc)::value] = slot_ld<S, Q, decltype(qc)::value>(slot(qc)); });
  }
  // Consume every loaded value before the solid test, so the compiler cannot
  // sink the population loads behind the mask branch: one memory latency per
  // cell instead of two.
#pragma unroll
  for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(fv[q]));
  // A solid cell of an active tile runs along with its wave and stores zeros
  // into dead slots (even steps: its own; odd steps, D3Q27 with fp32
  // storage: those of its targets that no fluid cell writes), so the tile's
  // stores cover whole cache lines.  With 16-bit storage the odd-step fill
  // speeds up the next even step about as much as it slows the odd one, and
  // on D3Q19 (the batched tanks) it measured 1.3 % slower, so both keep the
  // plain odd step.
  constexpr bool kOddFill = sizeof(S) == 4 && Q == 27;
  const bool dead = FILL && (!ODD || kOddFill) && (m & kMaskSolid) != 0;
  if (m & skip & (dead ? ~kMaskSolid : ~0u)) return;
  if constexpr (ODD) {
    if (!dead && (m & kMaskLinks)) {  // wall links: the bounced population is in the own slot
      // Every reload is issued before any is used: a 16-bit value converted
      // inside its own conditional made each load wait for the one before
      // (one memory latency per link direction).  So each direction issues
      // one unconditional wave-wide load: the own slot q when some lane of
      // the wave needs it, else the own slot 0 the step has just read (an L1
      // hit); the choice is wave-uniform, no branch, no merge to wait for.
      S raw[Q];
      sfor<1, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const bool need = __builtin_amdgcn_ballot_w64(((m >> q) & 1u) != 0u) != 0u;
        raw[q] = *(need ? sl.template at<q, 0, 0, 0>() : sl.template at<0, 0, 0, 0>());
      });
      sfor<1, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if ((m >> q) & 1u) {
          float v = Store<S>::ld(&raw[q], 0);
          if constexpr (Store<S>::kScaled) v = v * lat_wf(Q, q);
          fv[q] = v;
        }
      });
    }
  }
  float op = a.p.omega_p, cp = a.p.cp, os = a.p.omega_shear;
  if (WALE || a.omega) {  // per-cell omega_plus (kernels.rs:151-156)
    op = WALE ? wale_om : a.omega[i];
    cp = 1.0f - op / 2.0f;
    os = op;
    if constexpr (WALE)
      if (!dead) a.wale.omega[i] = op;
  }
  float r;
  if constexpr (KIND == 0) {
    float ux, uy, uz;
    moments<Q>(fv, Fm, fon, r, ux, uy, uz);
    collide_trt<Q, !Store<S>::kScaled>(fv, r, ux, uy, uz, Fc, fon, op, cp, a.p);
  } else if constexpr (Q == 19) {
    float ux, uy, uz;
    moments<Q>(fv, Fm, fon, r, ux, uy, uz);
    collide_cm19_general(fv, r, ux, uy, uz, Fc, fon, os);
  } else {
    static_assert(Q == 27, "central-moment kernels are D3Q19 or D3Q27");
    if constexpr (FON) {
      float ux, uy, uz;
      moments<Q>(fv, Fm, fon, r, ux, uy, uz);
      collide_cm27_general(fv, r, ux, uy, uz, Fc, true, os);
    } else {
      r = collide_cm27_free_direct(fv, os);
    }
  }
  // half-way bounce-back off a moving wall at i + c_q (stream_row,
  // kernels.rs:591-603): the reflected population enters i along c_o with
  // fin = fout + 6 w_o rho (c_o . u_wall)
  if (m & kMaskMoving) {
    sfor<1, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int o = lat_opp(q);
      if ((m >> o) & 1u) {
        // (no wrapping axis: a fluid cell's neighbours are inside the domain,
        // so the linear offset is the wrapped one)
        const uint32_t fwd =
            WRAP ? i + (uint32_t)sl.nb.template off<lat_c(q, 0), lat_c(q, 1), lat_c(q, 2)>()
                 : i + (uint32_t)(lat_c(q, 0) + lat_c(q, 1) * (int32_t)a.d.nx + lat_c(q, 2) * (int32_t)(a.d.nx * a.d.ny));
        const float* wu = a.wall_u + 3 * (size_t)fwd;
        const float cu = cdot<o>(wu[0], wu[1], wu[2]);
        constexpr float six_w = 6.0f * lat_wf(Q, o);
        fv[q] = fv[q] + six_w * r * cu;
      }
    });
  }
  // plain streaming store of direction q
  auto store_plain = [&](auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int o = lat_opp(q);
    if constexpr (!ODD)
      slot_st<S, Q, q>(sl.template at<o, 0, 0, 0>(), dead ? 0.0f : fv[q]);
    else
      slot_st<S, Q, q>(sl.template at<q, lat_c(q, 0), lat_c(q, 1), lat_c(q, 2)>(), fv[q]);
  };
  // even steps: the bounced population goes to the plain target as well
  if constexpr (!ODD || PLAIN) {
    sfor<0, Q>(store_plain);
  } else if constexpr (!FILL || !kOddFill) {
    // one exec-masked pair of stores per direction for the whole wave
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int o = lat_opp(q);
      if ((m >> o) & 1u)
        slot_st<S, Q, q>(sl.template at<o, 0, 0, 0>(), fv[q]);
      else
        store_plain(qc);
    });
  } else {
    // Odd steps of an active fp32 tile.  A wall-link lane stores the bounced
    // population in its own slot; a solid lane writes zeros to each of its
    // targets that no fluid cell writes (mask bit q clear), only inside the
    // tile's live x range [xlo, xhi], so no store reaches a line outside the
    // tile's own.  (Also writing a link lane's plain target, a dead slot,
    // measured slower.)
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int o = lat_opp(q);
      constexpr int cx = lat_c(q, 0);
      // xr: the coordinate the live range is in (x for row tiles, the cell
      // index for linear tiles)
      const uint32_t xc = xr == 0xFFFFFFFFu ? x : xr;
      const bool inr = cx == 0 || ((uint32_t)(xc + cx) >= xlo && (uint32_t)(xc + cx) <= xhi);
      const bool link = !dead && ((m >> o) & 1u);
      const bool plain = dead ? (!((m >> q) & 1u) && inr) : !link;
      if (link) slot_st<S, Q, q>(sl.template at<o, 0, 0, 0>(), fv[q]);
      if (plain)
        slot_st<S, Q, q>(sl.template at<q, lat_c(q, 0), lat_c(q, 1), lat_c(q, 2)>(), dead ? 0.0f : fv[q]);
    });
  }
}

template <int Q, typename S, int KIND, bool ODD, bool FON, bool WRAP, bool LIN, bool WALE>
__device__ __forceinline__ void hydro_tile(const HydroArgs& a) {
  // each wave takes one active 64-cell tile; tiles of only solid (or
  // force-listed) cells are never launched
  // What the tile entry's address needs is loaded at once: left to the compiler
  // each side of the remap's branch waited for its own scalar loads, a second
  // latency before the wave's first vector load.
  uint32_t n = gridDim.x, deal = a.deal, ntiles = a.ntiles;
  uint64_t list = (uint64_t)a.tiles;
  asm volatile("" : "+s"(n), "+s"(deal), "+s"(ntiles), "+s"(list));
  const auto* tiles = (const __attribute__((address_space(1))) uint32_t*)list;
  const uint32_t b = xcd_remap(blockIdx.x, n, deal);
  const uint32_t t = b * 4 + (threadIdx.x >> 6);
  if (t >= ntiles) return;
  const uint32_t te = __builtin_amdgcn_readfirstlane(tiles[t]);  // one tile per wave
  const uint32_t tile = te & kTileId;
  if (WRAP ? LIN : a.lin != 0) {
    // linear tile: cells 64 tile .. 64 tile + 63 across row ends (where no
    // axis wraps every neighbour shift is the linear one, elsewhere each lane
    // takes its own coordinates)
    const uint32_t i = tile * 64 + (threadIdx.x & 63);
    if (i >= a.d.N || (te & ((threadIdx.x & 32) ? kTileDeadHi : kTileDeadLo))) return;
    uint32_t x = 0u, y = 0u, z = 0u;
    if constexpr (WRAP) cell_xyz(a.d, i, x, y, z);
    if (te & kTilePlain) {
      cell_step<Q, S, KIND, ODD, FON, WRAP, true, true, WALE>(a, i, x, y, z, nullptr, 0u, a.p.F, a.p.F);
    } else {
      const uint32_t c0 = tile * 64;
      const uint32_t lo = (te & kTileDeadLo) ? c0 + 32 : c0;
      const uint32_t hi = min((te & kTileDeadHi) ? c0 + 31 : c0 + 63, a.d.N - 1);
      cell_step<Q, S, KIND, ODD, FON, WRAP, true, false, WALE>(a, i, x, y, z, a.mask + i, kMaskSolid | kMaskForced,
                                                         a.p.F, a.p.F, lo, hi, i);
    }
    return;
  }
  const uint32_t row = tile / a.nseg, seg = tile - row * a.nseg;
  const uint32_t x = seg * 64 + (threadIdx.x & 63);
  if (x >= a.d.nx || (te & ((threadIdx.x & 32) ? kTileDeadHi : kTileDeadLo))) return;
  const uint32_t y = row % a.d.ny, z = row / a.d.ny;
  const uint32_t i = row * a.d.nx + x;
  if (te & kTilePlain) {
    cell_step<Q, S, KIND, ODD, FON, WRAP, true, true, WALE>(a, i, x, y, z, nullptr, 0u, a.p.F, a.p.F);
  } else {
    // the tile's live x range (an all-solid half is not visited)
    const uint32_t x0 = seg * 64;
    const uint32_t xlo = (te & kTileDeadLo) ? x0 + 32 : x0;
    const uint32_t xhi = min((te & kTileDeadHi) ? x0 + 31 : x0 + 63, a.d.nx - 1);
    cell_step<Q, S, KIND, ODD, FON, WRAP, true, false, WALE>(a, i, x, y, z, a.mask + i, kMaskSolid | kMaskForced,
                                                       a.p.F, a.p.F, xlo, xhi);
  }
}

// WRAP with LIN: packed tiles on a wrapped domain, a kernel of their own.  Both
// tile forms in one kernel took up to 18 VGPRs more (odd D3Q19 CM with a force 127
// -> 137, a wave per SIMD fewer), which the row tiles paid for (periodic 256^3
// D3Q27 fp32 with a force 0.774 against 0.759 ms).
template <int Q, typename S, int KIND, bool ODD, bool FON, bool WRAP, bool LIN>
__global__ __launch_bounds__(256) void k_hydro(HydroArgs a) {
  hydro_tile<Q, S, KIND, ODD, FON, WRAP, LIN, false>(a);
}

// The step with the WALE closure inside (closed domains, no uniform force):
// the gradient, nu_t and omega_plus of each cell it updates, instead of a pass
// of their own that writes an omega field for this kernel to read.  The
// velocities of the neighbours come from L2 (18 loads); what is added from HBM
// is what that pass read (24 bytes per cell), what is saved is its launch, its
// masks and its waiting: it was bound by VALU and latency, and here both hide
// under the populations' loads.  Four waves per SIMD as k_hydro has.
// Per step, closure and collide-stream: 256^3 D3Q27 fp32 1.153 -> 1.094 ms (the
// velocity pass 0.365, this kernel 0.705 / 0.753); 512^3 fp16 with a D3Q7
// tracer taken along by that pass 8.31 -> 6.41 ms (3.10, and 3.03 / 3.58 here,
// where nu_t's 380 VALU instructions per wave make it VALU-bound).
template <int Q, typename S, int KIND, bool ODD>
__global__ __launch_bounds__(256, 4) void k_hydro_wale(HydroArgs a) {
  hydro_tile<Q, S, KIND, ODD, false, false, false, true>(a);
}

// Cells carrying a per-cell force: the velocity uses the force of the cached
// moments (F_mom, set when moments were last refreshed), the Guo source the
// current field (F_cur), as the reference's stale-moment step does
// (solver.rs:2805-2822 keeps moments across a non-uniform clear).  After the
// step the cached moments carry F_cur.
template <int Q, typename S, int KIND, bool ODD, bool WALE = false>
__device__ __forceinline__ void list_cell(const HydroArgs& a, uint32_t i) {
  const uint32_t m = a.mask[i];
  if (m & kMaskSolid) return;
  const uint32_t x = i % a.d.nx, t = i / a.d.nx;
  const uint32_t y = t % a.d.ny, z = t / a.d.ny;
  float Fm[3], Fc[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    Fm[c] = a.p.F[c] + a.F_mom[3 * (size_t)i + c];
    Fc[c] = a.p.F[c] + a.F_cur[3 * (size_t)i + c];
  }
  cell_step<Q, S, KIND, ODD, true, true, false, false, WALE>(a, i, x, y, z, a.mask + i, kMaskSolid, Fm, Fc);
#pragma unroll
  for (int c = 0; c < 3; ++c) a.F_mom[3 * (size_t)i + c] = a.F_cur[3 * (size_t)i + c];
}

template <int Q, typename S, int KIND, bool ODD, bool WALE = false>
__global__ __launch_bounds__(256) void k_hydro_list(HydroArgs a) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.nlist) return;
  list_cell<Q, S, KIND, ODD, WALE>(a, a.flist[k]);
}

// ---------------------------------------------------------------------------
// Batched domains: one launch walks the concatenated tile lists of K
// independent (non-periodic) domains; entry e = (tile, domain).  A wave takes
// one entry, or strides over them when the grid was set smaller, and reads its
// tile's domain arguments from the table (wave-uniform, so scalar loads).
// ---------------------------------------------------------------------------
template <int Q, typename S, int KIND, bool ODD>
__global__ __launch_bounds__(256) void k_hydro_batch(const HydroArgs* __restrict__ tab,
                                                     const uint32_t* __restrict__ ent, uint32_t nent,
                                                     uint32_t deal) {
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x, deal);
  const uint32_t stride = gridDim.x * 4;
  for (uint32_t e = b * 4 + (threadIdx.x >> 6); e < nent; e += stride) {
    const uint32_t te = __builtin_amdgcn_readfirstlane(ent[2 * (size_t)e]);
    const uint32_t k = __builtin_amdgcn_readfirstlane(ent[2 * (size_t)e + 1]);
    const HydroArgs& a = tab[k];
    const uint32_t tile = te & kTileId;
    if (a.lin) {  // linear tile (members never wrap)
      const uint32_t i = tile * 64 + (threadIdx.x & 63);
      if (i < a.d.N && !(te & ((threadIdx.x & 32) ? kTileDeadHi : kTileDeadLo))) {
        if (te & kTilePlain) {
          cell_step<Q, S, KIND, ODD, false, false, true, true>(a, i, 0u, 0u, 0u, nullptr, 0u, a.p.F, a.p.F);
        } else {
          const uint32_t c0 = tile * 64;
          const uint32_t lo = (te & kTileDeadLo) ? c0 + 32 : c0;
          const uint32_t hi = min((te & kTileDeadHi) ? c0 + 31 : c0 + 63, a.d.N - 1);
          cell_step<Q, S, KIND, ODD, false, false, true, false>(a, i, 0u, 0u, 0u, a.mask + i,
                                                                kMaskSolid | kMaskForced, a.p.F, a.p.F, lo, hi, i);
        }
      }
      continue;
    }
    const uint32_t row = tile / a.nseg, seg = tile - row * a.nseg;
    const uint32_t x = seg * 64 + (threadIdx.x & 63);
    if (x < a.d.nx && !(te & ((threadIdx.x & 32) ? kTileDeadHi : kTileDeadLo))) {
      const uint32_t y = row % a.d.ny, z = row / a.d.ny;
      const uint32_t i = row * a.d.nx + x;
      if (te & kTilePlain) {
        cell_step<Q, S, KIND, ODD, false, false, true, true>(a, i, x, y, z, nullptr, 0u, a.p.F, a.p.F);
      } else {
        const uint32_t x0 = seg * 64;
        const uint32_t xlo = (te & kTileDeadLo) ? x0 + 32 : x0;
        const uint32_t xhi = min((te & kTileDeadHi) ? x0 + 31 : x0 + 63, a.d.nx - 1);
        cell_step<Q, S, KIND, ODD, false, false, true, false>(a, i, x, y, z, a.mask + i, kMaskSolid | kMaskForced,
                                                              a.p.F, a.p.F, xlo, xhi);
      }
    }
  }
}

// forced cells of all domains: entry = (cell, domain)
template <int Q, typename S, int KIND, bool ODD>
__global__ __launch_bounds__(256) void k_hydro_list_batch(const HydroArgs* __restrict__ tab,
                                                          const uint32_t* __restrict__ cells, uint32_t n) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  list_cell<Q, S, KIND, ODD>(tab[cells[2 * (size_t)k + 1]], cells[2 * (size_t)k]);
}

static inline uint32_t blocks_for(size_t n, uint32_t bs = 256) { return (uint32_t)((n + bs - 1) / bs); }

template <int Q, typename S, int KIND, bool ODD, bool FON>
static void hydro_w(bool wrap, const HydroArgs& a, dim3 grid, hipStream_t s) {
  if (!wrap)
    hipLaunchKernelGGL((k_hydro<Q, S, KIND, ODD, FON, false, false>), grid, dim3(256), 0, s, a);
  else if (a.lin)
    hipLaunchKernelGGL((k_hydro<Q, S, KIND, ODD, FON, true, true>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_hydro<Q, S, KIND, ODD, FON, true, false>), grid, dim3(256), 0, s, a);
}

template <int Q, typename S, int KIND>
static hipError_t hydro_q(int odd, const HydroArgs& a, hipStream_t s, bool list) {
  if (list) {
    if (a.nlist == 0) return hipSuccess;
    const dim3 grid(blocks_for(a.nlist)), block(256);
    if (a.wale.vel) {
      if (odd)
        hipLaunchKernelGGL((k_hydro_list<Q, S, KIND, true, true>), grid, block, 0, s, a);
      else
        hipLaunchKernelGGL((k_hydro_list<Q, S, KIND, false, true>), grid, block, 0, s, a);
    } else if (odd)
      hipLaunchKernelGGL((k_hydro_list<Q, S, KIND, true>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((k_hydro_list<Q, S, KIND, false>), grid, block, 0, s, a);
    return hipGetLastError();
  }
  if (a.ntiles == 0) return hipSuccess;
  const dim3 grid((a.ntiles + 3) / 4), block(256);
  const bool fon = a.p.force_on != 0;
  const bool wrap = a.d.per[0] || a.d.per[1] || a.d.per[2] || a.open;
  if (a.wale.vel) {  // closed domains without a uniform force (wale_in_step)
    if (fon || wrap) return hipErrorInvalidValue;
    if (odd)
      hipLaunchKernelGGL((k_hydro_wale<Q, S, KIND, true>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((k_hydro_wale<Q, S, KIND, false>), grid, block, 0, s, a);
    return hipGetLastError();
  }
  if (odd)
    fon ? hydro_w<Q, S, KIND, true, true>(wrap, a, grid, s) : hydro_w<Q, S, KIND, true, false>(wrap, a, grid, s);
  else
    fon ? hydro_w<Q, S, KIND, false, true>(wrap, a, grid, s) : hydro_w<Q, S, KIND, false, false>(wrap, a, grid, s);
  return hipGetLastError();
}

template <int Q, typename S, int KIND>
static hipError_t batch_q(int odd, const HydroArgs* tab, const uint32_t* ent, uint32_t nent, uint32_t grid,
                          const uint32_t* cells, uint32_t ncells, hipStream_t s) {
  if (ent) {
    if (nent == 0) return hipSuccess;
    // one stretch of entries per XCD for a batch that the last-level cache
    // holds, the plain order for larger ones (ms per step: 4 tanks of edges 48
    // to 90, 0.16 GB: 0.0823, 0.0870; 4 of 100 to 160, 0.66 GB: 0.308, 0.295;
    // 40 tanks, 4.6 GB: 1.830, 1.758)
    const uint32_t deal = grid < 16384 ? kXcdStretch : 0;
    if (odd)
      hipLaunchKernelGGL((k_hydro_batch<Q, S, KIND, true>), dim3(grid), dim3(256), 0, s, tab, ent, nent, deal);
    else
      hipLaunchKernelGGL((k_hydro_batch<Q, S, KIND, false>), dim3(grid), dim3(256), 0, s, tab, ent, nent, deal);
  } else {
    if (ncells == 0) return hipSuccess;
    if (odd)
      hipLaunchKernelGGL((k_hydro_list_batch<Q, S, KIND, true>), dim3(blocks_for(ncells)), dim3(256), 0, s, tab,
                         cells, ncells);
    else
      hipLaunchKernelGGL((k_hydro_list_batch<Q, S, KIND, false>), dim3(blocks_for(ncells)), dim3(256), 0, s, tab,
                         cells, ncells);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// this object file's lattice, storage and collision
// ---------------------------------------------------------------------------
#if LBM_STORAGE == 0
using HydroS = float;
#elif LBM_STORAGE == 1
using HydroS = _Float16;
#else
using HydroS = bf16s;
#endif

template <>
hipError_t hydro_launch<LBM_Q, LBM_STORAGE, LBM_KIND>(int odd, const HydroArgs& a, hipStream_t s, bool list) {
  return hydro_q<LBM_Q, HydroS, LBM_KIND>(odd, a, s, list);
}

template <>
hipError_t batch_launch<LBM_Q, LBM_STORAGE, LBM_KIND>(int odd, const HydroArgs* tab, const uint32_t* ent,
                                                      uint32_t nent, uint32_t grid, const uint32_t* cells,
                                                      uint32_t ncells, hipStream_t s) {
  return batch_q<LBM_Q, HydroS, LBM_KIND>(odd, tab, ent, nent, grid, cells, ncells, s);
}

}  // namespace lbm
