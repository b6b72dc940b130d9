// The collision of an MD-coupled cell (device code): lbm_couple.hip re-collides the coupled cells with it
// after a step, lbm_small.hip collides them with it in the boxes around the coupled cells.
#pragma once

#include "lbm_capi.h"
#include "lbm_internal.h"

namespace lbm {

// The GET block of getAndSetV (:100-129) for coupled cell k, on the cell's rho and u: overwrite sets
// u = u_MD (:121-122); Dirichlet computes g = (u_MD - u)/dt and shifts u += dt/2 g (:110-117); with
// density coupling rho = rho_MD (:124-129).  g stays 0 in the overwrite mode.
__device__ __forceinline__ void couple_get(const CoupleArgs& a, int64_t k, double& rho, double (&u)[3],
                                           double (&g)[3]) {
  const double* um = a.u + 3 * k;
  g[0] = g[1] = g[2] = 0.0;
  if (a.mode == LBM_COUPLE_DIRICHLET) {
    for (int d = 0; d < 3; d++) {
      g[d] = (um[d] - u[d]) / a.dt;
      u[d] += a.dt / 2.0 * g[d];
    }
  } else {
    for (int d = 0; d < 3; d++) u[d] = um[d];
  }
  if (a.rho) rho = a.rho[k];
}

// FP64 collision of one coupled cell (reference operation order, as the oracle restates it).
__device__ __forceinline__ double collide_coupled_f64(double (&f)[Q], const CoupleArgs& a, int64_t k,
                                                      double (&uo)[3]) {
  double rho = 0.0;
#pragma unroll
  for (int q = 0; q < Q; q++) rho += f[q];
  double b0 = 0.0, b1 = 0.0, b2 = 0.0;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    if (CX(q) == 1) b0 += f[q];
    if (CX(q) == -1) b0 -= f[q];
    if (CY(q) == 1) b1 += f[q];
    if (CY(q) == -1) b1 -= f[q];
    if (CZ(q) == 1) b2 += f[q];
    if (CZ(q) == -1) b2 -= f[q];
  }
  const double inv = 1.0 / rho;
  double u[3] = {b0 * inv, b1 * inv, b2 * inv};
  double g[3];
  couple_get(a, k, rho, u, g);
  const bool dir = a.mode == LBM_COUPLE_DIRICHLET;
  uo[0] = u[0];
  uo[1] = u[1];
  uo[2] = u[2];
  double uu = u[0] * u[0];
  uu += u[1] * u[1];
  uu += u[2] * u[2];
  const double du = over_cs2x2(uu);
  f[REST] -= a.omega * (f[REST] - W64(REST) * rho * (1.0 - du));
#pragma unroll
  for (int q = 0; q < REST; q++) {
    const FeqPair e = feq_pair_f64(q, rho, cdot64(q, u[0], u[1], u[2]), du);
    f[q] -= a.omega * (f[q] - e.q);
    f[Q - 1 - q] -= a.omega * (f[Q - 1 - q] - e.mirror);
  }
  if (dir) {
    // adjustF / computeGi, with (c.u)^2 as the reference writes it; a direction and its mirror share
    // (c.u)^2 / cs4, and c.g changes its sign
    const double pref = 1.0 - 0.5 / a.tau;
    auto add = [&](int q, double quad) {
      const double m0 = (double)CX(q) - u[0], m1 = (double)CY(q) - u[1], m2 = (double)CZ(q) - u[2];
      double cmg = m0 * g[0];
      cmg += m1 * g[1];
      cmg += m2 * g[2];
      const double gi = pref * W64(q) * rho * (1.0 / (1.0 / 3.0) * cmg + quad);
      f[q] += a.dt * gi;
    };
    add(REST, 0.0);
#pragma unroll
    for (int q = 0; q < REST; q++) {
      const double cu = cdot64(q, u[0], u[1], u[2]);
      const double quad = over_cs4(cu * cu) * cdot64(q, g[0], g[1], g[2]);
      add(q, quad);
      add(Q - 1 - q, -quad);
    }
  }
  return rho;
}

// Coupled collision of cell k (stored index i, flag word w), then the boundary class of its links.
template <bool WALLS>
__device__ __forceinline__ void couple_collide(double (&f)[Q], const CoupleArgs& a, int64_t k, int64_t i, uint32_t w,
                                               const BoundaryArgs& bc) {
  double u[3];
  const double rho = collide_coupled_f64(f, a, k, u);
  if (WALLS) {
    const uint32_t cls = (w >> CLASS_SHIFT) & CLASS_BITS;
    if (cls) {
      const BoundaryClass& b = bc.table[cls];
      const uint32_t m = w & b.mask;
      if (m) apply_boundary_f64(f, m, b, bc.cell_u, i, rho, u[0], u[1], u[2]);
    }
  }
}

// The same for populations of the state's type: FP32-shifted ones are lifted to FP64.
template <typename T, bool WALLS>
__device__ __forceinline__ void couple_cell(T (&f)[Q], const CoupleArgs& a, int64_t k, int64_t i, uint32_t w,
                                            const BoundaryArgs& bc) {
  double d[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) d[q] = sizeof(T) == 8 ? (double)f[q] : (double)f[q] + W64(q);
  couple_collide<WALLS>(d, a, k, i, w, bc);
#pragma unroll
  for (int q = 0; q < Q; q++) f[q] = sizeof(T) == 8 ? (T)d[q] : (T)(d[q] - W64(q));
}

}  // namespace lbm
