// The cell update of the dense steps: collision and boundary classes of one fluid cell, and the
// whole-line rule of their stores (shared by the one-step, in-place and two-step kernels).
#pragma once

#include "lbm_geom.h"

namespace lbm {

// Collision of one fluid cell plus the boundary classes of its bounce-back links (shared by the
// two-buffer and the AA steps).  T = double: reference arithmetic; T = float: shifted populations,
// hybrid arithmetic (collide_f32s_h) unless M32 (all FP32).
template <typename T, bool FORCE, bool ALPHA, bool WALLS, bool M32, bool MIRROR = true>
__device__ __forceinline__ void collide_cell_bc(T (&f)[Q], uint32_t w, int64_t i, const T* __restrict__ alpha,
                                                const CollideParams& p64, const CollideParams32& p32,
                                                const BoundaryArgs& bc) {
  const T a = ALPHA ? alpha[i] : T(0);
  T rho;
  T uc[sizeof(T) == 8 ? 3 : 4];
  if constexpr (sizeof(T) == 8) {
    rho = collide_f64<FORCE, ALPHA>(f, p64, a, uc);
  } else if constexpr (M32) {
    rho = collide_f32s<FORCE, ALPHA>(f, p32, a, uc);
  } else {
    rho = collide_f32s_h<FORCE, ALPHA, MIRROR>(f, p64, p32, a, uc);
  }
  if (WALLS) {
    const uint32_t k = (w >> CLASS_SHIFT) & CLASS_BITS;
    if (k) {
      const BoundaryClass& b = bc.table[k];
      const uint32_t m = w & b.mask;
      if (m) {
        if constexpr (sizeof(T) == 8) apply_boundary_f64(f, m, b, bc.cell_u, i, rho, uc[0], uc[1], uc[2]);
        else apply_boundary_f32(f, m, b, bc.cell_u, i, rho, uc[3], uc[0], uc[1], uc[2]);
      }
    }
  }
}

// ------------------------------------------------------------------------------------------
// Whether this lane's 128-byte line of a population plane holds a fluid lane of the wavefront
// (`fluid` = the wavefront's ballot of fluid lanes).  A solid lane in such a line stores zeros into
// its own slots (never read: pulls and readers skip non-fluid cells) together with the fluid lanes'
// stores, so the line is written whole: partial-line writes at the solid surfaces cost more.
template <typename T>
__device__ __forceinline__ bool line_has_fluid(unsigned long long fluid) {
  constexpr int LANES = 128 / (int)sizeof(T);
  const int first = (int)(threadIdx.x & 63) & ~(LANES - 1);  // lane of the wavefront
  const unsigned long long line = (LANES >= 64) ? ~0ull : (((1ull << LANES) - 1ull) << first);
  return (fluid & line) != 0;
}

}  // namespace lbm
