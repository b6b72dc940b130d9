// Two to four time steps in one launch on small lattices: k_dense_small.
//
// A step of a small lattice takes 5-7 us however few its cells are: dispatch, the flag word, the populations,
// one collision and the stores, one after the other.  Here a workgroup loads a box of 8 x 8 x 8 cells, one per
// thread, and steps it `steps` times in its registers: after each step the populations pass through the
// LDS, and the box that still has all its neighbours shrinks by one cell on every side, so 6^3, 4^3 or
// 2^3 cells (two, three, four steps) remain to be stored.  The rest is computed by several workgroups, which
// CUs without work of their own do for nothing.  (8^3 cells are 8 waves: each SIMD interleaves two, and
// the LDS rows of a population are consecutive lanes.)  Every cell goes through the same collide_cell_bc:
// the same bits as single steps.
//
// With the MD coupling (CPL) it runs two steps of a list of boxes, after the two-step kernel has done the whole
// lattice without it: those that hold a coupled cell or a neighbour of one, the only cells that come out
// different.  (The coupled collision inside the two-step kernel made 96^3 FP64 149 us a step instead of 67: its
// 500 instructions a cell lie on the path of the few workgroups that hold the MD region, in every plane.)
//
// Per step, one-step kernel -> this one: 12^3 FP64 lid 5.8 -> 3.3 us (four steps a launch), periodic 5.2 -> 2.7;
// 18^3 lid 5.8 -> 3.7 (three), 24^3 5.9 -> 4.9; FP32 12^3 lid 5.4 -> 2.9, 24^3 5.3 -> 3.9.
#include "lbm_collide.h"
#include "lbm_couple.h"

namespace lbm {

namespace {

struct SmallGeom {
  int steps;
  int tx, ty, tz;  // boxes along x, y, z
};

constexpr int EDGE = 8, CELLS = EDGE * EDGE * EDGE;
constexpr int NCU = 256;

template <typename T, bool FORCE, bool ALPHA, bool WALLS, bool CPL, bool M32, bool AOS>
__global__ __launch_bounds__(CELLS, 4) void k_dense_small(DenseGeom g, SmallGeom sg, const T* __restrict__ src,
                                                          T* __restrict__ dst, const uint32_t* __restrict__ words,
                                                          const T* __restrict__ alpha, CollideParams p64,
                                                          CollideParams32 p32, BoundaryArgs bc, CoupleArgs cpl,
                                                          const int32_t* __restrict__ idx,
                                                          const int32_t* __restrict__ boxes) {
  __shared__ T lds[Q * CELLS];  // (the rest population's row is not used)
  __shared__ BoundaryClass classes[WALLS ? MAX_CLASSES : 1];
  const int tid = (int)threadIdx.x, lx = tid & 7, ly = (tid >> 3) & 7, lz = tid >> 6;
  const int halo = sg.steps - 1, out = EDGE - 2 * halo;
  const int b = CPL ? boxes[blockIdx.x] : (int)blockIdx.x, bx = b % sg.tx, by = (b / sg.tx) % sg.ty, bz = b / (sg.tx * sg.ty);
  int x = bx * out + lx - halo, y = by * out + ly - halo, z = bz * out + lz - halo;
  auto within = [&](int t) {
    return lx >= t && lx < EDGE - t && ly >= t && ly < EDGE - t && lz >= t && lz < EDGE - t;
  };
  const bool stored = within(halo) && x < g.nx && y < g.ny && z < g.nz;
  bool in = true;
  auto wrap = [&](int v, int n, int periodic) -> int {
    if (v >= 0 && v < n) return v;
    if (!periodic) {
      in = false;
      return 0;
    }
    return ((v % n) + n) % n;
  };
  CellPos c;
  c.x = wrap(x, g.nx, g.px);
  c.y = wrap(y, g.ny, g.py);
  c.z = wrap(z, g.nz, g.pz);
  c.i = stored_index(g, c.x, c.y, c.z);
  const uint32_t w = in ? words[c.i] : 0u;
  const int32_t k = CPL ? idx[c.i] : -1;
  if constexpr (WALLS) {
    if (tid < MAX_CLASSES) classes[tid] = bc.table[tid];
    __syncthreads();
    bc.table = classes;
  }
  const CellAddr<AOS> A = cell_addr<AOS>(g, c);
  bool fl = (w & FLUID) != 0;
  T f[Q];
  if (fl) {
#pragma unroll
    for (int q = 0; q < Q; q++) f[q] = src[((w >> (Q - 1 - q)) & 1u) ? A.own(Q - 1 - q) : A.pull(q)];
  }
  for (int t = 0;;) {
    if (fl) {
      if (CPL && k >= 0) couple_cell<T, WALLS>(f, cpl, k, c.i, w, bc);
      else collide_cell_bc<T, FORCE, ALPHA, WALLS, M32>(f, w, c.i, alpha, p64, p32, bc);
    }
    if (++t == sg.steps) break;
    if (fl) {
#pragma unroll
      for (int q = 0; q < Q; q++)
        if (q != REST) lds[q * CELLS + tid] = f[q];
    }
    __syncthreads();
    fl = fl && within(t);
    if (fl) {
#pragma unroll
      for (int q = 0; q < Q; q++) {
        if (q == REST) continue;
        const bool bounce = (w >> (Q - 1 - q)) & 1u;
        f[q] = lds[bounce ? (Q - 1 - q) * CELLS + tid : q * CELLS + tid - (CX(q) + EDGE * CY(q) + EDGE * EDGE * CZ(q))];
      }
    }
    __syncthreads();
  }
  if (fl && stored) {
#pragma unroll
    for (int q = 0; q < Q; q++) dst[A.own(q)] = f[q];
  }
}

struct SmallArgs {
  const void* src;
  void* dst;
  const uint32_t* words;
  const void* alpha;
  bool force, walls;
  CollideParams p64;
  CollideParams32 p32;
  BoundaryArgs bc;
  CoupleArgs cpl;
  const int32_t *idx, *boxes;  // coupled boxes, or null
  int nboxes;
};

template <typename T, bool M32, bool AOS>
hipError_t small_t(const DenseGeom& g, const SmallGeom& sg, const SmallArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.boxes ? a.nboxes : sg.tx * sg.ty * sg.tz)), block(CELLS);
#define LBM_SMALL_C(F, A, W, C)                                                                                    \
  hipLaunchKernelGGL((k_dense_small<T, F, A, W, C, M32, AOS>), grid, block, 0, s, g, sg, (const T*)a.src,           \
                     (T*)a.dst, a.words, (const T*)a.alpha, a.p64, a.p32, a.bc, a.cpl, a.idx, a.boxes)
#define LBM_SMALL(F, A, W) LBM_SMALL_C(F, A, W, false)
  if (a.boxes) {
    if (a.walls) LBM_SMALL_C(false, false, true, true);
    else LBM_SMALL_C(false, false, false, true);
    return hipGetLastError();
  }
  const int key = (a.force ? 4 : 0) | (a.alpha ? 2 : 0) | (a.walls ? 1 : 0);
  switch (key) {
    case 0: LBM_SMALL(false, false, false); break;
    case 1: LBM_SMALL(false, false, true); break;
    case 2: LBM_SMALL(false, true, false); break;
    case 3: LBM_SMALL(false, true, true); break;
    case 4: LBM_SMALL(true, false, false); break;
    case 5: LBM_SMALL(true, false, true); break;
    case 6: LBM_SMALL(true, true, false); break;
    default: LBM_SMALL(true, true, true); break;
  }
#undef LBM_SMALL
#undef LBM_SMALL_C
  return hipGetLastError();
}

template <bool AOS>
hipError_t small_type(const DenseGeom& g, const SmallGeom& sg, bool fp32, bool f32math, const SmallArgs& a, hipStream_t s) {
  if (fp32 && f32math) return small_t<float, true, AOS>(g, sg, a, s);
  if (fp32) return small_t<float, false, AOS>(g, sg, a, s);
  return small_t<double, false, AOS>(g, sg, a, s);
}

SmallGeom small_geom(const DenseGeom& g, int steps) {
  const int out = EDGE - 2 * (steps - 1);
  return SmallGeom{steps, (g.nx + out - 1) / out, (g.ny + out - 1) / out, (g.nz + out - 1) / out};
}

}  // namespace

// As many steps as leave every CU at most one box.  With two boxes a CU the work done twice costs what the
// launches save: 32^3 (512 boxes at three steps) FP64 periodic 5.2 us a step in single steps, 5.6 here, lid 6.2
// and 6.2; two steps a launch (216 boxes) 5.8 and 5.8.  48^3 10.2 and 14.8.  Below the line more steps are
// better: 12^3 FP64 lid 4.5, 3.7 and 3.3 us at two, three and four.
int small_steps(const DenseGeom& g) {
  for (int steps = 4; steps > 2; steps--) {
    const SmallGeom sg = small_geom(g, steps);
    if ((int64_t)sg.tx * sg.ty * sg.tz <= NCU) return steps;
  }
  return 1;
}

hipError_t launch_dense_small(const DenseGeom& g, int steps, bool fp32, bool f32math, const void* src, void* dst,
                              const uint32_t* words, const void* alpha, bool force, bool walls, const CollideParams& p64,
                              const CollideParams32& p32, const BoundaryArgs& bc, hipStream_t s) {
  const SmallGeom sg = small_geom(g, steps);
  const SmallArgs a{src, dst, words, alpha, force, walls, p64, p32, bc, CoupleArgs{}, nullptr, nullptr, 0};
  return g.aos ? small_type<true>(g, sg, fp32, f32math, a, s) : small_type<false>(g, sg, fp32, f32math, a, s);
}

std::vector<int32_t> small_box_list(const DenseGeom& g, const int64_t* cells, int64_t n) {
  const SmallGeom sg = small_geom(g, 2);
  const int64_t nboxes = (int64_t)sg.tx * sg.ty * sg.tz;
  std::vector<int32_t> list;
  if (nboxes > INT32_MAX) return list;
  const int out = EDGE - 2;
  // the boxes of v - 1, v and v + 1 along one axis (at most three, where the axis wraps)
  auto near = [&](int v, int size, int periodic, int (&at)[3]) {
    int m = 0;
    for (int d = -1; d <= 1; d++) {
      int w = v + d;
      if (w < 0 || w >= size) {
        if (!periodic) continue;
        w = w < 0 ? size - 1 : 0;
      }
      bool known = false;
      for (int j = 0; j < m; j++) known = known || at[j] == w / out;
      if (!known) at[m++] = w / out;
    }
    return m;
  };
  std::vector<uint8_t> taken((size_t)nboxes, 0);
  for (int64_t k = 0; k < n; k++) {
    const int64_t r = cells[k];
    int ax[3], ay[3], az[3];
    const int mx = near((int)(r % g.nx), g.nx, g.px, ax), my = near((int)((r / g.nx) % g.ny), g.ny, g.py, ay),
              mz = near((int)(r / ((int64_t)g.nx * g.ny)), g.nz, g.pz, az);
    for (int c = 0; c < mz; c++)
      for (int b = 0; b < my; b++)
        for (int a = 0; a < mx; a++) taken[(size_t)(ax[a] + (int64_t)sg.tx * (ay[b] + (int64_t)sg.ty * az[c]))] = 1;
  }
  for (int64_t b = 0; b < nboxes; b++)
    if (taken[(size_t)b]) list.push_back((int32_t)b);
  return list;
}

hipError_t launch_coupled_boxes(const DenseGeom& g, bool fp32, bool f32math, const void* src, void* dst,
                                const uint32_t* words, bool walls, const CollideParams& p64, const CollideParams32& p32,
                                const BoundaryArgs& bc, const CoupleArgs& cpl, const int32_t* idx, const int32_t* boxes,
                                int nboxes, hipStream_t s) {
  const SmallGeom sg = small_geom(g, 2);
  const SmallArgs a{src, dst, words, nullptr, false, walls, p64, p32, bc, cpl, idx, boxes, nboxes};
  return g.aos ? small_type<true>(g, sg, fp32, f32math, a, s) : small_type<false>(g, sg, fp32, f32math, a, s);
}

}  // namespace lbm
