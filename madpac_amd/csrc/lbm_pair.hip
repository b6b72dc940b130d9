// Two time steps in one launch on the two-buffer dense lattice (pull form): k_dense_pair.
//
// The one-step kernel reads and writes the state once per step and is bound by HBM.  Here a workgroup
// owns a column of TX x TY cells (its tile) over a chunk of planes and sweeps z upwards.  For each plane
// it pulls and collides the tile's cells and the ring of cells around them (first step), hands the
// results to their receivers through the LDS, and then collides the plane below, which has received
// everything by now (second step), and stores it: the state is read once and written once per two steps.
// The price is the ring, computed twice: 128 of 640 threads (32 x 16), 192 of 704 (64 x 8).
//
//  * A cell pushes its populations to the receiving column's slots, or across a bounce-back link to its
//    own mirrored slot, so the second step reads its own column only.  Populations that stay in the
//    column (0, 0, +-1) and the rest population pass through registers.
//  * Slots come in two sets, by the parity of the receiving plane.  The rising side populations of plane
//    k are complete after plane k's pushes and are read then, one plane early; a third set would not
//    fit two steps of 512 FP64 columns (2 x 16 x 528 x 8 B = 135 KB).
//  * The next plane's pulls are issued before the barriers and fly while the second step computes.
//  * All addresses are a uniform base per plane and population plus one of nine 32-bit per-lane offsets,
//    so the loads and stores cost no vector instructions beyond themselves.
//  * Every cell goes through the same collide_cell_bc as in the one-step kernel: the same bits.
//
// Tiles measured per step on 256^3 (all-fluid FP64 / porous FP64 bricks): 32 x 16 545 / 596 us, 64 x 8
// 526 / 619, 32 x 8 (two workgroups per CU) 674 / 812, one-step kernel 917 / 859.  FP32 all-fluid rows: 64 x 8
// 315 us, 32 x 16 336, 32 x 24 383, 32 x 8 369, one-step 442.  At 256^3 FP64 a pair moves 5.3 GB (fetched
// 1.08 x the state, counters) at 4.9 TB/s; vector issue is 33 % busy (FP32: 55 %), and each plane has a
// latency of 4 us (FP32 3.2 us) even on an idle chip.  Loading the next plane a whole pass ahead (FP32,
// +19 registers) and loading it only after the second step (for more workgroups per CU) were slower.
#include <algorithm>
#include <climits>

#include "lbm_collide.h"

namespace lbm {

namespace {

// Slot of a population that crosses a tile column's sides, in the LDS (the pure z movers and the rest
// population stay in registers).
__host__ __device__ constexpr int SLOT(int q) {
  return q < 2 ? q : q < 5 ? q - 1 : q < 9 ? q - 1 : q < 14 ? q - 2 : q < 16 ? q - 2 : q - 3;
}
constexpr int SLOTS = 16;
constexpr int SPARE = 16;  // values per slot that take the pushes leaving the tile

template <int TX, int TY>
struct Tile {
  static constexpr int INNER = TX * TY;
  static constexpr int RING = 2 * (TX + 2) + 2 * TY;
  static constexpr int THREADS = INNER + (RING + 63) / 64 * 64;
  static constexpr int STRIDE = INNER + SPARE;
};

// orders the LDS only: the global loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename T>
__device__ __forceinline__ T ld(const T* base, uint32_t byte_off) {
  return *(const T*)((const char*)base + byte_off);
}

template <typename T, bool FORCE, bool ALPHA, bool WALLS, bool M32, bool AOS, int TX, int TY>
__global__ __launch_bounds__((Tile<TX, TY>::THREADS), 3) void k_dense_pair(
    DenseGeom g, PairGeom pg, const T* __restrict__ src, T* __restrict__ dst, const uint32_t* __restrict__ words,
    const T* __restrict__ alpha, CollideParams p64, CollideParams32 p32, BoundaryArgs bc) {
  using Sh = Tile<TX, TY>;
  __shared__ T lds[2 * SLOTS * Sh::STRIDE];
  // the boundary classes, kept near: from global memory, a classed cell's mask and target were two more
  // round trips in each of a plane's two collisions (channel 131 x 70 x 53 FP64 37.7 -> 36.4 us a step)
  __shared__ BoundaryClass classes[WALLS ? MAX_CLASSES : 1];
  const int tid = (int)threadIdx.x;
  // XCD-contiguous ranges of tiles (x fastest, then y, then the z chunks)
  const int64_t bid = blockIdx.x;
  const int64_t b = (bid % NXCD) * (pg.nblocks_padded / NXCD) + bid / NXCD;
  if (b >= pg.nblocks) return;
  if constexpr (WALLS) {
    if (tid < MAX_CLASSES) classes[tid] = bc.table[tid];
    __syncthreads();
    bc.table = classes;
  }
  const int tx = (int)(b % pg.tx), ty = (int)((b / pg.tx) % pg.ty), tz = (int)(b / ((int64_t)pg.tx * pg.ty));
  const int x0 = tx * TX, y0 = ty * TY, z0 = tz * pg.cz, z1 = min(g.nz, z0 + pg.cz);
  const int vx = min(TX, g.nx - x0), vy = min(TY, g.ny - y0);

  // this thread's column of the tile, (rx, ry) in [-1, vx] x [-1, vy]
  const bool inner = tid < Sh::INNER;
  int rx, ry;
  bool act;
  if (inner) {
    if (g.bricked) {  // 16 consecutive lanes = one 4 x 4 layer of a brick
      const int grp = tid >> 4;
      rx = (grp % (TX / 4)) * 4 + (tid & 3);
      ry = (grp / (TX / 4)) * 4 + ((tid >> 2) & 3);
    } else {
      rx = tid % TX;
      ry = tid / TX;
    }
    act = rx < vx && ry < vy;
  } else {
    int r = tid - Sh::INNER;
    const int row = vx + 2;
    act = r < 2 * row + 2 * vy;
    if (r < 2 * row) {
      ry = r < row ? -1 : vy;
      rx = (r < row ? r : r - row) - 1;
    } else {
      r -= 2 * row;
      rx = r < vy ? -1 : vx;
      ry = r < vy ? r : r - vy;
    }
  }
  int x = x0 + rx, y = y0 + ry;
  if (x < 0 || x >= g.nx) {
    act = act && g.px;
    x = x < 0 ? g.nx - 1 : 0;
  }
  if (y < 0 || y >= g.ny) {
    act = act && g.py;
    y = y < 0 ? g.ny - 1 : 0;
  }
  if (!act) x = y = 0;

  // Addresses: a uniform part per plane and population, and one per-lane byte offset for each of the
  // nine columns around this one.
  auto term_x = [&](int v) -> int64_t { return AOS ? aos_term_x(g, v) : g.bricked ? brick_term_x(v) : (int64_t)v; };
  auto term_y = [&](int v) -> int64_t {
    return AOS ? aos_term_y(g, v) : g.bricked ? brick_term_y(g, v) : (int64_t)g.nx * v;
  };
  const int zsh = g.bricked ? 2 : 0, zmask = g.bricked ? 3 : 0;  // planes share a layer of bricks
  const int64_t layer = g.bricked ? (int64_t)64 * g.bnx * g.bny : (int64_t)g.nx * g.ny;
  auto cell_z = [&](int z) -> int64_t { return (z >> zsh) * layer + ((z & zmask) << 4); };
  auto term_z = [&](int z) -> int64_t { return (z >> zsh) * (AOS ? Q * layer : layer) + ((z & zmask) << 4); };
  auto pop = [&](int q) -> int64_t { return AOS ? (int64_t)(64 * q) : q * g.N; };
  uint32_t col[3][3];  // [y - 1, y, y + 1][x - 1, x, x + 1], clamped where no neighbour is
  {
    const int xm = x == 0 ? (g.px ? g.nx - 1 : 0) : x - 1, xp = x == g.nx - 1 ? (g.px ? 0 : x) : x + 1;
    const int ym = y == 0 ? (g.py ? g.ny - 1 : 0) : y - 1, yp = y == g.ny - 1 ? (g.py ? 0 : y) : y + 1;
    const int64_t ax[3] = {term_x(xm), term_x(x), term_x(xp)}, ay[3] = {term_y(ym), term_y(y), term_y(yp)};
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) col[j][i] = (uint32_t)((ax[i] + ay[j]) * (int64_t)sizeof(T));
  }
  const int64_t cell_xy = g.bricked ? brick_term_x(x) + brick_term_y(g, y) : (int64_t)x + (int64_t)g.nx * y;

  // LDS positions of the eight columns around this one (and its own); a spare value where the tile ends
  auto lds_index = [&](int cx, int cy) -> int {
    if (cx < 0 || cx >= TX || cy < 0 || cy >= TY) return Sh::INNER + (tid & (SPARE - 1));
    if (!g.bricked) return cx + TX * cy;
    return (((cy >> 2) * (TX / 4) + (cx >> 2)) << 4) + ((cy & 3) << 2) + (cx & 3);
  };
  int to[3][3];  // byte addresses in the set of the current plane's parity
#pragma unroll
  for (int j = 0; j < 3; j++)
#pragma unroll
    for (int i = 0; i < 3; i++) to[j][i] = lds_index(rx + i - 1, ry + j - 1) * (int)sizeof(T);
  auto slot = [&](int addr, int q) -> T& { return *(T*)((char*)lds + addr + SLOT(q) * Sh::STRIDE * (int)sizeof(T)); };

  // the plane that k stands for (wrapped; clamped to the box where z is not periodic)
  auto plane_of = [&](int k) -> int {
    const int lo = g.pz ? g.nz - 1 : 0, hi = g.pz ? 0 : g.nz - 1;
    return k < 0 ? lo : k >= g.nz ? hi : k;
  };
  auto load_word = [&](int k) -> uint32_t {
    const bool in = g.pz || (k >= 0 && k < g.nz);
    const uint32_t w = words[cell_z(plane_of(k)) + cell_xy];
    return (in && act) ? w : 0u;
  };
  // the populations of the reference state that plane k's cell collides
  auto load_cell = [&](int k, uint32_t w, T(&f)[Q]) {
    const int z = plane_of(k);
    const T *sz = src + term_z(z), *sm = src + term_z(plane_of(z - 1)), *sp = src + term_z(plane_of(z + 1));
    if (!(w & FLUID)) return;
#pragma unroll
    for (int q = 0; q < Q; q++)
      f[q] = ld((CZ(q) > 0 ? sm : CZ(q) < 0 ? sp : sz) + pop(q), col[1 - CY(q)][1 - CX(q)]);
    if (w & 0x7FFFFu) {
#pragma unroll
      for (int q = 0; q < Q; q++)
        if (q != REST && ((w >> (Q - 1 - q)) & 1u)) f[q] = ld(sz + pop(Q - 1 - q), col[1][1]);
    }
  };

  T f[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) f[q] = T(0);
  uint32_t w = load_word(z0 - 1), wn = load_word(z0), wp = 0;
  load_cell(z0 - 1, w, f);
  T r9 = T(0), r16 = T(0), s16 = T(0);
  T up[4] = {T(0), T(0), T(0), T(0)};  // rising side populations of plane k - 1
  int other = SLOTS * Sh::STRIDE * (int)sizeof(T);  // from the set of plane k's parity to the other set
  for (int k = z0 - 1; k <= z1; k++) {
    // opaque copies: what follows from these alone would be kept in registers over the whole sweep
#pragma unroll
    for (int d = 0; d < 3; d++) asm volatile("" : "+s"(p64.g[d]));
    asm volatile("" : "+s"(p64.omega), "+s"(p64.tau_eff), "+s"(p32.fpref));
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) asm volatile("" : "+v"(to[j][i]), "+v"(col[j][i]));
    if (w & FLUID) collide_cell_bc<T, FORCE, ALPHA, WALLS, M32>(f, w, cell_z(plane_of(k)) + cell_xy, alpha, p64, p32, bc);
    if (w & FLUID) {
      if (w & 0x7FFFFu) {
#pragma unroll
        for (int q = 0; q < Q; q++) {
          if (CX(q) == 0 && CY(q) == 0) continue;
          const int out = to[1 + CY(q)][1 + CX(q)] + (CZ(q) ? other : 0) + SLOT(q) * Sh::STRIDE * (int)sizeof(T);
          const int own = to[1][1] + SLOT(Q - 1 - q) * Sh::STRIDE * (int)sizeof(T);
          *(T*)((char*)lds + (((w >> q) & 1u) ? own : out)) = f[q];
        }
      } else {
#pragma unroll
        for (int q = 0; q < Q; q++) {
          if (CX(q) == 0 && CY(q) == 0) continue;
          slot(to[1 + CY(q)][1 + CX(q)] + (CZ(q) ? other : 0), q) = f[q];
        }
      }
    }
    const T c2 = f[2], c9 = f[REST], c16 = f[16];
    const uint32_t wc = w;
    w = wn;
    if (k < z1) {
      load_cell(k + 1, w, f);
      wn = k + 1 < z1 ? load_word(k + 2) : 0u;
    }
    lds_barrier();  // plane k - 1 has received everything
    const int p = k - 1;
    const bool out = inner && p >= z0, fl = out && (wp & FLUID) != 0;
    T h[Q];
    if (fl) {
#pragma unroll
      for (int q = 0; q < 14; q++) {
        if (CX(q) == 0 && CY(q) == 0) continue;
        h[q] = slot(to[1][1] + other, q);
      }
      h[14] = up[0];
      h[15] = up[1];
      h[17] = up[2];
      h[18] = up[3];
      h[REST] = r9;
      h[16] = r16;
      h[2] = ((wp >> 16) & 1u) ? s16 : c2;
    }
    if (inner && (wc & FLUID)) {
      up[0] = slot(to[1][1], 14);
      up[1] = slot(to[1][1], 15);
      up[2] = slot(to[1][1], 17);
      up[3] = slot(to[1][1], 18);
    }
    lds_barrier();  // plane k - 1 has been read
    const unsigned long long fluid = __ballot(fl);
    if (out && act && (fl || line_has_fluid<T>(fluid))) {
      if (fl) collide_cell_bc<T, FORCE, ALPHA, WALLS, M32>(h, wp, cell_z(p) + cell_xy, alpha, p64, p32, bc);
      T* dz = dst + term_z(p);
      if (g.cached_pair) {
        asm volatile("");
#pragma unroll
        for (int q = 0; q < Q; q++) *(T*)((char*)(dz + pop(q)) + col[1][1]) = fl ? h[q] : T(0);
        asm volatile("");
      } else {
#pragma unroll
        for (int q = 0; q < Q; q++) __builtin_nontemporal_store(fl ? h[q] : T(0), (T*)((char*)(dz + pop(q)) + col[1][1]));
      }
    }
    r16 = ((wc >> 2) & 1u) ? c2 : s16;
    r9 = c9;
    s16 = c16;
    wp = wc;
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) to[j][i] += other;
    other = -other;
  }
}

// Chunks of planes.  One workgroup runs on a CU at a time (registers and, in FP64, LDS), so the grid runs
// in rounds of NCU workgroups, and a workgroup's time is its planes plus two (its neighbours' planes that
// it recomputes) plus about one plane's time to fill its pipeline.  The chunk count with the least
// rounds x (planes + 3): 256^3 two chunks of 128 planes (256 workgroups, one round; FP64 528 us a step;
// 543 at four chunks, 562 at eight), 128 x 128 x 96 eight chunks of 12 (56 us; 74 in four chunks, 64 at
// 24), 64^3 32 chunks of 2 (13.2 us; 16.2 in 16 chunks).
constexpr int NCU = 256;

PairGeom pair_geom(const DenseGeom& g, int tile_x, int tile_y) {
  PairGeom p;
  p.tile_x = tile_x;
  p.tx = (g.nx + tile_x - 1) / tile_x;
  p.ty = (g.ny + tile_y - 1) / tile_y;
  const int64_t tiles = (int64_t)p.tx * p.ty;
  p.passes = INT64_MAX;
  // (beyond eight rounds, shorter chunks only add planes computed twice)
  const int64_t most = std::min<int64_t>(g.nz, 8 * NCU / std::min<int64_t>(tiles, NCU));
  for (int n = 1; n <= most; n++) {
    const int cz = (g.nz + n - 1) / n;
    const int64_t rounds = (tiles * ((g.nz + cz - 1) / cz) + NCU - 1) / NCU, cost = rounds * (cz + 3);
    if (cost < p.passes) {
      p.passes = cost;
      p.cz = cz;
    }
  }
  p.tz = (g.nz + p.cz - 1) / p.cz;
  p.nblocks = tiles * p.tz;
  p.nblocks_padded = (p.nblocks + NXCD - 1) / NXCD * NXCD;
  return p;
}

template <typename T, bool M32, bool AOS, int TX, int TY>
hipError_t pair_t(const DenseGeom& g, const PairGeom& pg, const void* src, void* dst, const uint32_t* words, const void* alpha, bool force,
                  bool walls, const CollideParams& p64, const CollideParams32& p32, const BoundaryArgs& bc, hipStream_t s) {
  const dim3 grid((unsigned)pg.nblocks_padded), block(Tile<TX, TY>::THREADS);
#define LBM_PAIR(F, A, W)                                                                                        \
  hipLaunchKernelGGL((k_dense_pair<T, F, A, W, M32, AOS, TX, TY>), grid, block, 0, s, g, pg, (const T*)src, (T*)dst, \
                     words, (const T*)alpha, p64, p32, bc)
  const int key = (force ? 4 : 0) | (alpha ? 2 : 0) | (walls ? 1 : 0);
  switch (key) {
    case 0: LBM_PAIR(false, false, false); break;
    case 1: LBM_PAIR(false, false, true); break;
    case 2: LBM_PAIR(false, true, false); break;
    case 3: LBM_PAIR(false, true, true); break;
    case 4: LBM_PAIR(true, false, false); break;
    case 5: LBM_PAIR(true, false, true); break;
    case 6: LBM_PAIR(true, true, false); break;
    default: LBM_PAIR(true, true, true); break;
  }
#undef LBM_PAIR
  return hipGetLastError();
}

template <typename T, bool M32, bool AOS>
hipError_t pair_tile(const DenseGeom& g, const PairGeom& pg, const void* src, void* dst, const uint32_t* words, const void* alpha, bool force,
                     bool walls, const CollideParams& p64, const CollideParams32& p32, const BoundaryArgs& bc,
                     hipStream_t s) {
  if (pg.tile_x == 32)
    return pair_t<T, M32, AOS, 32, 16>(g, pg, src, dst, words, alpha, force, walls, p64, p32, bc, s);
  return pair_t<T, M32, AOS, 64, 8>(g, pg, src, dst, words, alpha, force, walls, p64, p32, bc, s);
}

template <bool AOS>
hipError_t pair_type(const DenseGeom& g, const PairGeom& pg, bool fp32, bool f32math, const void* src, void* dst, const uint32_t* words,
                     const void* alpha, bool force, bool walls, const CollideParams& p64, const CollideParams32& p32,
                     const BoundaryArgs& bc, hipStream_t s) {
  if (fp32 && f32math)
    return pair_tile<float, true, AOS>(g, pg, src, dst, words, alpha, force, walls, p64, p32, bc, s);
  if (fp32) return pair_tile<float, false, AOS>(g, pg, src, dst, words, alpha, force, walls, p64, p32, bc, s);
  return pair_tile<double, false, AOS>(g, pg, src, dst, words, alpha, force, walls, p64, p32, bc, s);
}

}  // namespace

PairSplits pair_splits(const DenseGeom& g) { return PairSplits{pair_geom(g, 64, 8), pair_geom(g, 32, 16)}; }

// The rule weighs two launches of the one-step kernel against one of this kernel, in microseconds.
//  * One step: 3, a boundary's 1, and its bytes at 5.3 TB/s (7 where the caches hold them, state_cached), with half
//    of the lanes that rows leave idle, and a fifth more where rows do not start on 128-byte lines; of the
//    solid cells' bytes a half (where the caches hold them, none).
//  * This kernel: its planes in sequence (PairGeom::passes), each a latency: loads, two collisions, two
//    barriers.  Force, porosity and boundary classes lengthen the collisions, open boundaries most: their
//    cells' two equilibria per link hold up the whole workgroup.  Past the Infinity Cache (two states of 200 MB),
//    the FP32 planes with force or porosity take longer (not with FP32 arithmetic), as FP64 ones with solids do.
// Measured per step in long runs, one-step / this kernel, us:
//               periodic       lid            channel *      porous *       porosity
//   FP64 64^3   14.1 / 12.3    15.0 / 14.0    16.4 / 18.9    15.3 / 17.0    14.3 / 15.8     (* with a tenth of
//   80^3        31.0 / 21.6    30.9 / 22.0    33.5 / 29.7    34.5 / 31.3    30.4 / 25.3      the cells solid, at
//   131x70x53   31.4 / 21.5    32.5 / 24.9    36.4 / 33.2    36.8 / 32.8    32.6 / 28.7      random; porous: and
//   128^3        111 / 74       113 / 76       117 / 91       112 / 93       114 / 82        a force)
//   1000x1000x2  119 / 91       124 / 89       124 / 97       130 / 138      120 / 92
//   240^3        820 / 502      816 / 520      843 / 643      838 / 640      838 / 590
//   FP32 96^3   26.3 / 23.4    27.7 / 27.0    30.7 / 35.7    32.7 / 30.4    28.7 / 28.5
//   112^3       37.2 / 35.8    42.8 / 43.4    47.3 / 58.3    51.3 / 48.1    45.7 / 46.3
//   128^3       56.3 / 47.6    55.9 / 50.4    63.2 / 66.8    60.7 / 56.5    56.2 / 55.5
//   192x192x96  93.4 / 87.9    93.0 / 89.6     101 / 119      100 / 106     94.4 / 100
//   240^3        437 / 359      437 / 378      472 / 516      472 / 416      445 / 402
// The microseconds of a plane follow from these and 550 other runs.  Of what the rule sends here, two are more than
// 3 % slower than single steps: FP64 rows of 8 cells in a box of thousands of planes (8 x 8 x 8192 porous 112 /
// 90 us; the idle lanes are overrated there) and FP64 porosity on 72^3 (27.0 / 26.1).  Runs that start from a
// state in memory gain less: the forward sweep of the adjoint with its checkpoints takes on 128^3 FP32 59.7 us a step
// here and 57.6 in single steps, 128^3 FP64 83 and 113, 160^3 FP32 118 and 128.
//  * With the MD coupling this kernel is followed by the boxes around the coupled cells (lbm_small.hip): 16 us
//    and 45 ns a box (96^3 FP64: 14 us for 8 boxes, 23 for 216, 35 for 512, 173 for 3294), where a single step
//    is followed by its re-collision, 7.5 us.  Per step, single / this way: 96^3 FP64 24^3 coupled cells 66.5 /
//    52.3, 3000 scattered ones 74 / 127; 128^3 FP32 24^3 coupled cells 66.8 / 62.5.
//  * Two tiles of 512 columns, 64 x 8 and 32 x 16; where both need as many planes 64 x 8 is the faster one
//    by 5 % (32 x 16 in FP64 bricks, by 4 %: head of this file), but rows of 80, 96 or 160 cells leave it half
//    empty at their end.  A step in 64 x 8 / 32 x 16: FP64 80^3 force and porosity 30.8 / 24.4, 96^3 (13 and 10
//    planes) lid 40.0 / 34.5, channel 50.9 / 42.3, 160^3 (43 and 35) 155 / 145; FP32 160^3 118 / 105.
// A plane of populations has to fit the 32-bit offsets.
bool pair_plan(const DenseGeom& g, const PairSplits& splits, size_t esize, bool f32math, int64_t nfluid, bool extra,
               bool walls, bool open, int coupled_boxes, PairGeom* plan) {
  const int64_t plane = g.bricked ? (int64_t)64 * g.bnx * g.bny : (int64_t)g.nx * g.ny;
  if (plane * (g.aos ? Q : 1) * (int64_t)esize > (int64_t)UINT32_MAX) return false;
  const bool f64 = esize == 8;
  const PairGeom &wide = splits.wide, &tall = splits.tall;
  const bool bricks = f64 && g.bricked;
  const double t_wide = (double)wide.passes * (bricks ? 1.04 : 1.0), t_tall = (double)tall.passes * (bricks ? 1.0 : 1.05);
  *plan = t_tall < t_wide ? tall : wide;
  const double bytes = (double)Q * (double)g.N * (double)esize;
  const bool held = g.cached && bytes <= 125e6;
  double cells = held ? (double)nfluid : 0.5 * ((double)nfluid + (double)g.Nu);
  if (!g.bricked) {
    cells *= 0.5 + 0.5 * ((g.nx + 63) / 64 * 64) / g.nx;
    if ((g.nx * esize) % 128) cells *= 1.2;
  }
  const double step = 3.0 + (walls ? 1.0 : 0.0) + cells * 2 * Q * (double)esize / (held ? 7.0e6 : 5.3e6);
  const double more = f64 ? (nfluid < g.Nu && !held ? 6.8 : 6.2) : (!f32math && bytes > 200e6 ? 6.5 : 5.7);
  const double pass = open ? (f64 ? 8.0 : 8.5) : extra ? more : walls ? (f64 ? 5.9 : 5.7) : (f64 ? 5.2 : 5.1);
  const double two = std::min(t_wide, t_tall) * pass;
  return coupled_boxes ? two + 16.0 + 0.045 * coupled_boxes < 2.0 * (step + 7.5) : two < 2.0 * step;
}

hipError_t launch_dense_pair(const DenseGeom& g, const PairGeom& pg, bool fp32, bool f32math, const void* src, void* dst,
                             const uint32_t* words, const void* alpha, bool force, bool walls, const CollideParams& p64,
                             const CollideParams32& p32, const BoundaryArgs& bc, hipStream_t s) {
  return g.aos ? pair_type<true>(g, pg, fp32, f32math, src, dst, words, alpha, force, walls, p64, p32, bc, s)
               : pair_type<false>(g, pg, fp32, f32math, src, dst, words, alpha, force, walls, p64, p32, bc, s);
}

}  // namespace lbm
