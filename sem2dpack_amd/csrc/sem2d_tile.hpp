// Fused tile kernels for structured (MESH_CART) meshes.
//
// Fields live in node-grid order: node (X, Z) of the (4nx+1) x (4nz+1[+1]) GLL grid
// at index Z*NX1 + X (a split fault duplicates one grid row).  The element grid is
// cut into tiles of up to TX x TZ elements; one workgroup owns one tile and, in a
// single pass over HBM, does for the tile's patch of (4*nxe+1) x (4*nze+1) nodes:
//
//   1. load d, v, a; Newmark predictor (SRC/solver.f90:59-60), or, between the steps of a
//      call, the predicted state itself (StepOut); predicted d in LDS;
//   2. element forces f = -K d (ELAST_KD2_*, SRC/mat_elastic.f90:589-641,739-775),
//      summed per node in the order of the 2x2 checkerboard colours of the tile's
//      elements (no atomics, the summation order is fixed);
//   3. interior patch nodes: a = f*rmass, corrector (SRC/solver.f90:78-82), store;
//      patch-perimeter nodes and "special" nodes (point sources): store the
//      partial force of this tile to fpart and leave the node untouched.
//
// k_deferred then finishes every perimeter / special node: it sums the partial
// forces of the tiles that share it (fixed tile order), adds sources and absorbing
// boundaries (in BC order) and applies the corrector; the nodes of a split fault get
// there by pairs, with the traction solve in between.  k_run_steps does both for many
// steps of a small grid in one launch.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sem2d_commit.hpp"
#include "sem2d_fault.hpp"
#include "sem2d_kernels.hpp"

namespace sem2d {

constexpr int TX = 8, TZ = 8;
constexpr int PXM = 4 * TX + 1, PZM = 4 * TZ + 1;
constexpr int PMAX = PXM * PZM;
constexpr int PERIM_MAX = 2 * PXM + 2 * (PZM - 2);
constexpr int MAXSPECIAL = 16;
constexpr int SLOTS = PERIM_MAX + MAXSPECIAL;

struct TileDev {
  int ntiles;
  const int4* tiles;  // (tx0, tz0, nxe | nze << 8 | nx << 16, Z0), nx = elements per grid row
  const int4* grids;  // per tile: (node_base, ROW, NZ1, cell_base) of the grid the tile lies in
  const int* spec_cnt;
  const int* spec_idx;  // [ntiles][MAXSPECIAL] patch indices Z*PXM + X
  size_t NGp;           // component stride of the field arrays
  size_t FPS;           // component stride of fpart (ntiles*SLOTS)
};

// Storage index of patch node (X, Z) of the tile at (X0, Z0) whose left and right
// columns lie on vertical tile-edge lines kL and kR.  A grid of NZ1 node rows starting
// at node_base stores, row after row, the nodes strictly between its vertical
// tile-edge lines: each tile column's 4*TX-1 nodes in a segment of 4*TX slots (ROW
// slots per row), so that the segments start on cache-line boundaries; the nodes of
// the tile-edge lines follow column by column (NZ1 each, unit stride along Z).
// Several grids (one per scenario of a batch) can share the field arrays, each at its
// own node_base.
__device__ __forceinline__ size_t node_index(const int4 gr, int X, int Z, int PX, int X0, int Z0, int kL,
                                             int kR) {
  const size_t base = (size_t)gr.x, grid = (size_t)gr.y * gr.z;
  if (X == 0) return base + grid + (size_t)kL * gr.z + (Z0 + Z);
  if (X == PX - 1) return base + grid + (size_t)kR * gr.z + (Z0 + Z);
  return base + (size_t)(Z0 + Z) * gr.y + X0 + X - 1;
}

// element (cell) index of local element (lx, lz) of a tile at (tx0, tz0).  The
// fourth descriptor field is the grid's first cell for per-cell coefficients; with
// shared coefficients (one element array per grid) it is the offset of the grid's
// array instead and the cell index is not used.
__device__ __forceinline__ size_t cell_index(const int4 gr, int nx, int tx0, int tz0, int lx, int lz) {
  return (size_t)gr.w + (size_t)(tz0 + lz) * nx + tx0 + lx;
}

__device__ __forceinline__ int perim_slot(int X, int Z, int PX, int PZ) {
  // branch-free form of: Z == 0 -> X; Z == PZ-1 -> PX + X; X == 0 -> 2PX + Z-1;
  // X == PX-1 -> 2PX + PZ-2 + Z-1; otherwise -1
  int s = X == PX - 1 ? 2 * PX + (PZ - 2) + (Z - 1) : -1;
  s = X == 0 ? 2 * PX + (Z - 1) : s;
  s = Z == PZ - 1 ? PX + X : s;
  s = Z == 0 ? X : s;
  return s;
}

// LDS node value of NDOF components stored together (one vector access for P-SV)
template <typename R, int N>
struct LVec {
  using T = R;
};
template <typename R>
struct LVec<R, 2> {
  typedef R T __attribute__((ext_vector_type(2)));
};
template <typename R, int N>
__device__ __forceinline__ typename LVec<R, N>::T lv_make(const R* x) {
  if constexpr (N == 2) return typename LVec<R, N>::T{x[0], x[1]};
  else return x[0];
}
template <typename R, int N>
__device__ __forceinline__ R lv_get(const typename LVec<R, N>::T& v, int c) {
  if constexpr (N == 2) return c == 0 ? v.x : v.y;
  else return v;
}

// Element i of an array below 4 GiB, addressed as a uniform base plus a 32-bit byte
// offset (the scalar-base / vector-offset form of the memory instructions, with no
// 64-bit address arithmetic per access).
template <typename T>
__device__ __forceinline__ T& at32(T* base, uint32_t i) {
  using C = std::conditional_t<std::is_const<T>::value, const char, char>;
  return *reinterpret_cast<T*>(reinterpret_cast<C*>(base) + i * (uint32_t)sizeof(T));
}

// p, as a value the compiler cannot look through: a uniform base kept in scalar
// registers, so that base + 32-bit offset is not re-associated into 64-bit vector
// address arithmetic
template <typename T>
__device__ __forceinline__ T* sgpr_base(T* p) {
  using G = __attribute__((address_space(1))) T*;  // global memory
  G g = (G)p;
  asm("" : "+s"(g));
  return (T*)g;
}

// Order of LDS accesses among the lanes of one wavefront (which the hardware executes in
// program order): no access moves across it.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exchange slots of the forces of the elements at a patch node (X, Z), node Z * PXM + X of
// the table (slot = element * NP + point, elements row by row of a full tile; slot NEL * NP
// stands for an element outside the patch).  Of the two element columns (rows) that share a
// node the even one comes first, rows before columns: the order of the colours.  A table
// that the kernels copy to LDS behind their first loads: computed there it was some 600
// instructions of a lane before the tile's first load.
struct alignas(8) NodeSlots {
  unsigned short q[4];
};
struct SlotTable {
  NodeSlots node[PMAX];
};
constexpr SlotTable make_slot_table() {
  SlotTable T{};
  for (int Z = 0; Z < PMAX / PXM; ++Z)
    for (int X = 0; X < PXM; ++X)
      for (int q = 0; q < 4; ++q) {
        const int cx = q & 1, cz = q >> 1;
        const int lx = ((X >> 2) & 1) == cx ? X >> 2 : (X >> 2) - 1;
        const int lz = ((Z >> 2) & 1) == cz ? Z >> 2 : (Z >> 2) - 1;
        const bool ok = lx >= 0 && lx < TX && (lx == X >> 2 || (X & 3) == 0) && lz >= 0 && lz < TZ &&
                        (lz == Z >> 2 || (Z & 3) == 0);
        T.node[Z * PXM + X].q[q] =
            (unsigned short)(ok ? (lz * TX + lx) * NP + (Z - 4 * lz) * NG + (X - 4 * lx) : TX * TZ * NP);
      }
  return T;
}
__device__ const SlotTable c_slots = make_slot_table();

// Element phase of the tile kernels: element e, its lane s (row or column s), base the patch
// index of its first node, ex its part of the exchange array; on: the element is inside the
// grid.  Between the four steps the lanes of an element exchange through ex (wave_order).
// A: column s, d/deta of its nodes' displacement (EP: of d + eta v)
template <typename R, int NDOF, bool EP, typename LV>
__device__ __forceinline__ void el_gradient(bool on, int base, int s, int e, LV* ex, const LV* Ud, const LV* Vp,
                                            const R* Eta, const R (&H)[NG][NG]) {
  constexpr int PS = PXM;
  if (on) {
    R g[NG][NDOF];
#pragma unroll
    for (int j = 0; j < NG; ++j)
#pragma unroll
      for (int c = 0; c < NDOF; ++c) g[j][c] = 0;
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const LV x = Ud[base + k * PS + s];
      LV y{};
      R et = 0;
      if constexpr (EP) {
        y = Vp[base + k * PS + s];
        et = Eta[e * NP + k * NG + s];
      }
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        R xc = lv_get<R, NDOF>(x, c);
        if constexpr (EP) xc = xc + et * lv_get<R, NDOF>(y, c);
#pragma unroll
        for (int j = 0; j < NG; ++j) g[j][c] += xc * H[k][j];
      }
    }
#pragma unroll
    for (int j = 0; j < NG; ++j) ex[j * NG + s] = lv_make<R, NDOF>(g[j]);
  }
}
// B: row s, the fluxes at its points: the eta fluxes into ex, the row's xi sums into s1r
template <typename R, int NDOF, int NELAST, int MODE, bool EP, typename LV, typename M, typename F>
__device__ __forceinline__ void el_flux(bool on, int base, int s, int e, LV* ex, const LV* Ud, const LV* Vp,
                                        const R* Eta, const R (&H)[NG][NG], const R (*Gm)[3], const R* sW2,
                                        const R* Sa, const LV* Mn, const M& m, F coef, R (&s1r)[NG][NDOF]) {
  constexpr int PS = PXM;
  if (on) {
    R x[NG][NDOF];
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const LV xv = Ud[base + s * PS + k];
      LV y{};
      R et = 0;
      if constexpr (EP) {
        y = Vp[base + s * PS + k];
        et = Eta[e * NP + s * NG + k];
      }
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        x[k][c] = lv_get<R, NDOF>(xv, c);
        if constexpr (EP) x[k][c] = x[k][c] + et * lv_get<R, NDOF>(y, c);
        s1r[k][c] = 0;
      }
    }
    R g0 = 0, g1 = 0, g2 = 0;
    if constexpr (MODE == COEF_COMPACT || MODE == COEF_NODE || MODE == COEF_ELEM) {
      g0 = Gm[e][0];
      g1 = Gm[e][1];
      g2 = Gm[e][2];
    }
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int pt = s * NG + i;
      R A[NELAST];
      if constexpr (MODE == COEF_COMPACT || MODE == COEF_NODE || MODE == COEF_ELEM) {
        const R w2 = sW2[pt];
        R m0, m1;
        if constexpr (MODE == COEF_NODE) {
          const LV mm = Mn[base + s * PS + i];
          m0 = lv_get<R, NDOF>(mm, 0);
          m1 = lv_get<R, NDOF>(mm, NDOF - 1);
        } else {
          m0 = m[MODE == COEF_ELEM ? 0 : i][0];
          m1 = m[MODE == COEF_ELEM ? 0 : i][NDOF - 1];
        }
        if constexpr (NDOF == 2) {
          const R la = m0, mu = m1, kx = la + 2 * mu;
          A[0] = w2 * kx * g0;
          A[1] = w2 * la * g2;
          A[2] = w2 * kx * g1;
          A[3] = w2 * mu * g1;
          A[4] = w2 * mu * g2;
          A[5] = w2 * mu * g0;
        } else {
          A[0] = w2 * m0 * g0;
          A[1] = w2 * m0 * g1;
        }
      } else if constexpr (MODE == COEF_SHARED) {
#pragma unroll
        for (int k = 0; k < NELAST; ++k) A[k] = Sa[k * NP + pt];
      } else {
#pragma unroll
        for (int k = 0; k < NELAST; ++k) A[k] = coef(k, pt);
      }
      R dxi[NDOF], deta[NDOF];
      const LV gv = ex[pt];
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        R sum = 0;
#pragma unroll
        for (int k = 0; k < NG; ++k) sum += H[k][i] * x[k][c];
        dxi[c] = sum;
        deta[c] = lv_get<R, NDOF>(gv, c);
      }
      R t1[NDOF], t2[NDOF];
      if constexpr (NDOF == 2) {
        t1[0] = A[0] * dxi[0] + A[1] * deta[1];
        t2[0] = A[3] * (deta[0] + dxi[1]);
        t1[1] = A[4] * deta[0] + A[5] * dxi[1];
        t2[1] = A[1] * dxi[0] + A[2] * deta[1];
      } else {
        t1[0] = A[0] * dxi[0];
        t2[0] = A[1] * deta[0];
      }
      ex[pt] = lv_make<R, NDOF>(t2);
#pragma unroll
      for (int q = 0; q < NG; ++q)
#pragma unroll
        for (int c = 0; c < NDOF; ++c) s1r[q][c] += H[q][i] * t1[c];
      // one point at a time: hoisting the later points' LDS reads costs the registers
      // of the next tile's loads
      if constexpr (MODE != COEF_SHARED) __builtin_amdgcn_sched_barrier(0);
    }
  }
}
// C: column s, the eta sums of the fluxes
template <typename R, int NDOF, typename LV>
__device__ __forceinline__ void el_divergence(bool on, int s, LV* ex, const R (&H)[NG][NG]) {
  if (on) {
    R g[NG][NDOF];
#pragma unroll
    for (int j = 0; j < NG; ++j)
#pragma unroll
      for (int c = 0; c < NDOF; ++c) g[j][c] = 0;
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const LV tv = ex[k * NG + s];
#pragma unroll
      for (int j = 0; j < NG; ++j)
#pragma unroll
        for (int c = 0; c < NDOF; ++c) g[j][c] += lv_get<R, NDOF>(tv, c) * H[j][k];
    }
#pragma unroll
    for (int j = 0; j < NG; ++j) ex[j * NG + s] = lv_make<R, NDOF>(g[j]);
  }
}
// D: row s, the forces of its points (slot: an element outside the grid, zero)
template <typename R, int NDOF, bool EP, typename LV>
__device__ __forceinline__ void el_force(bool on, bool slot, bool b25, int base, int s, int e, LV* ex, const LV* Ud,
                                         const LV* Vp, const R* Eta, const R* Bet, const R (&s1r)[NG][NDOF]) {
  constexpr int PS = PXM;
  if (on) {
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const LV c2v = ex[s * NG + i];
      R f[NDOF];
#pragma unroll
      for (int c = 0; c < NDOF; ++c) f[c] = s1r[i][c] + lv_get<R, NDOF>(c2v, c);
      if constexpr (EP) {
        if (b25) {  // 2.5D: the point force loses b25 (d + eta v) of its own point
          const int own = base + s * PS + i;
          const LV uo = Ud[own], wo = Vp[own];
          const R eo = Eta[e * NP + s * NG + i], bo = Bet[e * NP + s * NG + i];
#pragma unroll
          for (int c = 0; c < NDOF; ++c)
            f[c] = f[c] - bo * (lv_get<R, NDOF>(uo, c) + eo * lv_get<R, NDOF>(wo, c));
        }
      }
      ex[s * NG + i] = lv_make<R, NDOF>(f);
    }
  } else if (slot) {
#pragma unroll
    for (int i = 0; i < NG; ++i) ex[s * NG + i] = LV{};
  }
}

// Touches the cache lines of H that hconst reads as scalars.
template <typename R>
__device__ __forceinline__ void warm_h() {
  const auto* hp = hconst<R>();
  const R a = hp[0], b = hp[8], c = hp[16], d = hp[24];
  asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d));
}

// Persistent tile kernel.  Each workgroup walks a strided sequence of tiles inside its
// XCD's share (see below); the state a tile reads is loaded into registers while the
// previous tile is processed.
//
// Element phase: a lane per element row or column, 12 elements (60 lanes) per wavefront,
// 6 wavefronts for the 64 elements of a tile.  Five points per lane make the entries of H
// compile-time indices (scalar operands), and the two directions of an element are
// exchanged through LDS between lanes of the same wavefront, without a barrier:
//   A  column i:  deta(i, .) from the column's nodes, to the exchange array
//   B  row j:     dxi(., j) from the row's nodes, stresses of the row's points, the row
//                 part of the forces (kept in registers), the column fluxes to the array
//   C  column i:  the column part of the forces
//   D  row j:     both parts added: the element's forces
//   E  (barrier)  every node adds the forces of its 1, 2 or 4 elements, in the order of
//                 the 2x2 checkerboard of colours
// An element costs 300 LDS accesses of a node value where a lane per point took 650
// (10 + 2 + 10 + 4 per point), and a tile two barriers instead of five.
//
// Bound by HBM latency and bandwidth: P-SV with moduli per node, 1000 x 500 elements, moves
// 0.70 GB (FP64) per step in 182 us and half of it (FP32) in 117 us with the deferred nodes'
// kernel (3.9 and 3.0 TB/s; a large copy reaches 5.0); with a lane per point and (d, v, a)
// handed on it was 283 and 140 us.  Two workgroups per CU overlap one's loads with the
// other's phases; they fit only while a wavefront needs 128 registers at most, and a
// spilled register costs more than it saves (the spill of a prefetched value waits for it):
// FP64 with 34 registers spilled took 290 us.
//
// Per tile:
//   1. the predicted displacement goes to LDS (the state read is the predicted one, PIN:
//      nothing to compute), from loads issued an element phase earlier;
//   2. the loads of this tile's predicted velocity (needed by its stores only), then of the
//      next tile's displacement and moduli are issued;
//   3. phases A and B; the inverse mass is loaded, which only the stores need; phases C, D
//      and E;
//   4. the tile's stores, which complete during the next tile's phases.
// Vector memory operations retire in issue order, loads and stores in one counter, so
// that a wait for a load also waits for what was issued before it: the order above has
// each wait behind the longest stretch of work.
// Tile descriptors are scalar loads, counted apart from vector memory.  The patch is laid
// out with the row length of a full tile whatever the tile's size, so that the index
// arithmetic has constant divisors; a smaller tile leaves slots and lanes idle.
//
// W32: the field, inverse-mass, partial-force and per-cell arrays are below 4 GiB per
// component and are addressed with 32-bit offsets from per-component bases.
//
// EP: element-point terms, per element point in cell order [cell][25] (either may be
// null): Kelvin-Voigt viscosity eta, the element displacement being d + eta v at each
// point (MAT_KV_add_etav, SRC/mat_kelvin_voigt.f90:139-150), and the 2.5D coefficient
// b25, the point force then losing b25 (d + eta v) (MAT_ELAST_add_25D_f,
// SRC/mat_elastic.f90:447-459).  The predicted velocity then passes through LDS.
constexpr int TS_NT = 384;                  // threads per workgroup
constexpr int TS_EPW = 12;                  // elements per wavefront (5 lanes each)
constexpr int TS_ITER = (PMAX + TS_NT - 1) / TS_NT;  // patch nodes per thread
static_assert(TS_EPW * (TS_NT / 64) >= TX * TZ, "not enough wavefronts for a tile's elements");
static_assert(3 * TX * TZ <= TS_NT, "per-tile tables larger than the workgroup");

constexpr int MARK_WORDS = (PMAX + 31) / 32;

// Arguments of k_tile_step.  The kernel reads them from the argument segment where it uses
// them (kernel_args): kept in scalar registers throughout, next to the 25 entries of H,
// they would not fit, and the compiler spills scalars to vector registers.
template <typename R>
struct TileArgs {
  R *d, *v, *a;
  const R *din, *vin, *ain;  // state read by an out-of-place step; null vin / ain: v / a
  const R *rmass0, *coefs, *geom, *eta, *b25;
  R *fpart, *rec;  // rec: where recorded nodes go (StepOut::rec)
  size_t S, FPS;  // component strides of the field arrays and of fpart
  const int4 *tiles, *grids;
  const int *spec_cnt, *spec_idx;
  // recorded nodes inside tiles: per tile its row of marks (or -1), MARK_WORDS words each
  const int* mark_of;
  const uint32_t* marks;
  int* tick;  // device step counter moved to this step, or null
  int ntiles;
  R dt, c1, c2, c3, c4;
  StepOut out;
};
// entry i (uniform) of an array that no kernel writes: a scalar load
__device__ __forceinline__ int sload(const int* p, int i) {
  return ((const __attribute__((address_space(4))) int*)p)[i];
}
__device__ __forceinline__ int4 sload(const int4* p, int i) {
  typedef int I4 __attribute__((ext_vector_type(4)));
  const I4 x = ((const __attribute__((address_space(4))) I4*)p)[i];
  return make_int4(x.x, x.y, x.z, x.w);
}
// the argument struct of a kernel whose only parameter it is, by a pointer the compiler
// cannot look through (so that loads from it are not merged across uses)
template <typename A>
__device__ __forceinline__ const __attribute__((address_space(4))) A* kernel_args() {
  auto p = (const __attribute__((address_space(4))) A*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// Launched with TS_NT threads.  The bound of 512 makes the compiler count two workgroups of
// eight wavefronts per CU, that is 128 registers; two of six would seem to admit 168, but
// the dispatcher may place four wavefronts of two workgroups on one SIMD.
template <typename R, int NDOF, int NELAST, int MODE, bool OOP = false, bool W32 = true, bool EP = false,
          bool PIN = false>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(EP || (!PIN && NDOF == 2 && sizeof(R) == 8) ? 2 : 4))) void
k_tile_step(TileArgs<R> args) {
  constexpr int PS = PXM;        // patch row length
  constexpr int NEL = TX * TZ;   // element slots
  constexpr bool NODEM = MODE == COEF_NODE;
  constexpr bool COMP = MODE == COEF_COMPACT || MODE == COEF_ELEM;
  constexpr int NM = MODE == COEF_COMPACT ? NG : 1;  // moduli of a row's points, or the element's
  // FULLPF: the registers admit the prefetch of everything a tile reads but per-element
  // moduli, and of a tile's forces until the next tile's loads have arrived.  Otherwise
  // (FP64 P-SV) the predicted velocity and the inverse mass, which only the stores need,
  // are loaded late (LATEV), and the stores follow the forces.
  constexpr bool FULLPF = (sizeof(R) == 4 || NDOF == 1) && !EP;
  constexpr bool LATEV = PIN && !EP && !FULLPF;
  // node values with both components side by side: one LDS access moves both
  using LV = typename LVec<R, NDOF>::T;
  __shared__ LV Ud[PMAX];               // predicted displacement
  // exchange array: deta, column fluxes, forces; the last slot stays zero
  __shared__ LV Ex[NEL * NP + 1];
  // per patch node the exchange slots of its elements' forces, in the order of the
  // colours; the zero slot stands for an element outside the patch
  __shared__ NodeSlots Eg[PMAX];
  __shared__ LV Vp[EP ? PMAX : 1];      // predicted velocity
  __shared__ LV Mn[NODEM ? PMAX : 1];   // moduli of the patch nodes
  __shared__ R Sa[MODE == COEF_SHARED ? NELAST * NP : 1];  // the grid's point coefficients
  __shared__ R Gm[NEL][3];              // geometric factors of the elements
  __shared__ R sW2[NP];
  constexpr int NEPT = EP ? NEL * NP : 1;  // eta and b25 of the tile's element points
  __shared__ R Eta[NEPT];
  __shared__ R Bet[NEPT];

  const int nlist = args.ntiles;
  const int nwg = gridDim.x;
  const int bid = blockIdx.x;
  // Workgroups reach the 8 XCDs round-robin (XCD = bid & 7).  XCD x owns the x-th
  // eighth of the listed tiles [s0, s1); its W workgroups take them interleaved
  // (workgroup k: s0 + k, s0 + k + W, ...), so at any time one XCD works on consecutive
  // tiles and the cache lines and halo nodes shared by x-neighbours are fetched once
  // into its L2.
  const int W = nwg >> 3;  // nwg is a multiple of 8
  const int slice = (nlist + 7) >> 3;
  const int s0 = (bid & 7) * slice;
  const int s1 = min(s0 + slice, nlist);
  const int q0 = s0 + (bid >> 3);
  if (args.tick && bid == 0 && threadIdx.x == 0) ++*args.tick;
  if (q0 >= s1) return;
  const int tid = threadIdx.x;
  // this thread's patch nodes (X, Z), packed
  int xz[TS_ITER];
#pragma unroll
  for (int r = 0; r < TS_ITER; ++r) {
    const int p = tid + TS_NT * r, Z = p / PS, X = p - Z * PS;
    xz[r] = X | Z << 8;
  }
  struct Geo {
    int tx0, tz0, nxe, nze, Z0, PX, PZ, X0, kL, kR;
  };
  auto geo = [&](const int4 tg) {
    Geo g;
    g.tx0 = tg.x;
    g.tz0 = tg.y;
    g.nxe = tg.z & 0xff;
    g.nze = (tg.z >> 8) & 0xff;
    g.Z0 = tg.w;
    g.PX = 4 * g.nxe + 1;
    g.PZ = 4 * g.nze + 1;
    g.X0 = 4 * g.tx0;
    g.kL = g.tx0 / TX;
    g.kR = (g.tx0 + g.nxe + TX - 1) / TX;
    return g;
  };
  // storage index of patch node (X, Z), as node_index: a tile-edge column or a row segment
  auto nidx = [&](const int4 gr, const Geo& G, int X, int Z) {
    using I = std::conditional_t<W32, uint32_t, size_t>;
    const I row = (I)gr.x + (I)G.Z0 * (I)gr.y + (I)(G.X0 - 1);            // uniform
    const I edge = (I)gr.x + (I)gr.y * (I)gr.z + (I)G.Z0;                 // uniform
    const I eL = edge + (I)G.kL * (I)gr.z, eR = edge + (I)G.kR * (I)gr.z;  // uniform
    const I in = row + (I)((uint32_t)Z * (uint32_t)gr.y + (uint32_t)X);
    const I ed = (X == 0 ? eL : eR) + (I)Z;
    return X == 0 || X == G.PX - 1 ? ed : in;
  };
  auto fld = [&](auto* cbase, auto g) -> auto& {
    if constexpr (W32) return at32(cbase, (uint32_t)g);
    else return cbase[g];
  };
  auto ubase = [&](auto* p) {
    if constexpr (W32) return sgpr_base(p);
    else return p;
  };
  auto cidx = [&](const int4 gr, int nx, const Geo& G, int lx, int lz) {
    if constexpr (W32) return (uint32_t)gr.w + (uint32_t)(G.tz0 + lz) * (uint32_t)nx + (uint32_t)(G.tx0 + lx);
    else return cell_index(gr, nx, G.tx0, G.tz0, lx, lz);
  };

  // lane index the compiler cannot look through: index arithmetic derived from it is
  // recomputed where it is used rather than held in registers across tiles
  auto lane_id = [&]() {
    int q = tid;
    asm volatile("" : "+v"(q));
    __builtin_assume(q >= 0 && q < TS_NT);
    return q;
  };

  // registers of the next tile, issued in one group at the start of the current tile's
  // element phase.  Slots outside the patch load its nearest node: with loads under a
  // condition the registers' old values would have to be kept for the other lanes.
  constexpr int NEP = EP ? (NEL * NP + TS_NT - 1) / TS_NT : 1;
  R pd[TS_ITER][NDOF] = {}, pv[LATEV ? 1 : TS_ITER][NDOF] = {}, pa[PIN ? 1 : TS_ITER][NDOF] = {};
  R pmod[NODEM ? TS_ITER : 1][NDOF] = {}, pm[FULLPF ? TS_ITER : 1] = {};
  R peta[NEP] = {}, pbet[NEP] = {};
  R psa = 0, pg = 0;
  auto issue = [&](int t) {
    const auto* P = kernel_args<TileArgs<R>>();
    const int4 tg = sload(P->tiles, t);
    const int4 gr = sload(P->grids, t);
    const Geo G = geo(tg);
    const R *bD[NDOF], *bV[NDOF], *bA[NDOF], *bMo[NDOF];
#pragma unroll
    for (int c = 0; c < NDOF; ++c) {
      const size_t o = c * P->S;
      bD[c] = ubase((OOP ? P->din : P->d) + o);
      bV[c] = ubase((OOP && P->vin ? P->vin : P->v) + o);
      bA[c] = ubase((OOP && P->ain ? P->ain : P->a) + o);
      bMo[c] = NODEM ? ubase(P->coefs + o) : nullptr;
    }
    const R* bRm = ubase(P->rmass0);
    const R* bCo = ubase(P->coefs);
    const R* bGe = ubase(P->geom);
    const R* bEt = EP && P->eta ? ubase(P->eta) : nullptr;
    const R* bBe = EP && P->b25 ? ubase(P->b25) : nullptr;
    const int nx = tg.z >> 16;
    const int tl = lane_id();
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const auto g = nidx(gr, G, min(xz[r] & 0xff, G.PX - 1), min(xz[r] >> 8, G.PZ - 1));
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        pd[r][c] = fld(bD[c], g);
        if constexpr (!LATEV) pv[r][c] = fld(bV[c], g);
        if constexpr (!PIN) pa[r][c] = fld(bA[c], g);
        if constexpr (NODEM) pmod[r][c] = fld(bMo[c], g);
      }
      if constexpr (FULLPF) pm[r] = fld(bRm, g);
    }
    if constexpr (COMP || NODEM) {
      const int e = tl / 3, k = tl - 3 * (tl / 3);
      const int lx = min(e % TX, G.nxe - 1), lz = min(e / TX, G.nze - 1);
      pg = fld(bGe, cidx(gr, nx, G, lx, lz) * 3 + k);
    }
    if constexpr (MODE == COEF_SHARED) {
      psa = bCo[gr.w + min(tl, NELAST * NP - 1)];
    }
    if constexpr (EP) {
#pragma unroll
      for (int j = 0; j < NEP; ++j) {
        const int q = tl + TS_NT * j;
        const int e = q / NP, o = q - e * NP;
        const auto cell = cidx(gr, nx, G, min(e % TX, G.nxe - 1), min(e / TX, G.nze - 1));
        peta[j] = bEt ? fld(bEt, cell * NP + o) : R(0);
        pbet[j] = bBe ? fld(bBe, cell * NP + o) : R(0);
      }
    }
  };

  // predicted velocity and inverse mass of the tile's nodes, for its stores
  R wk[EP ? 1 : TS_ITER][NDOF] = {}, rk[TS_ITER] = {};

  // Stores of a finished tile: partial forces for perimeter and special nodes, new a, v,
  // d for the others.
  auto store_tile = [&](const int tp, const int4 tgp, const int4 grp, const int ns, const int mark,
                        const R (*fk)[NDOF]) {
    const auto* P = kernel_args<TileArgs<R>>();
    const Geo G = geo(tgp);
    R *oD[NDOF], *oV[NDOF], *oA[NDOF], *bF[NDOF];
#pragma unroll
    for (int c = 0; c < NDOF; ++c) {
      const size_t o = c * P->S;
      oD[c] = ubase(P->d + o);
      oV[c] = ubase(P->v + o);
      oA[c] = ubase(P->a + o);
      bF[c] = ubase(P->fpart + c * P->FPS);
    }
    const R c3 = P->c3, c4 = P->c4, dt = P->dt, c1 = P->c1, c2 = P->c2;
    const StepOut so = {P->out.final, P->out.accel, P->out.rec};
    const int mrow = so.rec >= 0 ? mark : -1;
    const uint32_t fbase = (uint32_t)tp * SLOTS;
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const int X = xz[r] & 0xff, Z = xz[r] >> 8;
      if (X < G.PX && Z < G.PZ) {
        int slot = perim_slot(X, Z, G.PX, G.PZ);
        for (int k = 0; k < ns; ++k)  // a handful of tiles have special nodes
          if (sload(P->spec_idx, tp * MAXSPECIAL + k) == tid + TS_NT * r) slot = PERIM_MAX + k;
        if (slot >= 0) {
#pragma unroll
          for (int c = 0; c < NDOF; ++c) fld(bF[c], fbase + slot) = fk[r][c];
        } else {
          const auto g = nidx(grp, G, X, Z);
          const LV u = Ud[tid + TS_NT * r];
#pragma unroll
          for (int c = 0; c < NDOF; ++c) {
            const R ak = fk[r][c] * rk[r];
            const R vn = (EP ? lv_get<R, NDOF>(Vp[EP ? tid + TS_NT * r : 0], c) : wk[EP ? 0 : r][c]) + c3 * ak;
            const R dn = lv_get<R, NDOF>(u, c) + c4 * ak;
            if (so.final) {
              fld(oA[c], g) = ak;
              fld(oV[c], g) = vn;
              fld(oD[c], g) = dn;
            } else {
              fld(oV[c], g) = vn + c2 * ak;
              fld(oD[c], g) = dn + dt * vn + c1 * ak;
              if (so.accel) fld(oA[c], g) = ak;
              if (mrow >= 0) {  // few tiles hold recorded nodes
                const int p = tid + TS_NT * r;
                if (P->marks[mrow * MARK_WORDS + (p >> 5)] >> (p & 31) & 1)
                  fld(ubase(P->rec + c * P->S), g) = so.rec == 0 ? dn : (so.rec == 1 ? vn : ak);
              }
            }
          }
        }
      }
    }
  };

  issue(q0);
  // behind the first tile's loads: the exchange slots, the GLL weights, and the lines of H,
  // which the element phase reads as scalars, into the scalar cache
#pragma unroll
  for (int r = 0; r < TS_ITER; ++r)
    if (const int p = tid + TS_NT * r; p < PMAX) Eg[p] = c_slots.node[p];
  if (tid < NP) sW2[tid] = (R)c_W2[tid];
  if (tid == 0) Ex[NEL * NP] = LV{};
  warm_h<R>();
  int tp = -1;  // FULLPF: the previous tile of this workgroup, not yet stored
  int4 tgp = {}, grp = {};
  int nsp = 0, markp = -1;
  R fk[TS_ITER][NDOF] = {};

#pragma unroll 1
  for (int qi = q0; qi < s1; qi += W) {
    const int t = qi;
    const int tn = qi + W < s1 ? qi + W : -1;  // next tile of this workgroup
    const auto* P = kernel_args<TileArgs<R>>();
    const int4 tg = sload(P->tiles, t);
    const int4 gr = sload(P->grids, t);
    // for the stores (there the loads would be waited for: they are the tile's first)
    const int ns = sload(P->spec_cnt, t), mark = sload(P->mark_of, t);
    const Geo G = geo(tg);
    const R dt = P->dt, c1 = P->c1, c2 = P->c2;

    // the moduli of the points of this lane's row (element phase below), ahead of the waits
    // for the tile's node values
    R m[NM][NDOF];
    if constexpr (COMP) {
      const int tl = lane_id(), lane = tl & 63;
      const int e = min((tl >> 6) * TS_EPW + lane / NG, NEL - 1), s = lane % NG;
      const R* bCo = ubase(P->coefs);
      const auto cell = cidx(gr, tg.z >> 16, G, min(e % TX, G.nxe - 1), min(e / TX, G.nze - 1));
#pragma unroll
      for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int c = 0; c < NDOF; ++c)
          m[i][c] = fld(bCo, NM == 1 ? cell * NDOF + c : (cell * NDOF + c) * NP + s * NG + i);
    }

    // predictor
    R u[TS_ITER][NDOF], w[TS_ITER][NDOF];
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r)
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        if constexpr (PIN) {
          u[r][c] = pd[r][c];
          if constexpr (!LATEV) w[r][c] = pv[r][c];
        } else {
          u[r][c] = pd[r][c] + dt * pv[r][c] + c1 * pa[r][c];
          w[r][c] = pv[r][c] + c2 * pa[r][c];
        }
      }
    if constexpr (FULLPF) {
      // the waits for this tile's loads stay ahead of the previous tile's stores
#pragma unroll
      for (int r = 0; r < TS_ITER; ++r) {
#pragma unroll
        for (int c = 0; c < NDOF; ++c) asm volatile("" : "+v"(u[r][c]), "+v"(w[r][c]));
        asm volatile("" : "+v"(pm[r]));
      }
      if (tp >= 0) store_tile(tp, tgp, grp, nsp, markp, fk);
    }
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const int p = tid + TS_NT * r;
      if (p < PMAX) {
        Ud[p] = lv_make<R, NDOF>(u[r]);
        if constexpr (EP) Vp[p] = lv_make<R, NDOF>(w[r]);
        if constexpr (NODEM) Mn[p] = lv_make<R, NDOF>(pmod[r]);
      }
      if constexpr (!LATEV && !EP) {
#pragma unroll
        for (int c = 0; c < NDOF; ++c) wk[r][c] = w[r][c];
      }
      if constexpr (FULLPF) rk[r] = pm[r];
    }
    if constexpr (COMP || NODEM) {
      if (tid < NEL * 3) Gm[tid / 3][tid - 3 * (tid / 3)] = pg;
    }
    if constexpr (MODE == COEF_SHARED) {
      if (tid < NELAST * NP) Sa[tid] = psa;
    }
    if constexpr (EP) {
#pragma unroll
      for (int j = 0; j < NEP; ++j)
        if (tid + TS_NT * j < NEPT) {
          Eta[tid + TS_NT * j] = peta[j];
          Bet[tid + TS_NT * j] = pbet[j];
        }
    }
    __syncthreads();

    // element phase: element e, row or column s
    {
      const int tl = lane_id(), lane = tl & 63;
      const int e = (tl >> 6) * TS_EPW + lane / NG, s = lane % NG;
      const int lx = e % TX, lz = e / TX;
      const bool on = lane < TS_EPW * NG && e < NEL && lx < G.nxe && lz < G.nze;
      const int base = 4 * lz * PS + 4 * lx;
      LV* ex = Ex + e * NP;
      if (tn >= 0) {
        issue(tn);
      } else {  // no old values to keep
#pragma unroll
        for (int r = 0; r < TS_ITER; ++r)
#pragma unroll
          for (int c = 0; c < NDOF; ++c) {
            pd[r][c] = 0;
            if constexpr (!LATEV) pv[r][c] = 0;
            if constexpr (!PIN) pa[r][c] = 0;
          }
        if constexpr (NODEM) {
#pragma unroll
          for (int r = 0; r < TS_ITER; ++r)
#pragma unroll
            for (int c = 0; c < NDOF; ++c) pmod[r][c] = 0;
        }
        if constexpr (FULLPF) {
#pragma unroll
          for (int r = 0; r < TS_ITER; ++r) pm[r] = 0;
        }
        pg = psa = 0;
      }

      // H as scalar operands, read once per tile
      const auto* hp = hconst<R>();
      R H[NG][NG];
#pragma unroll
      for (int k = 0; k < NG; ++k)
#pragma unroll
        for (int i = 0; i < NG; ++i) H[k][i] = hp[k * NG + i];
      el_gradient<R, NDOF, EP>(on, base, s, e, ex, Ud, Vp, Eta, H);
      wave_order();
      R s1r[NG][NDOF];
      el_flux<R, NDOF, NELAST, MODE, EP>(on, base, s, e, ex, Ud, Vp, Eta, H, Gm, sW2, Sa, Mn, m,
                                         [&](int k, int pt) {
                                           return fld(ubase(P->coefs),
                                                      (cidx(gr, tg.z >> 16, G, lx, lz) * NELAST + k) * NP + pt);
                                         },
                                         s1r);
      wave_order();
      // what the stores need besides the forces, loaded when the registers of B are free
      // and used after C, D and E
      if constexpr (!FULLPF) {
        const R* bRm = ubase(P->rmass0);
        const R* bV[NDOF];
#pragma unroll
        for (int c = 0; c < NDOF; ++c) bV[c] = ubase((OOP && P->vin ? P->vin : P->v) + c * P->S);
#pragma unroll
        for (int r = 0; r < TS_ITER; ++r) {
          const auto g = nidx(gr, G, min(xz[r] & 0xff, G.PX - 1), min(xz[r] >> 8, G.PZ - 1));
          rk[r] = fld(bRm, g);
          if constexpr (LATEV) {
#pragma unroll
            for (int c = 0; c < NDOF; ++c) wk[r][c] = fld(bV[c], g);
          }
        }
      }
      el_divergence<R, NDOF>(on, s, ex, H);
      wave_order();
      el_force<R, NDOF, EP>(on, lane < TS_EPW * NG && e < NEL, EP && P->b25, base, s, e, ex, Ud, Vp, Eta, Bet, s1r);
    }
    __syncthreads();
    // E: nodes (elements outside the tile left zero)
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const int p = tid + TS_NT * r;
#pragma unroll
      for (int c = 0; c < NDOF; ++c) fk[r][c] = 0;
      if (p < PMAX) {
        const NodeSlots sl = Eg[p];
        const LV f0 = Ex[sl.q[0]], f1 = Ex[sl.q[1]], f2 = Ex[sl.q[2]], f3 = Ex[sl.q[3]];
#pragma unroll
        for (int c = 0; c < NDOF; ++c)
          fk[r][c] = (((lv_get<R, NDOF>(f0, c)) + lv_get<R, NDOF>(f1, c)) + lv_get<R, NDOF>(f2, c)) +
                     lv_get<R, NDOF>(f3, c);
      }
    }
    if constexpr (FULLPF) {
      tp = t;
      tgp = tg;
      grp = gr;
      nsp = ns;
      markp = mark;
    } else {
      store_tile(t, tg, gr, ns, mark, fk);
    }
  }
  if constexpr (FULLPF) {
    if (tp >= 0) store_tile(tp, tgp, grp, nsp, markp, fk);
  }
}

// One deferred node: tile-perimeter, special or split-fault node.
struct DefNode {
  int g;        // grid index
  int pstart;   // partial offsets part_off[pstart .. pstart+pcnt)
  int pcnt;
  int sstart;   // sources src[sstart .. sstart+scnt)
  int scnt;
  int astart;   // absorbing coefficients abso[astart .. astart+acnt), [ndof] each
  int acnt;
  int fault;    // 1: split-fault node (finished with its pair)
  int dmask;    // Dirichlet components zeroed in the force (bit c: component c), after the
                // absorbing terms; at a fault node, those of the Dirichlet boundaries that
                // act before the fault
  int rec;      // recorded node (StepOut::rec)
  int rec_at;   // its first entry in the receiver list (RecOut), or -1
  int pinl;     // device form only: 1 when the two partial offsets are poff (pcnt == 2)
  int poff[2];  // the second is -1 when pcnt == 1
};

// Device form of a deferred-node list: 16 bytes per node (one vector load) plus a side
// table for the few nodes with sources, absorbing terms or receivers.  cnt packs pcnt (bits 0-7),
// scnt (bits 8-15), acnt (bits 16-23), fault (bit 24), "offsets inline" (bit 25), the
// Dirichlet mask (bits 26-27) and "recorded" (bit 28); x
// is the node's (sstart, astart, rec_at, -) entry in ext, or -1 when it has none of them.  A node with
// one or two partial forces and no ext entry (a tile-edge node, most nodes of the general
// path) holds its partial offsets in pstart and x instead (bit 25 set), so part_off is not
// read for it.
struct alignas(16) DefDev {
  int g, pstart, cnt, x;
};
struct DefTable {
  const DefDev* node = nullptr;
  const int4* ext = nullptr;
};
__device__ __forceinline__ DefNode def_unpack(const DefTable& D, const DefDev e) {
  DefNode n;
  n.g = e.g;
  n.pstart = e.pstart;
  n.pcnt = e.cnt & 0xff;
  n.scnt = (e.cnt >> 8) & 0xff;
  n.acnt = (e.cnt >> 16) & 0xff;
  n.fault = (e.cnt >> 24) & 1;
  n.pinl = (e.cnt >> 25) & 1;
  n.dmask = (e.cnt >> 26) & 3;
  n.rec = (e.cnt >> 28) & 1;
  n.sstart = 0;
  n.astart = 0;
  n.rec_at = -1;
  n.poff[0] = n.poff[1] = 0;
  if (n.pinl) {
    n.poff[0] = e.pstart;
    n.poff[1] = e.x;
  } else if (e.x >= 0) {
    const int4 x = D.ext[e.x];
    n.sstart = x.x;
    n.astart = x.y;
    n.rec_at = x.z;
  }
  return n;
}
__device__ __forceinline__ DefNode def_unpack(const DefTable& D, int q) { return def_unpack(D, D.node[q]); }

// Stacey terms of the absorbing entries of the deferred nodes: entry q (the q-th
// absorbing coefficient set of the step, in boundary order) subtracts kxd[idx[t]],
// t = off[q] .. off[q+1]-1 (its boundary elements in order), after its -C v term.
struct StaceyRefs {
  const int* off = nullptr;
  const int* idx = nullptr;
  const double* kxd = nullptr;  // [boundary element][k][2], from k_stacey_pre
  const double* K = nullptr;  // general path: kxd holds the derivatives, still without K
};

// Stacey term of flat P-SV absorbing boundaries (BC_ABSO_apply, SRC/bc_abso.f90:321-333)
// per boundary element e and edge point k: kxd[e][k][c] = K[e][k][c] * sum_j h'_j(x_k)
// D_c(node[e][j]), D the predicted displacement d + dt v + c1 a.  The boundary nodes are
// deferred nodes, which k_deferred predicts later in the step, so the prediction is formed
// here from the state of the previous step (the same expression as in k_deferred), or is
// the d array itself (pin: the state is the predicted one).  K null: the sums without K.
template <typename R>
__global__ void k_stacey_pre(int nbe, const int* __restrict__ enode, const double* __restrict__ K,
                             const R* __restrict__ d, const R* __restrict__ v, const R* __restrict__ a, size_t GS,
                             R dt, R c1, double* __restrict__ kxd, int pin, int ng,
                             const double* __restrict__ hg) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;  // e * ng + k
  if (q >= nbe * ng) return;
  const int e = q / ng, k = q - ng * e;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    double s = 0.0;
    for (int j = 0; j < ng; ++j) {
      const size_t g = (size_t)c * GS + enode[e * ng + j];
      const R dp = pin ? d[g] : d[g] + dt * v[g] + c1 * a[g];
      s += hg[j * ng + k] * (double)dp;
    }
    kxd[(size_t)q * 2 + c] = K ? K[(size_t)q * 2 + c] * s : s;
  }
}

// Receivers at nodes, recorded where the nodes are finished.  seis[sample][ndof][nrec]; a
// sample is taken at the steps isamp, 2 isamp, ... below nsamp samples.  Receivers inside
// tiles (int_g, int_r: storage index and receiver) read the recorded field from src, which
// the tile kernel has stored; those on deferred nodes (def_q, def_r) and on fault nodes
// (flt_q: 2 * pair + side, flt_r) take it from the node's lane.  Each list is sorted.
struct RecOut {
  double* seis = nullptr;  // null: no receivers, or receivers inside elements
  int nrec = 0, isamp = 1, nsamp = 0, field = 0;
  int nint = 0, ndefr = 0, nfltr = 0;
  const int *int_g = nullptr, *int_r = nullptr, *def_q = nullptr, *def_r = nullptr;
  const int *flt_q = nullptr, *flt_r = nullptr;
  const void* src = nullptr;  // field array of the interior receivers (bulk type)
};
// the sample's rows of step it, or null
__device__ __forceinline__ double* rec_rows(const RecOut& P, int ndof, int it) {
  if (!P.seis || it % P.isamp || it / P.isamp >= P.nsamp) return nullptr;
  return P.seis + (size_t)(it / P.isamp) * ndof * P.nrec;
}
// The receivers of one node: entries at, at + 1, ... of the list with the same key.  The
// first one and the key after it are loaded ahead of the node's stores, not searched for in
// the list after them (log2(n) loads one after the other).
struct RecRef {
  int at = -1, r = 0, next = -1;
};
__device__ __forceinline__ RecRef rec_ref(const int* __restrict__ q, const int* __restrict__ r, int n, int at) {
  RecRef p;
  p.at = at;
  if (at >= 0) {
    p.r = r[at];
    p.next = q[min(at + 1, n - 1)];
  }
  return p;
}
__device__ __forceinline__ void rec_put(double* rows, const RecOut& P, const int* __restrict__ q,
                                        const int* __restrict__ r, int n, const RecRef& p, int key, int c, double x) {
  rows[(size_t)c * P.nrec + p.r] = x;
  if (p.next != key) return;
  for (int l = p.at + 1; l < n && q[l] == key; ++l) rows[(size_t)c * P.nrec + r[l]] = x;
}

// Arguments of k_deferred
template <typename R>
struct DefArgs {
  int ndef;
  DefTable defs;
  const int* part_off;
  const R* fpart;
  size_t FPS;
  const SrcEntry* src;
  const double* ampl;
  int nt, it;      // amplitude table length, step index
  const int* itp;  // step index in device memory (graph replay), or null
  const double* abso;   // [entry][NDOF]
  const double* abson;  // [entry][2] normals of entries of boundaries that are not flat
                        // (zero: flat), or null
  const R* rmdef;
  R *d, *v, *a;
  size_t GS;
  R dt, c1, c2, c3, c4;
  StepOut so;
  R* recp;  // where recorded nodes go (StepOut::rec)
  const R *din, *vin, *ain;
  StaceyRefs SR;
  RecOut rec;
  FaultDev F;
  FaultOut fo;
  const DefDev* fdef;  // [side][np]: the list entries of the pairs' nodes
};

// What a deferred node reads, loaded in one group before anything is stored: its state,
// inverse mass, up to four partial forces, its first source and absorbing entry.  The launch
// is bound by the chain list entry -> values -> stores, a round trip to memory each: with
// loads behind the first stores (which may alias them) and the partial forces one by one it
// took 7.8 us on 100 x 100 P-SV elements and 14.7 us on the 386 000 nodes of a 201 x 120
// layered mesh, now 4.0 and 11.0.
template <typename R, int NDOF>
struct DefVals {
  R d[NDOF], v[NDOF], a[NDOF], rm[NDOF], f[4][NDOF];
  double C[NDOF], am;
  SrcEntry e;
};
// places of the first four partial forces (the last one again past their number)
template <typename R>
__device__ __forceinline__ void def_offsets(const DefArgs<R>& A, const DefNode& n, int (&o)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = 0;
  if (n.pinl) {
    o[0] = n.poff[0];
    o[1] = n.poff[1] >= 0 ? n.poff[1] : o[0];
  } else if (n.pcnt > 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = A.part_off[n.pstart + min(k, n.pcnt - 1)];
  }
}
template <typename R, int NDOF, bool OOP, bool PIN>
__device__ __forceinline__ DefVals<R, NDOF> def_load(const DefArgs<R>& A, const DefNode& n, int q, int it) {
  const size_t g = n.g, GS = A.GS;
  DefVals<R, NDOF> s;
  // out of place: a null vin / ain reads v / a (their step is then in place)
  const R* dsrc = OOP ? A.din : A.d;
  const R* vsrc = OOP && A.vin ? A.vin : A.v;
  const R* asrc = OOP && A.ain ? A.ain : A.a;
  int o[4];
  def_offsets<R>(A, n, o);
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    s.d[c] = dsrc[c * GS + g];
    s.v[c] = vsrc[c * GS + g];
    if constexpr (!PIN) s.a[c] = asrc[c * GS + g];
    s.rm[c] = A.rmdef[(size_t)c * A.ndef + q];
  }
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    s.f[0][c] = A.fpart[c * A.FPS + o[0]];
    s.f[1][c] = A.fpart[c * A.FPS + o[1]];
  }
  if (!n.pinl) {
#pragma unroll
    for (int c = 0; c < NDOF; ++c) {
      s.f[2][c] = A.fpart[c * A.FPS + o[2]];
      s.f[3][c] = A.fpart[c * A.FPS + o[3]];
    }
  }
  if (n.acnt > 0) {
#pragma unroll
    for (int c = 0; c < NDOF; ++c) s.C[c] = A.abso[(size_t)n.astart * NDOF + c];
  }
  if (n.scnt > 0) {
    s.e = A.src[n.sstart];
    s.am = (it >= 1 && it <= A.nt) ? A.ampl[(size_t)s.e.src * A.nt + (it - 1)] : 0.0;
  }
  return s;
}

// Predicted state of deferred node n and its force: the partial forces of its tiles, the
// sources, the absorbing terms and the Dirichlet components
template <typename R, int NDOF, bool PIN>
__device__ __forceinline__ NodeState<R> def_state(const DefArgs<R>& A, const DefNode& n,
                                                  const DefVals<R, NDOF>& x, int it) {
  NodeState<R> s;
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    if constexpr (PIN) {
      s.d[c] = x.d[c];
      s.v[c] = x.v[c];
    } else {
      s.d[c] = x.d[c] + A.dt * x.v[c] + A.c1 * x.a[c];
      s.v[c] = x.v[c] + A.c2 * x.a[c];
    }
    R f = 0;
    if (n.pcnt > 0) f = f + x.f[0][c];
    if (n.pcnt > 1) f = f + x.f[1][c];
    if (!n.pinl) {
      if (n.pcnt > 2) f = f + x.f[2][c];
      if (n.pcnt > 3) f = f + x.f[3][c];
      for (int k = 4; k < n.pcnt; ++k) f = f + A.fpart[c * A.FPS + A.part_off[n.pstart + k]];
    }
    s.f[c] = f;
  }
  for (int k = 0; k < n.scnt; ++k) {
    const SrcEntry e = k == 0 ? x.e : A.src[n.sstart + k];
    double am = x.am;
    if (k) am = (it >= 1 && it <= A.nt) ? A.ampl[(size_t)e.src * A.nt + (it - 1)] : 0.0;
#pragma unroll
    for (int c = 0; c < NDOF; ++c)
      if (c == e.comp) s.f[c] = (R)((double)s.f[c] + e.coef * am);
  }
  for (int k = 0; k < n.acnt; ++k) {
    double C[NDOF];
#pragma unroll
    for (int c = 0; c < NDOF; ++c) C[c] = k == 0 ? x.C[c] : A.abso[(size_t)(n.astart + k) * NDOF + c];
    bool skew = false;
    if constexpr (NDOF == 2) {
      if (A.abson) {  // a boundary that is not flat (k_abso_normal)
        const double nx = A.abson[(size_t)(n.astart + k) * 2], nz = A.abson[(size_t)(n.astart + k) * 2 + 1];
        skew = nx != 0.0 || nz != 0.0;
        if (skew) {
          const double v1 = (double)s.v[0], v2 = (double)s.v[1];
          const double dot = v1 * nx + v2 * nz;
          const double vn1 = dot * nx, vn2 = dot * nz;
          s.f[0] = (R)((double)s.f[0] - C[0] * vn1 - C[1] * (v1 - vn1));
          s.f[1] = (R)((double)s.f[1] - C[0] * vn2 - C[1] * (v2 - vn2));
        }
      }
    }
    if (!skew) {
#pragma unroll
      for (int c = 0; c < NDOF; ++c) s.f[c] = (R)((double)s.f[c] - C[c] * (double)s.v[c]);
    }
    if (A.SR.off) {  // Stacey (P-SV)
      const int t0 = A.SR.off[n.astart + k], t1 = A.SR.off[n.astart + k + 1];
      if (t1 > t0) {
#pragma unroll
        for (int c = 0; c < NDOF; ++c) {
          double x = 0.0;
          for (int t = t0; t < t1; ++t) {
            const size_t i = (size_t)A.SR.idx[t] * 2 + c;
            if (A.SR.K) x += A.SR.K[i] * A.SR.kxd[i];
            else x += A.SR.kxd[i];
          }
          s.f[c] = (R)((double)s.f[c] - x);
        }
      }
    }
  }
  // Dirichlet components (BC_DIRNEU_apply, SRC/bc_dirneu.f90:148-169): absorbing
  // boundaries act first, then the others in their order
#pragma unroll
  for (int c = 0; c < NDOF; ++c)
    if (n.dmask >> c & 1) s.f[c] = 0;
  return s;
}

// Corrector of component c of a deferred node from its predicted state and its new
// acceleration ak, and the stores, as in the tile kernel (StepOut); the displacement and
// velocity after the step are left in s.  rec: a recorded node
template <typename R>
__device__ __forceinline__ void def_store(const DefArgs<R>& A, NodeState<R>& s, int c, size_t i, R ak, bool rec) {
  const R vn = s.v[c] + A.c3 * ak;
  const R dn = s.d[c] + A.c4 * ak;
  s.v[c] = vn;
  s.d[c] = dn;
  if (A.so.final) {
    A.a[i] = ak;
    A.v[i] = vn;
    A.d[i] = dn;
  } else {
    A.v[i] = vn + A.c2 * ak;
    A.d[i] = dn + A.dt * vn + A.c1 * ak;
    if (A.so.accel) A.a[i] = ak;
    if (rec && A.so.rec >= 0) A.recp[i] = A.so.rec == 0 ? dn : (A.so.rec == 1 ? vn : ak);
  }
}
template <typename R>
__device__ __forceinline__ double rec_value(const RecOut& P, const NodeState<R>& s, int c, R ak) {
  const R dn = s.d[c], vn = s.v[c];
  return (double)(P.field == 0 ? dn : (P.field == 1 ? vn : ak));
}

// Everything a step does after the tile kernel, in one launch: the deferred nodes (those
// of the tile perimeters and the sources), the receivers, and, FLT, the fault: the first
// fo.nwave wavefronts take the fault pairs, each lane both nodes of a pair
// from their partial forces to their stores, with the pair's traction solve, its record
// and the step's potency row; the nodes' other lanes skip them.
// PIN: the state read is the predicted one.
template <typename R, int NDOF, bool OOP = false, bool PIN = false, bool FLT = false>
__global__ __launch_bounds__(256) void k_deferred(DefArgs<R> A) {
  const int it = A.itp ? *A.itp : A.it;
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  double* const rows = rec_rows(A.rec, NDOF, it);
  if constexpr (FLT) {
    const int w = q >> 6;  // uniform in a wavefront
    if (w < A.fo.nwave) {
      const FaultDev& F = A.F;
      const FaultOut& O = A.fo;
      const int4 wv = O.wave[w];
      const int2 mw = O.member[wv.z];
      const int lane = q & 63, k = wv.x + lane;
      const bool on = lane < wv.y;
      PairData P;
      double dj[2] = {0, 0}, vj[2] = {0, 0};
      if (on) {
        const int np = F.np;
        const int q1 = F.def1[k], q2 = F.def2[k];
        const DefDev e1 = A.fdef[k], e2 = A.fdef[np + k];
        const bool two = q2 >= 0;
        int rs = O.rec_slot;
        if (A.itp) rs = it >= O.oit0 && (it - O.oit0) % O.oitd == 0 ? (it - O.oit0) / O.oitd : -1;
        const int slot = rs >= 0 && rs < O.nsamp ? O.slot[k] : -1;
        const int dm = F.dmask ? F.dmask[k] : 0;
        P = pair_load<NDOF>(F, k, two);
        const DefNode m1 = def_unpack(A.defs, e1), m2 = def_unpack(A.defs, e2);
        const DefVals<R, NDOF> x1 = def_load<R, NDOF, OOP, PIN>(A, m1, q1, it);
        DefVals<R, NDOF> x2;
        if (two) x2 = def_load<R, NDOF, OOP, PIN>(A, m2, q2, it);
        RecRef r1, r2;
        if (rows) {
          r1 = rec_ref(A.rec.flt_q, A.rec.flt_r, A.rec.nfltr, m1.rec_at);
          if (two) r2 = rec_ref(A.rec.flt_q, A.rec.flt_r, A.rec.nfltr, m2.rec_at);
        }
        NodeState<R> n1 = def_state<R, NDOF, PIN>(A, m1, x1, it), n2;
        if (two) n2 = def_state<R, NDOF, PIN>(A, m2, x2, it);
        const PairOut po = fault_solve<R, NDOF>(F, P, k, (double)it * F.dt, two, n1, n2);
        R* side = (R*)F.side + k;  // [d, v][node][ndof][np]
#pragma unroll
        for (int c = 0; c < NDOF; ++c) {
          if (dm >> c & 1) n1.f[c] = 0;
          const R a1 = n1.f[c] * x1.rm[c];
          def_store<R>(A, n1, c, (size_t)c * A.GS + m1.g, a1, m1.rec);
          side[(size_t)c * np] = n1.d[c];
          side[(size_t)(2 * NDOF + c) * np] = n1.v[c];
          if (r1.at >= 0)
            rec_put(rows, A.rec, A.rec.flt_q, A.rec.flt_r, A.rec.nfltr, r1, 2 * k, c,
                    rec_value<R>(A.rec, n1, c, a1));
          if (two) {
            if (dm >> (2 + c) & 1) n2.f[c] = 0;
            const R a2 = n2.f[c] * x2.rm[c];
            def_store<R>(A, n2, c, (size_t)c * A.GS + m2.g, a2, m2.rec);
            side[(size_t)(NDOF + c) * np] = n2.d[c];
            side[(size_t)(3 * NDOF + c) * np] = n2.v[c];
            if (r2.at >= 0)
              rec_put(rows, A.rec, A.rec.flt_q, A.rec.flt_r, A.rec.nfltr, r2, 2 * k + 1, c,
                      rec_value<R>(A.rec, n2, c, a2));
          }
          // get_jump (SRC/bc_dynflt.f90:692-704): x2 - x1, or -2 x1 on a one-sided fault
          dj[c] = two ? (double)n2.d[c] - (double)n1.d[c] : -2.0 * (double)n1.d[c];
          vj[c] = two ? (double)n2.v[c] - (double)n1.v[c] : -2.0 * (double)n1.v[c];
        }
        if (slot >= 0) {
          double* out = O.rec + (size_t)rs * 6 * O.nout + slot;
          out[0] = po.D0;
          out[(size_t)1 * O.nout] = po.V0;
          out[(size_t)2 * O.nout] = po.T[0];
          out[(size_t)3 * O.nout] = po.T[1];
          out[(size_t)4 * O.nout] = po.mu;
          out[(size_t)5 * O.nout] = po.Ts0;
        }
      }
      potency_wave<NDOF>(P, O, w, wv.z, mw, on, dj, vj, O.pot_row + (A.itp ? it : 0));
      return;
    }
    q -= A.fo.nwave * 64;
  }
  if (q >= A.ndef) {  // receivers inside tiles
    const int r = q - A.ndef;
    if (rows && r < A.rec.nint)
      for (int c = 0; c < NDOF; ++c)
        rows[(size_t)c * A.rec.nrec + A.rec.int_r[r]] =
            (double)((const R*)A.rec.src)[(size_t)c * A.GS + A.rec.int_g[r]];
    return;
  }
  const DefNode n = def_unpack(A.defs, q);
  if (FLT && n.fault) return;
  const DefVals<R, NDOF> x = def_load<R, NDOF, OOP, PIN>(A, n, q, it);
  RecRef rr;
  if (rows) rr = rec_ref(A.rec.def_q, A.rec.def_r, A.rec.ndefr, n.rec_at);
  NodeState<R> s = def_state<R, NDOF, PIN>(A, n, x, it);
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    const R ak = s.f[c] * x.rm[c];
    def_store<R>(A, s, c, (size_t)c * A.GS + n.g, ak, n.rec);
    if (rr.at >= 0)
      rec_put(rows, A.rec, A.rec.def_q, A.rec.def_r, A.rec.ndefr, rr, q, c, rec_value<R>(A.rec, s, c, ak));
  }
}

// Arguments of k_run_steps
template <typename R>
struct RunArgs {
  TileArgs<R> T;
  DefArgs<R> D;         // D.it: the first step
  R* fpart2;            // partial forces of every second step
  const int* nbr;       // [ntiles][8] tiles that share a node with a tile, or -1
  const int* slot_def;  // [ntiles][SLOTS] deferred node of a partial force, or -1
  unsigned* flag;       // [ntiles][FLAG_STRIDE] epoch + the steps whose partial forces a tile has stored
  unsigned* arrived;    // the word of run_commit
  unsigned epoch;
  int nsteps, spins;
  int* fail;
};
constexpr int FLAG_STRIDE = 16;
// run_commit's word, accessed past the L2 caches
struct RunWord {
  unsigned* p;
  __device__ unsigned add(unsigned x) {
    return __hip_atomic_fetch_add(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ unsigned load() { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  __device__ bool cas(unsigned& e, unsigned d) {
    return __hip_atomic_compare_exchange_strong(p, &e, d, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
  }
};

// nsteps steps of a small grid in one launch, a workgroup per tile, all of them resident
// together (cooperative launch): a step by its two launches is bound by their start and by
// the reads and stores of a state that fits in the compute units (100 x 100 P-SV elements,
// FP64: 14.2 us a step of two launches, 6.0 here).  The state is the predicted one, the
// displacement in LDS, velocity and inverse mass in the registers of the node's lane.  After
// the element phase a tile stores the partial forces of its perimeter and special nodes,
// raises its flag, waits for the flags of the up to eight tiles that share nodes with it and
// finishes those nodes itself, as k_deferred does; a node that several tiles share is
// computed by each of them from the same values in the same order.  Partial forces alternate
// between two arrays: a tile stores those of step s + 2 when its neighbours have raised their
// flags for step s + 1, that is, have read those of step s.
//
// Partial forces, flags and the count go past the L2 caches of the XCDs (atomic accesses at
// agent scope); a tile's stores are waited for before its flag is raised, so no cache is
// written back or invalidated.
//
// A wait ends after `spins` polls.  Nothing of the state is stored before the tiles have
// agreed that every one is through (run_commit), so that a launch that has given up leaves
// the state it started from, and the steps are then taken by the other kernels.
template <typename R, int NDOF, int NELAST, int MODE>
__global__ __launch_bounds__(TS_NT) __attribute__((amdgpu_waves_per_eu(2))) void k_run_steps(RunArgs<R> A) {
  constexpr int PS = PXM, NEL = TX * TZ;
  constexpr bool NODEM = MODE == COEF_NODE, COMP = MODE == COEF_COMPACT || MODE == COEF_ELEM;
  constexpr int NM = MODE == COEF_COMPACT ? NG : 1;
  using LV = typename LVec<R, NDOF>::T;
  __shared__ LV Ud[PMAX];
  __shared__ LV Ex[NEL * NP + 1];
  __shared__ LV Mn[NODEM ? PMAX : 1];
  __shared__ R Sa[MODE == COEF_SHARED ? NELAST * NP : 1];
  __shared__ R Gm[NEL][3];
  __shared__ R sW2[NP];
  __shared__ int stop;
  const TileArgs<R>& T = A.T;
  const DefArgs<R>& D = A.D;
  const int t = blockIdx.x, tid = threadIdx.x;
  const int4 tg = T.tiles[t], gr = T.grids[t];
  const int nxe = tg.z & 0xff, nze = (tg.z >> 8) & 0xff, nx = tg.z >> 16;
  const int PX = 4 * nxe + 1, PZ = 4 * nze + 1, X0 = 4 * tg.x, Z0 = tg.w;
  const int kL = tg.x / TX, kR = (tg.x + nxe + TX - 1) / TX;
  const int ns = T.spec_cnt[t];
  if (tid < NP) sW2[tid] = (R)c_W2[tid];
  if (tid == 0) Ex[NEL * NP] = LV{}, stop = 0;

  // this lane's patch nodes: storage index, slot of the partial force (-1: the node is
  // finished here), velocity, inverse mass, first receiver
  size_t g[TS_ITER];
  int slot[TS_ITER], ir[TS_ITER];
  bool in[TS_ITER];
  NodeSlots sl[TS_ITER];
  R vr[TS_ITER][NDOF], rm[TS_ITER];
#pragma unroll
  for (int r = 0; r < TS_ITER; ++r) {
    const int p = tid + TS_NT * r, Z = p / PS, X = p - Z * PS;
    in[r] = X < PX && Z < PZ;
    g[r] = node_index(gr, min(X, PX - 1), min(Z, PZ - 1), PX, X0, Z0, kL, kR);
    slot[r] = in[r] ? perim_slot(X, Z, PX, PZ) : -1;
    for (int k = 0; k < ns; ++k)
      if (T.spec_idx[t * MAXSPECIAL + k] == p) slot[r] = PERIM_MAX + k;
    sl[r] = c_slots.node[min(p, PMAX - 1)];
    rm[r] = T.rmass0[g[r]];
    R u[NDOF], m[NDOF];
#pragma unroll
    for (int c = 0; c < NDOF; ++c) {
      u[c] = T.d[c * T.S + g[r]];
      vr[r][c] = T.v[c * T.S + g[r]];
      if constexpr (NODEM) m[c] = T.coefs[c * T.S + g[r]];
    }
    if (p < PMAX) {
      Ud[p] = lv_make<R, NDOF>(u);
      if constexpr (NODEM) Mn[p] = lv_make<R, NDOF>(m);
    }
    ir[r] = -1;
    if (D.rec.seis && in[r] && slot[r] < 0) {
      int lo = 0, hi = D.rec.nint;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((size_t)D.rec.int_g[mid] < g[r]) lo = mid + 1;
        else hi = mid;
      }
      if (lo < D.rec.nint && (size_t)D.rec.int_g[lo] == g[r]) ir[r] = lo;
    }
  }
  if constexpr (MODE == COEF_SHARED) {
    for (int k = tid; k < NELAST * NP; k += TS_NT) Sa[k] = T.coefs[gr.w + k];
  } else {
    if (tid < NEL * 3) {
      const int e = tid / 3, k = tid - 3 * (tid / 3);
      Gm[e][k] = T.geom[cell_index(gr, nx, tg.x, tg.y, min(e % TX, nxe - 1), min(e / TX, nze - 1)) * 3 + k];
    }
  }
  const int lane = tid & 63;
  const int e = (tid >> 6) * TS_EPW + lane / NG, s = lane % NG;
  const int lx = e % TX, lz = e / TX;
  const bool eslot = lane < TS_EPW * NG && e < NEL, on = eslot && lx < nxe && lz < nze;
  const int base = 4 * lz * PS + 4 * lx;
  LV* ex = Ex + min(e, NEL - 1) * NP;
  R m[NM][NDOF];
  if constexpr (COMP) {
    const size_t cell = cell_index(gr, nx, tg.x, tg.y, min(lx, nxe - 1), min(lz, nze - 1));
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
      for (int c = 0; c < NDOF; ++c)
        m[i][c] = T.coefs[NM == 1 ? cell * NDOF + c : (cell * NDOF + c) * NP + s * NG + i];
  }

  // the deferred node of this lane (one lane per slot), its values and its patch node
  const int nper = 2 * PX + 2 * (PZ - 2);
  const bool dl = tid < nper || (tid >= PERIM_MAX && tid < PERIM_MAX + ns);
  int pp = 0, dq = 0, o[4] = {0, 0, 0, 0};
  DefNode n{};
  DefVals<R, NDOF> x{};
  RecRef rr;
  if (dl) {
    if (tid < nper) {
      const int w = tid - 2 * PX;
      const int X = tid < 2 * PX ? tid % PX : (w < PZ - 2 ? 0 : PX - 1);
      const int Z = tid < PX ? 0 : (tid < 2 * PX ? PZ - 1 : w % (PZ - 2) + 1);
      pp = Z * PS + X;
    } else {
      pp = T.spec_idx[t * MAXSPECIAL + tid - PERIM_MAX];
    }
    dq = A.slot_def[t * SLOTS + tid];
    n = def_unpack(D.defs, dq);
    def_offsets<R>(D, n, o);
    x = def_load<R, NDOF, false, true>(D, n, dq, D.it);
    if (D.rec.seis) rr = rec_ref(D.rec.def_q, D.rec.def_r, D.rec.ndefr, n.rec_at);
  }
  const bool own = dl && o[0] / SLOTS == t;  // stores and records the node
  const int nb = tid < 8 ? A.nbr[t * 8 + tid] : -1;
  const R dt = T.dt, c1 = T.c1, c2 = T.c2, c3 = T.c3, c4 = T.c4;
  const int field = D.rec.field;
  R fa[TS_ITER][NDOF], fd[NDOF] = {};  // last step: the accelerations, for the stores
#pragma unroll
  for (int r = 0; r < TS_ITER; ++r)
#pragma unroll
    for (int c = 0; c < NDOF; ++c) fa[r][c] = 0;
  __syncthreads();

#pragma unroll 1
  for (int k = 0; k < A.nsteps; ++k) {
    const int it = D.it + k;
    const bool last = k == A.nsteps - 1;
    double* const rows = rec_rows(D.rec, NDOF, it);
    if (dl && n.scnt > 0) x.am = it >= 1 && it <= D.nt ? D.ampl[(size_t)x.e.src * D.nt + (it - 1)] : 0.0;
    {
      const auto* hp = hconst<R>();
      R H[NG][NG];
#pragma unroll
      for (int a = 0; a < NG; ++a)
#pragma unroll
        for (int b = 0; b < NG; ++b) H[a][b] = hp[a * NG + b];
      el_gradient<R, NDOF, false>(on, base, s, e, ex, Ud, Ud, (const R*)nullptr, H);
      wave_order();
      R s1r[NG][NDOF];
      el_flux<R, NDOF, NELAST, MODE, false>(on, base, s, e, ex, Ud, Ud, (const R*)nullptr, H, Gm, sW2, Sa, Mn, m,
                                            [](int, int) { return R(0); }, s1r);
      wave_order();
      el_divergence<R, NDOF>(on, s, ex, H);
      wave_order();
      el_force<R, NDOF, false>(on, eslot, false, base, s, e, ex, Ud, Ud, (const R*)nullptr, (const R*)nullptr, s1r);
    }
    __syncthreads();
    R* const fp = k & 1 ? A.fpart2 : T.fpart;
    R F[TS_ITER][NDOF];
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const LV f0 = Ex[sl[r].q[0]], f1 = Ex[sl[r].q[1]], f2 = Ex[sl[r].q[2]], f3 = Ex[sl[r].q[3]];
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        F[r][c] = ((lv_get<R, NDOF>(f0, c) + lv_get<R, NDOF>(f1, c)) + lv_get<R, NDOF>(f2, c)) + lv_get<R, NDOF>(f3, c);
        if (slot[r] >= 0)
          __hip_atomic_store(&fp[c * T.FPS + (size_t)t * SLOTS + slot[r]], F[r][c], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    // nodes that are finished here
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r)
      if (in[r] && slot[r] < 0) {
        const int p = tid + TS_NT * r;
        const LV u = Ud[p];
        R nu[NDOF];
#pragma unroll
        for (int c = 0; c < NDOF; ++c) {
          const R ak = F[r][c] * rm[r];
          const R vn = vr[r][c] + c3 * ak;
          const R dn = lv_get<R, NDOF>(u, c) + c4 * ak;
          vr[r][c] = last ? vn : vn + c2 * ak;
          nu[c] = last ? dn : dn + dt * vn + c1 * ak;
          if (last) fa[r][c] = ak;
          if (rows && ir[r] >= 0)
            for (int q = ir[r]; q < D.rec.nint && (size_t)D.rec.int_g[q] == g[r]; ++q)
              rows[(size_t)c * D.rec.nrec + D.rec.int_r[q]] = (double)(field == 0 ? dn : (field == 1 ? vn : ak));
        }
        Ud[p] = lv_make<R, NDOF>(nu);
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the partial forces are past the L2
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(&A.flag[(size_t)t * FLAG_STRIDE], A.epoch + k + 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    if (nb >= 0) {
      int left = A.spins;
      while ((int)(__hip_atomic_load(&A.flag[(size_t)nb * FLAG_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) -
                   (A.epoch + k + 1)) < 0) {
        if (--left < 0) {
          stop = 1;
          break;
        }
      }
    }
    __syncthreads();
    if (stop) break;
    if (dl) {
#pragma unroll
      for (int c = 0; c < NDOF; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < 2 || !n.pinl)
            x.f[q][c] = __hip_atomic_load(&fp[c * T.FPS + o[q]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      NodeState<R> st = def_state<R, NDOF, true>(D, n, x, it);
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        const R ak = st.f[c] * x.rm[c];
        const R vn = st.v[c] + c3 * ak;
        const R dn = st.d[c] + c4 * ak;
        x.v[c] = last ? vn : vn + c2 * ak;
        x.d[c] = last ? dn : dn + dt * vn + c1 * ak;
        if (last) fd[c] = ak;
        if (rows && own && rr.at >= 0)
          rec_put(rows, D.rec, D.rec.def_q, D.rec.def_r, D.rec.ndefr, rr, dq, c,
                  (double)(field == 0 ? dn : (field == 1 ? vn : ak)));
      }
      Ud[pp] = lv_make<R, NDOF>(x.d);
    }
    __syncthreads();
  }

  // the state is stored when every tile is through
  if (tid == 0) {
    RunWord word{A.arrived};
    const bool ok = run_commit(word, !stop, gridDim.x, A.spins);
    if (!ok) *A.fail = 1;
    stop = !ok;
  }
  __syncthreads();
  if (stop) return;
#pragma unroll
  for (int r = 0; r < TS_ITER; ++r)
    if (in[r] && slot[r] < 0) {
      const LV u = Ud[tid + TS_NT * r];
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        T.a[c * T.S + g[r]] = fa[r][c];
        T.v[c * T.S + g[r]] = vr[r][c];
        T.d[c * T.S + g[r]] = lv_get<R, NDOF>(u, c);
      }
    }
  if (own) {
#pragma unroll
    for (int c = 0; c < NDOF; ++c) {
      T.a[c * T.S + n.g] = fd[c];
      T.v[c * T.S + n.g] = x.v[c];
      T.d[c * T.S + n.g] = x.d[c];
    }
  }
}

// ===========================================================================
// Adjoint (reverse-mode) step on structured grids, P-SV with compact coefficients.
//
// Forward step n (SRC/solver.f90:42-84 with beta = 0):
//   dp = d + dt v + c1 a,  vp = v + c2 a,  a' = (-K dp - C vp + s) / Mt,
//   v' = vp + c3 a',  d' = dp,                       Mt = M + c3 C (ABC-modified mass)
// Its transpose, from the adjoint (ad, av, aa) of step n to that of step n-1:
//   fb = (aa + c3 av) / Mt
//   ad <- ad - K^T fb,  vbp = av - C fb,  av <- vbp + dt ad,  aa <- c2 vbp + c1 ad
// and the sensitivities of J to the step's parameters:
//   dJ/dMt = -fb * a_n,  dJ/dC = -fb * vp_n,
//   dJ/dA_k = (B fb)^T dPhi/dA_k (B d_n)   per GLL point, A_k the KD2 coefficients
// with Phi the point flux matrix of ELAST_KD2_PSV (SRC/mat_elastic.f90:589-641):
//   flux(xi,x) = A0 gxx + A1 gez,  flux(eta,x) = A3 (gex + gxz),
//   flux(xi,z) = A4 gex + A5 gxz,  flux(eta,z) = A1 gxx + A2 gez,
// (g.. the xi/eta derivatives of the x/z components).  -K^T uses Phi^T:
//   flux(eta,x) = A3 gex + A4 gxz,  flux(xi,z) = A3 gex + A5 gxz  (others unchanged).
// A = W2 * modulus * geometric factor (A0 = W2 (l+2m) g0, A1 = W2 l g2, A2 = W2 (l+2m) g1,
// A3 = W2 m g1, A4 = W2 m g2, A5 = W2 m g0), so per point
//   dJ/dl = W2 [g0 pxx gxx + g2 (pxx gez + pez gxx) + g1 pez gez]
//   dJ/dm = W2 [2 g0 pxx gxx + 2 g1 pez gez + g1 pex (gex + gxz) + g2 pxz gex + g0 pxz gxz]
// (p.. the derivatives of fb, g.. those of d_n), summed over the element's points.
// One workgroup per tile; interior nodes finish here, perimeter nodes in k_adj_deferred.
// ===========================================================================
// Forward acceleration a_n from a history of displacements: the second difference
// (d_{n+1} - 2 d_n + d_{n-1}) / dt^2, which equals a_n for the explicit Newmark scheme
// (beta = 0, gamma = 1/2): d_{n+1} - d_n = dt v_n + dt^2/2 a_n and v_n - v_{n-1} =
// dt/2 (a_{n-1} + a_n).
__device__ __forceinline__ double fwd_accel(double dprev, double dcur, double dnext, double idt2) {
  return ((dnext - dcur) - (dcur - dprev)) * idt2;
}

// Injection of dJ/d(recorded field): the sample of step n is added to the adjoint state
// that step n starts from, at the injection nodes unode[0 .. nu) (ascending storage
// indices), node u with the contributions (receiver rec[k], weight w[k], k in [off[u],
// off[u+1])) in receiver order.
struct InjectPlan {
  int nu = 0, nrec = 0, field = 1;
  const int *unode = nullptr, *off = nullptr, *rec = nullptr;
  const double* w = nullptr;
  const double* g = nullptr;  // the sample, [ndof][nrec]; null: no injection
  const int* udef = nullptr;  // injection node of deferred node q, or -1
  const unsigned char* tile = nullptr;  // tiles with an injection node in their patch
};
template <typename R>
__device__ __forceinline__ R inject_at(const InjectPlan& P, int u, int c, R x) {
  for (int k = P.off[u]; k < P.off[u + 1]; ++k) x = (R)((double)x + P.w[k] * P.g[(size_t)c * P.nrec + P.rec[k]]);
  return x;
}
__device__ __forceinline__ int inject_find(const InjectPlan& P, int node) {
  int lo = 0, hi = P.nu;
  while (lo < hi) {
    const int m = (lo + hi) >> 1;
    if (P.unode[m] < node) lo = m + 1;
    else hi = m;
  }
  return lo < P.nu && P.unode[lo] == node ? lo : -1;
}

// The adjoint state is kept as the pair (ad, w) that the last update formed it from,
// av = w + dt ad and aa = c2 w + c1 ad; the injected values come on top where the state is
// read.  (Two field arrays each way instead of three.)
template <typename R>
struct AdjNode {
  R d, v, a;
};
template <typename R>
__device__ __forceinline__ AdjNode<R> adj_node(R dn, R w, R dt, R c1, R c2) {
  return {dn, w + dt * dn, c2 * w + c1 * dn};
}

template <typename R>
struct AdjArgs {
  R *ad, *w;
  const R *rmass, *dfw, *x1, *x2;  // x1, x2: forward acceleration and null, or d_{n-1} and d_{n+1}
  const R *coefs, *geom;
  R* fpart;
  double *glam, *gmu, *mbar;
  size_t S, FPS;
  const int4 *tiles, *grids;
  const int *spec_cnt, *spec_idx;
  int ntiles;
  R dt, c1, c2, c3;
  double idt2;
  InjectPlan inj;
};

// Adjoint tile step, one tile per workgroup, with the element phase of k_tile_step (a lane
// per element row or column, exchanges inside a wavefront): the gradient of the forward
// displacement first, kept for the row's five points in registers, then that of fb, the
// transposed fluxes and the sensitivities, whose sums over an element are the rows' sums
// added in row order.  HIST: the forward acceleration is the second difference of the
// displacement history (fwd_accel).  The adjoint state of the interior nodes is read again
// for the stores (a register each through the element phase would halve the wavefronts).
// ELEM: moduli per element (COEF_ELEM).  Bound by memory where the tiles fill the chip, by
// the chain of a tile's phases where they do not: 400 x 400 elements, FP64, 113.6 us for 390
// MB; 150 x 101 16.1 us.  (A lane per element point, with a workgroup barrier per colour and
// three state arrays, in two launches: 162 and 18.8 + 16.9 us.)
template <typename R, bool HIST, bool ELEM, bool W32>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_adj_step(AdjArgs<R> args) {
  constexpr int NDOF = 2, PS = PXM, NEL = TX * TZ;
  using LV = typename LVec<R, NDOF>::T;
  __shared__ LV Uf[PMAX];  // fb
  __shared__ LV Ud[PMAX];  // forward d_n
  __shared__ LV Ex[NEL * NP + 1];
  __shared__ NodeSlots Eg[PMAX];
  __shared__ R Gm[NEL][3];
  __shared__ R sW2[NP];
  // each XCD (bid & 7) takes a contiguous eighth of the tiles
  const int per = (args.ntiles + 7) >> 3, bid = blockIdx.x;
  const int t = (bid & 7) * per + (bid >> 3);
  if ((bid >> 3) >= per || t >= args.ntiles) return;
  const int tid = threadIdx.x;
  const auto* P = kernel_args<AdjArgs<R>>();
  const int4 tg = sload(P->tiles, t), gr = sload(P->grids, t);
  const int nxe = tg.z & 0xff, nze = (tg.z >> 8) & 0xff, nx = tg.z >> 16;
  const int PX = 4 * nxe + 1, PZ = 4 * nze + 1, X0 = 4 * tg.x, Z0 = tg.w;
  const int kL = tg.x / TX, kR = (tg.x + nxe + TX - 1) / TX;
  using I = std::conditional_t<W32, uint32_t, size_t>;
  auto nidx = [&](int X, int Z) {
    const I row = (I)gr.x + (I)Z0 * (I)gr.y + (I)(X0 - 1);
    const I edge = (I)gr.x + (I)gr.y * (I)gr.z + (I)Z0;
    const I eL = edge + (I)kL * (I)gr.z, eR = edge + (I)kR * (I)gr.z;
    const I in = row + (I)((uint32_t)Z * (uint32_t)gr.y + (uint32_t)X);
    return X == 0 || X == PX - 1 ? (X == 0 ? eL : eR) + (I)Z : in;
  };
  auto cidx = [&](int lx, int lz) { return (I)gr.w + (I)(tg.y + lz) * (I)nx + (I)(tg.x + lx); };
  auto ub = [&](auto* p) {
    if constexpr (W32) return sgpr_base(p);
    else return p;
  };
  auto at = [&](auto* base, auto g) -> auto& {
    if constexpr (W32) return at32(base, (uint32_t)g);
    else return base[g];
  };
  const size_t S = P->S;
  // lane index the compiler cannot look through (as in k_tile_step)
  auto lane_id = [&]() {
    int q = tid;
    asm volatile("" : "+v"(q));
    __builtin_assume(q >= 0 && q < TS_NT);
    return q;
  };
  const int ns = sload(P->spec_cnt, t);
  auto special = [&](int p) {
    int k = -1;
    for (int q = 0; q < ns; ++q)
      if (sload(P->spec_idx, t * MAXSPECIAL + q) == p) k = q;
    return k;
  };
  const bool inj = P->inj.g && P->inj.tile[t];
  const int field = P->inj.field;
  const R dt = P->dt, c1 = P->c1, c2 = P->c2, c3 = P->c3;
  // adds the injected values of node g to the arrays f of its components
  auto inject = [&](I g, auto&&... f) {
    const InjectPlan J = args.inj;
    const int u = inject_find(J, (int)g);
    if (u >= 0) {
      int c = 0;
      ((f = inject_at<R>(J, u, c++, f)), ...);
    }
  };
  {
    const int tl = lane_id();
    I g[TS_ITER];
    R u[TS_ITER][NDOF], v[TS_ITER][NDOF], a[TS_ITER][NDOF], rm[TS_ITER][NDOF];
    R x1[TS_ITER][NDOF], x2[TS_ITER][NDOF];
    double mb[TS_ITER];
    double* const bmb = ub(P->mbar);
    // all loads first
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const int p = tl + TS_NT * r, Z = p / PS, X = p - Z * PS;
      g[r] = nidx(min(X, PX - 1), min(Z, PZ - 1));
    }
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        v[r][c] = at(ub(P->w + c * S), g[r]);
        a[r][c] = at(ub(P->ad + c * S), g[r]);
        rm[r][c] = at(ub(P->rmass + c * S), g[r]);
        u[r][c] = at(ub(P->dfw + c * S), g[r]);
        x1[r][c] = at(ub(P->x1 + c * S), g[r]);
        if constexpr (HIST) x2[r][c] = at(ub(P->x2 + c * S), g[r]);
      }
      mb[r] = at(bmb, g[r]);
    }
    // behind these loads, as in k_tile_step
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r)
      if (const int p = tl + TS_NT * r; p < PMAX) Eg[p] = c_slots.node[p];
    if (tl < NP) sW2[tl] = (R)c_W2[tl];
    if (tl == 0) Ex[NEL * NP] = LV{};
    if (tl < NEL * 3) {
      const int e = tl / 3, k = tl - 3 * (tl / 3);
      Gm[e][k] = at(ub(P->geom), cidx(min(e % TX, nxe - 1), min(e / TX, nze - 1)) * 3 + k);
    }
    warm_h<R>();
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r)
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        const AdjNode<R> s = adj_node<R>(a[r][c], v[r][c], dt, c1, c2);
        v[r][c] = s.v;
        a[r][c] = s.a;
      }
    if (inj && field) {
#pragma unroll
      for (int r = 0; r < TS_ITER; ++r) {
        if (field == 1) inject(g[r], v[r][0], v[r][1]);
        else inject(g[r], a[r][0], a[r][1]);
      }
    }
    const double idt2 = P->idt2;
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      R f[NDOF];
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        f[c] = (a[r][c] + c3 * v[r][c]) * rm[r][c];
        double acc = (double)x1[r][c];
        if constexpr (HIST) acc = fwd_accel((double)x1[r][c], (double)u[r][c], (double)x2[r][c], idt2);
        mb[r] -= (double)f[c] * acc;
      }
      const int p = tl + TS_NT * r, Z = p / PS, X = p - Z * PS;
      if (p < PMAX) {
        Uf[p] = lv_make<R, NDOF>(f);
        Ud[p] = lv_make<R, NDOF>(u[r]);
      }
      // the mass sensitivity of interior nodes (perimeter and special nodes: k_adj_deferred)
      if (X < PX && Z < PZ && perim_slot(X, Z, PX, PZ) < 0 && special(p) < 0) at(bmb, g[r]) = mb[r];
    }
  }
  __syncthreads();

  const int ts = lane_id();
  R ad[TS_ITER][NDOF], av[TS_ITER][NDOF];  // the adjoint state again, for the stores
  {
    const int te = lane_id(), lane = te & 63;
    const int e = (te >> 6) * TS_EPW + lane / NG, s = lane % NG;
    const int lx = e % TX, lz = e / TX;
    const bool on = lane < TS_EPW * NG && e < NEL && lx < nxe && lz < nze;
    const int base = 4 * lz * PS + 4 * lx;
    const I cell = cidx(min(lx, nxe - 1), min(lz, nze - 1));
    LV* ex = Ex + min(e, NEL - 1) * NP;
    const auto* hp = hconst<R>();
    R H[NG][NG];
#pragma unroll
    for (int k = 0; k < NG; ++k)
#pragma unroll
      for (int i = 0; i < NG; ++i) H[k][i] = hp[k * NG + i];
    // column derivatives of a patch array into the exchange array
    auto column = [&](const LV* U) {
      el_gradient<R, NDOF, false>(on, base, s, e, ex, U, U, (const R*)nullptr, H);
      wave_order();
    };
    column(Ud);
    R gxi[NG][NDOF], get[NG][NDOF];  // gradient of d_n at the row's points
    {
      R x[NG][NDOF];
#pragma unroll
      for (int k = 0; k < NG; ++k) {
        const LV xv = Ud[min(base + s * PS + k, PMAX - 1)];
#pragma unroll
        for (int c = 0; c < NDOF; ++c) x[k][c] = lv_get<R, NDOF>(xv, c);
      }
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const LV gv = ex[s * NG + i];
#pragma unroll
        for (int c = 0; c < NDOF; ++c) {
          R sum = 0;
#pragma unroll
          for (int k = 0; k < NG; ++k) sum += H[k][i] * x[k][c];
          gxi[i][c] = sum;
          get[i][c] = lv_get<R, NDOF>(gv, c);
        }
      }
    }
    wave_order();
    // moduli of the row's points, the element's running sensitivities
    constexpr int NM = ELEM ? 1 : NG;
    R m[NM][NDOF];
    {
      const R* bco = ub(P->coefs);
#pragma unroll
      for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int c = 0; c < NDOF; ++c)
          m[i][c] = at(bco, ELEM ? cell * NDOF + c : (cell * NDOF + c) * NP + s * NG + i);
    }
    column(Uf);
    // the sensitivities first, then the fluxes: the gradient of d_n and the transposed
    // sums are not in registers together (FP64: 128 of them, without spills)
    R x[NG][NDOF];
    double rl = 0, rmu = 0;
    const int em = min(e, NEL - 1);
    const R g0 = Gm[em][0], g1 = Gm[em][1], g2 = Gm[em][2];
    auto pgrad = [&](int i, R (&pxi)[NDOF]) {
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        R sum = 0;
#pragma unroll
        for (int k = 0; k < NG; ++k) sum += H[k][i] * x[k][c];
        pxi[c] = sum;
      }
    };
    if (on) {
#pragma unroll
      for (int k = 0; k < NG; ++k) {
        const LV xv = Uf[base + s * PS + k];
#pragma unroll
        for (int c = 0; c < NDOF; ++c) x[k][c] = lv_get<R, NDOF>(xv, c);
      }
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        R pxi[NDOF];
        pgrad(i, pxi);
        const LV pv = ex[s * NG + i];
        const double wd = (double)(R)sW2[s * NG + i];
        const R pxx = pxi[0], pxz = pxi[1], pex = lv_get<R, NDOF>(pv, 0), pez = lv_get<R, NDOF>(pv, 1);
        const R gxx = gxi[i][0], gxz = gxi[i][1], gex = get[i][0], gez = get[i][1];
        rl += wd * ((double)g0 * pxx * gxx + (double)g2 * (pxx * gez + pez * gxx) + (double)g1 * pez * gez);
        rmu += wd * (2.0 * g0 * pxx * gxx + 2.0 * g1 * pez * gez + (double)g1 * pex * (gex + gxz) +
                     (double)g2 * pxz * gex + (double)g0 * pxz * gxz);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the element's running sensitivities, for the sums below
    const double gl0 = at(ub(P->glam), cell), gm0 = at(ub(P->gmu), cell);
    R s1r[NG][NDOF] = {};
    if (on) {
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const int pt = s * NG + i;
        const R w = sW2[pt];
        const R la = m[ELEM ? 0 : i][0], mu = m[ELEM ? 0 : i][1], kx = la + 2 * mu;
        const R A0 = w * kx * g0, A1 = w * la * g2, A2 = w * kx * g1;
        const R A3 = w * mu * g1, A4 = w * mu * g2, A5 = w * mu * g0;
        R pxi[NDOF];
        pgrad(i, pxi);
        const LV pv = ex[pt];
        const R pxx = pxi[0], pxz = pxi[1], pex = lv_get<R, NDOF>(pv, 0), pez = lv_get<R, NDOF>(pv, 1);
        const R t1[NDOF] = {A0 * pxx + A1 * pez, A3 * pex + A5 * pxz};
        const R t2[NDOF] = {A3 * pex + A4 * pxz, A1 * pxx + A2 * pez};
        ex[pt] = lv_make<R, NDOF>(t2);
#pragma unroll
        for (int q = 0; q < NG; ++q)
#pragma unroll
          for (int c = 0; c < NDOF; ++c) s1r[q][c] += H[q][i] * t1[c];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    {  // rows of the element in order, by its first lane
      double sl = 0, sm = 0;
#pragma unroll
      for (int q = 0; q < NG; ++q) {
        const int from = min(lane - s + q, 63);
        sl += __shfl(rl, from);
        sm += __shfl(rmu, from);
      }
      if (on && s == 0) {
        at(ub(P->glam), cell) = gl0 + sl;
        at(ub(P->gmu), cell) = gm0 + sm;
      }
    }
    wave_order();
#pragma unroll
    for (int r = 0; r < TS_ITER; ++r) {
      const int p = ts + TS_NT * r, Z = p / PS, X = p - Z * PS;
      const I g = nidx(min(X, PX - 1), min(Z, PZ - 1));
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        ad[r][c] = at(ub(P->ad + c * S), g);
        av[r][c] = at(ub(P->w + c * S), g);
      }
    }
    el_divergence<R, NDOF>(on, s, ex, H);
    wave_order();
    el_force<R, NDOF, false>(on, lane < TS_EPW * NG && e < NEL, false, base, s, e, ex, Uf, Uf, (const R*)nullptr,
                             (const R*)nullptr, s1r);
  }
  __syncthreads();
  const uint32_t fbase = (uint32_t)t * SLOTS;
#pragma unroll
  for (int r = 0; r < TS_ITER; ++r) {
    const int p = ts + TS_NT * r, Z = p / PS, X = p - Z * PS;
    if (X < PX && Z < PZ) {
      const NodeSlots sl = Eg[p];
      const LV f0 = Ex[sl.q[0]], f1 = Ex[sl.q[1]], f2 = Ex[sl.q[2]], f3 = Ex[sl.q[3]];
      const I g = nidx(X, Z);
      int slot = perim_slot(X, Z, PX, PZ);
      if (const int k = special(p); k >= 0) slot = PERIM_MAX + k;
      R F[NDOF];
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        F[c] = ((lv_get<R, NDOF>(f0, c) + lv_get<R, NDOF>(f1, c)) + lv_get<R, NDOF>(f2, c)) + lv_get<R, NDOF>(f3, c);
        av[r][c] = av[r][c] + dt * ad[r][c];
      }
      if (inj && field == 0) inject(g, ad[r][0], ad[r][1]);
      if (inj && field == 1) inject(g, av[r][0], av[r][1]);
#pragma unroll
      for (int c = 0; c < NDOF; ++c) {
        if (slot >= 0) {
          at(ub(P->fpart + c * P->FPS), fbase + slot) = F[c];
        } else {
          at(ub(P->ad + c * S), g) = ad[r][c] + F[c];
          at(ub(P->w + c * S), g) = av[r][c];
        }
      }
    }
  }
}

// Adjoint step at the deferred nodes (tile perimeters, source nodes): the partial
// forces -K^T fb of the tiles, the absorbing term, the mass and ABC sensitivities.
// gabs[c][q] accumulates dJ/dC_c of the node (for nodes with absorbing entries):
// -fb_c (vp_c + c3 a_c), vp = v_{n-1} + c2 a_{n-1} the forward predicted velocity.
template <typename R>
__global__ __launch_bounds__(256) void k_adj_deferred(int ndef, DefTable defs,
                                                      const int* __restrict__ part_off, const R* __restrict__ fpart,
                                                      size_t FPS, const double* __restrict__ abso,
                                                      const R* __restrict__ rmdef, R* __restrict__ ad,
                                                      R* __restrict__ aw, size_t GS,
                                                      const R* __restrict__ afw, const R* __restrict__ vprev,
                                                      const R* __restrict__ aprev, double* __restrict__ mbar,
                                                      double* __restrict__ gabs, R dt, R c1, R c2, R c3,
                                                      const R* __restrict__ dcur = nullptr,
                                                      const R* __restrict__ dprev = nullptr,
                                                      const R* __restrict__ dnext = nullptr, double idt = 0.0,
                                                      double idt2 = 0.0, InjectPlan IP = {}) {
  constexpr int NDOF = 2;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ndef) return;
  const DefNode n = def_unpack(defs, q);
  const size_t g = n.g;
  const int u = IP.g ? IP.udef[q] : -1;
  // all loads first
  R xd[NDOF], xw[NDOF], rm[NDOF], u0[NDOF], u1[NDOF], u2[NDOF], F[NDOF];
  double C[NDOF] = {}, gb[NDOF] = {};
  const bool two = n.pinl && n.poff[1] >= 0;
  const int o0 = n.pinl ? n.poff[0] : 0, o1 = two ? n.poff[1] : o0;
  R p0[NDOF], p1[NDOF];
  double mb = mbar[g];
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    const size_t i = c * GS + g;
    xd[c] = ad[i];
    xw[c] = aw[i];
    rm[c] = rmdef[(size_t)c * ndef + q];
    p0[c] = fpart[c * FPS + o0];
    p1[c] = fpart[c * FPS + o1];
    if (dcur) {
      u0[c] = dcur[i];
      u1[c] = dprev[i];
      u2[c] = afw ? afw[i] : dnext[i];
    } else {
      u0[c] = afw[i];
      u1[c] = 0, u2[c] = 0;
      if (n.acnt > 0) u1[c] = vprev[i], u2[c] = aprev[i];
    }
    if (n.acnt > 0) {
      C[c] = abso[(size_t)n.astart * NDOF + c];
      gb[c] = gabs[(size_t)c * ndef + q];
    }
  }
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    F[c] = 0;
    if (n.pinl) {  // the loop below with pcnt = 1 or 2
      F[c] = F[c] + p0[c];
      if (two) F[c] = F[c] + p1[c];
    } else {
      for (int k = 0; k < n.pcnt; ++k) F[c] = F[c] + fpart[c * FPS + part_off[n.pstart + k]];
    }
  }
  double sum = 0;
#pragma unroll
  for (int c = 0; c < NDOF; ++c) {
    AdjNode<R> s = adj_node<R>(xd[c], xw[c], dt, c1, c2);
    if (u >= 0) {
      R& x = IP.field == 0 ? s.d : (IP.field == 1 ? s.v : s.a);
      x = inject_at<R>(IP, u, c, x);
    }
    const R fb = (s.a + c3 * s.v) * rm[c];
    double Cc = 0;
    for (int k = 0; k < n.acnt; ++k) Cc += k == 0 ? C[c] : abso[(size_t)(n.astart + k) * NDOF + c];
    ad[c * GS + g] = s.d + F[c];
    aw[c * GS + g] = (R)((double)s.v - Cc * (double)fb);
    // with a displacement history (dcur set) the predicted velocity is
    // velocity v_{n-1} + dt/2 a_{n-1} = (d_n - d_{n-1}) / dt
    double an = (double)u0[c];
    if (dcur) an = afw ? (double)u2[c] : fwd_accel((double)u1[c], (double)u0[c], (double)u2[c], idt2);
    sum -= (double)fb * an;
    if (n.acnt > 0) {
      const double vp = dcur ? ((double)u0[c] - (double)u1[c]) * idt : (double)u1[c] + (double)c2 * (double)u2[c];
      gabs[(size_t)c * ndef + q] = gb[c] - (double)fb * (vp + (double)c3 * an);
    }
  }
  mbar[g] = mb + sum;
}

}  // namespace sem2d
