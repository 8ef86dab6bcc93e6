// mg.hip -- aggregation multigrid preconditioner for the linearised staggered
// DIVA/SSA system (src/ice_velocity_module.f90:1762-2589), in FP64 or FP32.
//
// Level 0 is the matrix-free fine operator (stencil.h).  Coarse levels hold
// explicit staggered 9-point stencils built on the device as Galerkin products
// R A P, with P piecewise constant on 2 x 2 aggregates of each velocity
// component ('infinite' boundary unknowns follow the aggregate of their
// interior source; 'zero' and 'periodic' boundary unknowns get no coarse
// counterpart) and R = P^T over the interior and calving-front rows.  A 2 x 2
// aggregation of the staggered u (cx) and v (cy) points keeps the u-v coupling
// pattern of the fine rows, so every coarse level has the same 9-point form.
// Smoothing is one four-colour Gauss-Seidel sweep (u red, u black, v red,
// v black, then the boundary rows at level 0) before and after the coarse
// correction; each member's coarsest level (at most IMAU_CMAX x IMAU_CMAX)
// is solved by symmetric Gauss-Seidel sweeps in LDS by one workgroup.
#include <type_traits>

#include "mg.h"
#include "stencil.h"

// the FP32 V-cycle (a preconditioner) divides by the diagonal with the
// hardware reciprocal (v_rcp_f32, about 1 ulp); the FP64 one divides exactly
__device__ __forceinline__ float mdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double mdiv(double a, double b) { return a / b; }

#define TILE_SETUP                                  \
  const int tb = imau_xcd_tile();                   \
  const Tile t = tiles[tb];                         \
  const Member m = mem[t.g];                        \
  const int j = t.j0 + (int)threadIdx.x;

#define CTILE_SETUP                                  \
  const int tb = imau_xcd_tile();                    \
  const Tile t = L.tiles[tb];                        \
  const CMember cm = L.mem[t.g];                     \
  const int J = t.j0 + (int)threadIdx.x;

#define FOR_TILE_ROWS for (int ii = threadIdx.y; ii < IMAU_TI; ii += IMAU_WG_I)

namespace {

template <class T>
struct VecT {
  T *u, *v;
};
template <class T>
struct CVecT {
  const T *u, *v;
};

__device__ __forceinline__ long long cp2(const CMember &m, int J, int I) { return m.off + (long long)I * m.ny + J; }

__device__ __forceinline__ bool cvalid(const CMember &m, int comp, int J, int I) {
  return comp == 0 ? (J >= 0 && I >= 0 && J < m.nyu && I < m.nxu) : (J >= 0 && I >= 0 && J < m.nyv && I < m.nxv);
}

// coarse slot of the coupling from a row of component rowc to an unknown of
// component colc at aggregate offset (dJ, dI); -1 outside the 9-point pattern
__device__ __forceinline__ int agg_slot(int rowc, int colc, int dJ, int dI) {
  if (rowc == colc) {
    if (dJ == 0 && dI == 0) return 0;
    if (dJ == 0 && dI == -1) return 1;
    if (dJ == 0 && dI == 1) return 2;
    if (dJ == -1 && dI == 0) return 3;
    if (dJ == 1 && dI == 0) return 4;
    return -1;
  }
  if (rowc == 0) {  // u row, v column
    if (dJ == -1 && dI == 0) return 5;
    if (dJ == -1 && dI == 1) return 6;
    if (dJ == 0 && dI == 0) return 7;
    if (dJ == 0 && dI == 1) return 8;
    return -1;
  }
  if (dJ == 0 && dI == -1) return 5;  // v row, u column
  if (dJ == 0 && dI == 0) return 6;
  if (dJ == 1 && dI == -1) return 7;
  if (dJ == 1 && dI == 0) return 8;
  return -1;
}

// unknown (component cc, JJ, II) addressed by slot k of a row of component rowc at (J, I)
__device__ __forceinline__ void slot_pos(int rowc, int k, int J, int I, int &cc, int &JJ, int &II) {
  if (k < 5) {
    cc = rowc;
    JJ = J + (k == 3 ? -1 : (k == 4 ? 1 : 0));
    II = I + (k == 1 ? -1 : (k == 2 ? 1 : 0));
  } else if (rowc == 0) {
    cc = 1;
    JJ = J + (k < 7 ? -1 : 0);
    II = I + ((k & 1) ? 0 : 1);
  } else {
    cc = 0;
    JJ = J + (k < 7 ? 0 : 1);
    II = I + ((k & 1) ? -1 : 0);
  }
}

// nonzeros of the fine u row (interior or calving front) at (j,i):
// f(comp, dj, di, value) for the unknown (comp, j + dj, i + di).  The offsets
// of an interior row are constants, so a caller that unrolls over the rows of
// an aggregate resolves every coarse slot at compile time.
// CROSS: 1 / 0 fixes the cross-term choice at compile time, -1 reads kp.cross
template <int CROSS, class F>
__device__ __forceinline__ void u_couplings(const Member &m, const KP &kp, const CoefT<double> &c, int j, int i,
                                            uint8_t rt, F &&f) {
  const double dx2 = m.dx * m.dx;
  if (rt == RT_FREE) {
    if (CROSS >= 0 ? CROSS != 0 : kp.cross != 0) {
      const double Na0 = c.Na[p2(m, j, i)], Na1 = c.Na[p2(m, j, i + 1)];
      const double Nb0 = c.Nb[p2(m, j, i)], Nbm = c.Nb[p2(m, j - 1, i)];
      f(0, 0, 1, 4.0 * Na1); f(0, 0, -1, 4.0 * Na0); f(0, 1, 0, Nb0); f(0, -1, 0, Nbm);
      f(0, 0, 0, -4.0 * (Na1 + Na0) + -1.0 * (Nb0 + Nbm) - c.bcx[p2(m, j, i)] * dx2);
      f(1, 0, 0, -2.0 * Na0 - Nb0); f(1, 0, 1, 2.0 * Na1 + Nb0);
      f(1, -1, 0, 2.0 * Na0 + Nbm); f(1, -1, 1, -2.0 * Na1 - Nbm);
    } else {
      const double Ncx = c.Ncx[p2(m, j, i)];
      f(0, 0, 1, 4.0); f(0, 0, -1, 4.0); f(0, 1, 0, 1.0); f(0, -1, 0, 1.0);
      f(0, 0, 0, -10.0 - dx2 * c.bcx[p2(m, j, i)] / Ncx);
      f(1, 0, 0, -3.0); f(1, 0, 1, 3.0); f(1, -1, 0, 3.0); f(1, -1, 1, -3.0);
    }
  } else {  // RT_MARGIN_I / RT_MARGIN_O
    const int d1 = (rt == RT_MARGIN_I) ? 0 : 1;  // column i1 = i + d1
    const double Na = c.Na[p2(m, j, i + d1)] / m.dx;
    f(0, 0, d1 - 1, -4.0 * Na); f(0, 0, d1, 4.0 * Na); f(1, -1, d1, -2.0 * Na); f(1, 0, d1, 2.0 * Na);
  }
}
template <int CROSS, class F>
__device__ __forceinline__ void v_couplings(const Member &m, const KP &kp, const CoefT<double> &c, int j, int i,
                                            uint8_t rt, F &&f) {
  const double dx2 = m.dx * m.dx;
  if (rt == RT_FREE) {
    if (CROSS >= 0 ? CROSS != 0 : kp.cross != 0) {
      const double Na0 = c.Na[p2(m, j, i)], Na1 = c.Na[p2(m, j + 1, i)];
      const double Nb0 = c.Nb[p2(m, j, i)], Nbm = c.Nb[p2(m, j, i - 1)];
      f(1, 1, 0, 4.0 * Na1); f(1, -1, 0, 4.0 * Na0); f(1, 0, 1, Nb0); f(1, 0, -1, Nbm);
      f(1, 0, 0, -4.0 * (Na1 + Na0) + -1.0 * (Nb0 + Nbm) - c.bcy[p2(m, j, i)] * dx2);
      f(0, 1, -1, -2.0 * Na1 - Nbm); f(0, 1, 0, 2.0 * Na1 + Nb0);
      f(0, 0, -1, 2.0 * Na0 + Nbm); f(0, 0, 0, -2.0 * Na0 - Nb0);
    } else {
      const double Ncy = c.Ncy[p2(m, j, i)];
      f(1, 1, 0, 4.0); f(1, -1, 0, 4.0); f(1, 0, 1, 1.0); f(1, 0, -1, 1.0);
      f(1, 0, 0, -10.0 - dx2 * c.bcy[p2(m, j, i)] / Ncy);
      f(0, 1, -1, -3.0); f(0, 1, 0, 3.0); f(0, 0, -1, 3.0); f(0, 0, 0, -3.0);
    }
  } else {
    const int d1 = (rt == RT_MARGIN_I) ? 0 : 1;  // row j1 = j + d1
    const double Na = c.Na[p2(m, j + d1, i)] / m.dx;
    f(1, d1 - 1, 0, -4.0 * Na); f(1, d1, 0, 4.0 * Na); f(0, d1, -1, -2.0 * Na); f(0, d1, 0, 2.0 * Na);
  }
}

// level-1 aggregate of the fine unknown (comp, jj, ii); false if it has none
__device__ __forceinline__ bool fine_agg(const Member &m, const uint8_t *rt_u, const uint8_t *rt_v, int comp, int jj,
                                         int ii, int &J, int &I) {
  uint8_t rt = comp == 0 ? rt_u[p2(m, jj, ii)] : rt_v[p2(m, jj, ii)];
  if (rt == RT_BND_INF) {
    int jo, io;
    bnd_src(rt, ii, jj, comp == 0 ? m.nx - 2 : m.nx - 1, comp == 0 ? m.ny - 1 : m.ny - 2, jo, io);
    jj = jo;
    ii = io;
    rt = comp == 0 ? rt_u[p2(m, jj, ii)] : rt_v[p2(m, jj, ii)];
  }
  if (!in_row(rt)) return false;
  J = jj >> 1;
  I = ii >> 1;
  return true;
}

__device__ __forceinline__ bool fine_valid(const Member &m, int comp, int j, int i) {
  return comp == 0 ? (i <= m.nx - 2 && j <= m.ny - 1) : (i <= m.nx - 1 && j <= m.ny - 2);
}

// ---------------------------------------------------------------------------
// Galerkin products
// ---------------------------------------------------------------------------
// fine (level 0, FP64 coefficients) -> level 1
// fine -> level 1 on the cells that are not plain (boundary rows, calving
// fronts, zero rows and their neighbours): a compact list built with the
// flags, so no wavefront of the interior waits for one such lane.
// Every coupling's unknown is mapped to its aggregate (fine_agg) and slot at
// run time, a chain of three dependent loads (row type, the unknown's row type,
// for 'infinite' boundaries its source's).  Bound by that latency: one thread
// per cell walked its eight rows and their couplings in turn (34-48 us, whatever
// the size); here eight lanes share a cell (component x fine row), a row's
// couplings are gathered first so that their loads are in flight together, and
// four lanes add the slots of a component, in the order of the rows: 10.7 us on the
// 401 x 41 channel (36 before), 14.6 us on 12 caps of 96-512 cells (46 before).
template <class T, int CROSS>
__global__ void __launch_bounds__(256) k_gal0_list(const Member *__restrict__ mem, const KP kp, const CoefT<double> c,
                                                   CLevelT<T> L, const int *__restrict__ active,
                                                   const uint8_t *__restrict__ plain, const int2 *__restrict__ list,
                                                   int n) {
  const int idx = (int)(blockIdx.x * 256 + threadIdx.x);
  const int comp = (idx >> 2) & 1, dj = (idx >> 1) & 1, di = idx & 1;
  const int2 e = list[min(idx >> 3, n - 1)];
  const CMember cm = L.mem[e.x];
  const Member m = mem[e.x];
  const int I = e.y / cm.ny, J = e.y - I * cm.ny;
  const long long pc = cm.off + e.y;
  const bool own = (idx >> 3) < n && active[e.x] && cvalid(cm, comp, J, I) && !((plain[pc] >> comp) & 1);
  double val[9];
  int slot[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) { val[k] = 0.0; slot[k] = -1; }
  const int j = 2 * J + dj, i = 2 * I + di;
  if (own && fine_valid(m, comp, j, i)) {
    const uint8_t rt = comp == 0 ? c.rt_u[p2(m, j, i)] : c.rt_v[p2(m, j, i)];
    if (in_row(rt)) {
      int cc[9], jj[9], ii[9], num = 0;
#pragma unroll
      for (int k = 0; k < 9; ++k) { cc[k] = comp; jj[k] = j; ii[k] = i; }
      auto put = [&](int c2, int oj, int oi, double v) {
        cc[num] = c2; jj[num] = j + oj; ii[num] = i + oi; val[num] = v;
        ++num;
      };
      if (comp == 0) u_couplings<CROSS>(m, kp, c, j, i, rt, put);
      else v_couplings<CROSS>(m, kp, c, j, i, rt, put);
      uint8_t rk[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) rk[k] = (cc[k] == 0 ? c.rt_u : c.rt_v)[p2(m, jj[k], ii[k])];
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        if (rk[k] == RT_BND_INF) {
          int jo, io;
          bnd_src(rk[k], ii[k], jj[k], cc[k] == 0 ? m.nx - 2 : m.nx - 1, cc[k] == 0 ? m.ny - 1 : m.ny - 2, jo, io);
          jj[k] = jo;
          ii[k] = io;
          rk[k] = (cc[k] == 0 ? c.rt_u : c.rt_v)[p2(m, jo, io)];
        }
        slot[k] = in_row(rk[k]) ? agg_slot(comp, cc[k], (jj[k] >> 1) - J, (ii[k] >> 1) - I) : -1;
      }
    }
  }
  // lane a of the four sums the slots a, a + 4, a + 8, over the rows in the
  // order (dj, di) = (0,0), (0,1), (1,0), (1,1) and each row's couplings in turn
  const int a = idx & 3;
  double sum[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int row = 0; row < 4; ++row)
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const double v = __shfl(val[k], row, 4);
      const int s = __shfl(slot[k], row, 4);
#pragma unroll
      for (int n = 0; n < 3; ++n) sum[n] += (s == a + 4 * n) ? v : 0.0;
    }
  T *dst = comp == 0 ? L.cu : L.cv;
#pragma unroll
  for (int n = 0; n < 3; ++n)
    if (own && a + 4 * n < 9) dst[(a + 4 * n) * L.na + pc] = (T)sum[n];
}

// Plain aggregates: all four fine rows of a level-1 aggregate of component
// comp are interior rows (RT_FREE) and every unknown their couplings reach is
// an interior or calving-front unknown.  The aggregate of each such unknown
// is then (j >> 1, i >> 1), so a coupling's coarse slot follows from its
// offsets alone.  Bit comp of plain[level-1 cell]; once per solve (the row
// types are fixed for a solve).
__device__ __forceinline__ bool plain_row(const Member &m, const uint8_t *rt_u, const uint8_t *rt_v, int comp, int j,
                                          int i) {
  if (!fine_valid(m, comp, j, i)) return false;
  if ((comp == 0 ? rt_u[p2(m, j, i)] : rt_v[p2(m, j, i)]) != RT_FREE) return false;
  // the unknowns of u_couplings / v_couplings for an interior row
  bool ok;
  if (comp == 0)
    ok = in_row(rt_u[p2(m, j, i + 1)]) && in_row(rt_u[p2(m, j, i - 1)]) && in_row(rt_u[p2(m, j + 1, i)]) &&
         in_row(rt_u[p2(m, j - 1, i)]) && in_row(rt_v[p2(m, j, i)]) && in_row(rt_v[p2(m, j, i + 1)]) &&
         in_row(rt_v[p2(m, j - 1, i)]) && in_row(rt_v[p2(m, j - 1, i + 1)]);
  else
    ok = in_row(rt_v[p2(m, j + 1, i)]) && in_row(rt_v[p2(m, j - 1, i)]) && in_row(rt_v[p2(m, j, i + 1)]) &&
         in_row(rt_v[p2(m, j, i - 1)]) && in_row(rt_u[p2(m, j + 1, i - 1)]) && in_row(rt_u[p2(m, j + 1, i)]) &&
         in_row(rt_u[p2(m, j, i - 1)]) && in_row(rt_u[p2(m, j, i)]);
  return ok;
}
// The cells with a valid component that is not plain are appended to list
// (member, index within the member's level), counted in *n (zeroed first).
__global__ void __launch_bounds__(IMAU_WG) k_gal_plain_flags(const Member *__restrict__ mem,
                                                             const uint8_t *__restrict__ rt_u,
                                                             const uint8_t *__restrict__ rt_v, CLevelT<float> L,
                                                             uint8_t *__restrict__ plain, int2 *__restrict__ list,
                                                             int *__restrict__ n) {
  CTILE_SETUP
  if (J >= cm.ny) return;
  const Member m = mem[t.g];
  FOR_TILE_ROWS {
    const int I = t.i0 + ii;
    if (I >= cm.nx) break;
    int fl = 0, valid = 0;
    for (int comp = 0; comp < 2; ++comp) {
      bool ok = cvalid(cm, comp, J, I);
      if (ok) valid |= 1 << comp;
      for (int q = 0; q < 4 && ok; ++q) ok = plain_row(m, rt_u, rt_v, comp, 2 * J + (q >> 1), 2 * I + (q & 1));
      if (ok) fl |= 1 << comp;
    }
    plain[cp2(cm, J, I)] = (uint8_t)fl;
    // one atomic per wavefront: the lanes with a cell to append take
    // consecutive slots after the wavefront's base
    const bool add = (valid & ~fl) != 0;
    const unsigned long long mask = __ballot(add);
    if (mask) {
      const int lane = (int)__lane_id(), lead = __ffsll((long long)mask) - 1;
      int base = 0;
      if (lane == lead) base = atomicAdd(n, __popcll(mask));
      base = __shfl(base, lead);
      if (add) list[base + __popcll(mask & ((1ull << lane) - 1ull))] = make_int2(t.g, I * cm.ny + J);
    }
  }
}

// one fine row (2J+DJ, 2I+DI) of a plain aggregate: every coupling offset is a
// literal after inlining, so the slot is a constant and cf stays in registers
template <int CROSS, int COMP, int DJ, int DI>
__device__ __forceinline__ void gal_plain_row(const Member &m, const KP &kp, const CoefT<double> &c, int J, int I,
                                              double (&cf)[9]) {
  auto acc = [&](int cc, int oj, int oi, double val) {
    const int s = agg_slot(COMP, cc, (DJ + oj) >> 1, (DI + oi) >> 1);
    if (s >= 0) cf[s] += val;
  };
  if (COMP == 0) u_couplings<CROSS>(m, kp, c, 2 * J + DJ, 2 * I + DI, RT_FREE, acc);
  else v_couplings<CROSS>(m, kp, c, 2 * J + DJ, 2 * I + DI, RT_FREE, acc);
}

// fine -> level 1 on the plain aggregates: the same sums in the same order as
// k_gal0_list, with straight-line loads and no aggregate look-ups
template <class T, int CROSS, int COMP>
__device__ __forceinline__ void gal_plain(const Member &m, const KP &kp, const CoefT<double> &c, const CLevelT<T> &L,
                                          int J, int I, long long pc) {
  double cf[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  gal_plain_row<CROSS, COMP, 0, 0>(m, kp, c, J, I, cf);
  gal_plain_row<CROSS, COMP, 0, 1>(m, kp, c, J, I, cf);
  gal_plain_row<CROSS, COMP, 1, 0>(m, kp, c, J, I, cf);
  gal_plain_row<CROSS, COMP, 1, 1>(m, kp, c, J, I, cf);
  T *dst = COMP == 0 ? L.cu : L.cv;
#pragma unroll
  for (int k = 0; k < 9; ++k) dst[k * L.na + pc] = (T)cf[k];
}
template <class T, int CROSS>
__global__ void __launch_bounds__(IMAU_WG) k_gal0_plain(const Member *__restrict__ mem, const KP kp,
                                                        const CoefT<double> c, CLevelT<T> L,
                                                        const int *__restrict__ active,
                                                        const uint8_t *__restrict__ plain) {
  CTILE_SETUP
  if (J >= cm.ny || !active[t.g]) return;
  const Member m = mem[t.g];
  FOR_TILE_ROWS {
    const int I = t.i0 + ii;
    if (I >= cm.nx) break;
    const long long pc = cp2(cm, J, I);
    const int fl = plain[pc];
    if (fl & 1) gal_plain<T, CROSS, 0>(m, kp, c, L, J, I, pc);
    if (fl & 2) gal_plain<T, CROSS, 1>(m, kp, c, L, J, I, pc);
  }
}

// level l (Fl) -> level l+1 (L), accumulated in FP64; two workgroups per tile,
// one per component.  Slot k of a fine row addresses the unknown at constant
// offsets, so its coarse slot is a constant, at the level's edges too: a slot
// whose unknown lies outside the level holds zero (no sum ever writes another
// value into it), and only whole fine cells past an odd edge have to be masked.
// Bound by load latency, so the 36 coefficients of a cell are loaded before any
// is added; testing every coupling's bounds instead, with a straight-line path
// for the interior beside it, serialised the loads: 38-41 us, now 6.1 us (401 x
// 41 channel, FP64) and 7.2 us (12 caps, FP32).
template <class T, int COMP>
__device__ __forceinline__ void galc_cell(const CLevelT<T> &Fl, const CMember &fm, const CLevelT<T> &L, int J, int I,
                                          long long pc) {
  const T *src = COMP == 0 ? Fl.cu : Fl.cv;
  T v[4][9];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = 2 * J + (q >> 1), i = 2 * I + (q & 1);
    const bool ok = cvalid(fm, COMP, j, i);
    const long long pf = ok ? cp2(fm, j, i) : cp2(fm, 2 * J, 2 * I);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const T a = src[k * Fl.na + pf];
      v[q][k] = ok ? a : (T)0.0;
    }
  }
  double cf[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      int cc, jj, i2;
      slot_pos(COMP, k, q >> 1, q & 1, cc, jj, i2);  // offsets from the coarse cell's first fine cell
      const int s = agg_slot(COMP, cc, jj >> 1, i2 >> 1);
      if (s >= 0) cf[s] += (double)v[q][k];
    }
  T *dst = COMP == 0 ? L.cu : L.cv;
#pragma unroll
  for (int k = 0; k < 9; ++k) dst[k * L.na + pc] = (T)cf[k];
}

template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_galc(CLevelT<T> Fl, CLevelT<T> L, const int *__restrict__ active) {
  const int tp = imau_xcd_tile(), comp = tp & 1;
  const Tile t = L.tiles[tp >> 1];
  const CMember cm = L.mem[t.g];
  const int J = t.j0 + (int)threadIdx.x;
  if (J >= cm.ny || !active[t.g] || L.depth[t.g] < L.lev) return;
  const CMember fm = Fl.mem[t.g];
  FOR_TILE_ROWS {
    const int I = t.i0 + ii;
    if (I >= cm.nx) break;
    const long long pc = cp2(cm, J, I);
    if (comp == 0) {
      if (cvalid(cm, 0, J, I)) galc_cell<T, 0>(Fl, fm, L, J, I, pc);
    } else {
      if (cvalid(cm, 1, J, I)) galc_cell<T, 1>(Fl, fm, L, J, I, pc);
    }
  }
}

// ---------------------------------------------------------------------------
// coarse-level smoothing and transfers
// ---------------------------------------------------------------------------
// off-diagonal sum S and diagonal D of a coarse row at (J,I)
template <class T>
__device__ __forceinline__ void crow(const CLevelT<T> &L, const CMember &m, int comp, int J, int I, const T *xu,
                                     const T *xv, T &S, T &D) {
  const long long p = cp2(m, J, I);
  const T *cf = comp == 0 ? L.cu : L.cv;
  D = cf[p];
  S = (T)0.0;
#pragma unroll
  for (int k = 1; k < 9; ++k) {
    int cc, JJ, II;
    slot_pos(comp, k, J, I, cc, JJ, II);
    if (!cvalid(m, cc, JJ, II)) continue;
    S += cf[k * L.na + p] * (cc == 0 ? xu : xv)[cp2(m, JJ, II)];
  }
}

// one colour (0 u red, 1 u black, 2 v red, 3 v black) of Gauss-Seidel, in place
template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_cgs(CLevelT<T> L, int color, const int *__restrict__ active) {
  CTILE_SETUP
  if (J >= cm.ny || !active[t.g] || L.depth[t.g] <= L.lev) return;
  const int comp = color >> 1;
  FOR_TILE_ROWS {
    const int I = t.i0 + ii;
    if (I >= cm.nx) break;
    if (((I + J) & 1) != (color & 1) || !cvalid(cm, comp, J, I)) continue;
    T S, D;
    crow(L, cm, comp, J, I, L.xu, L.xv, S, D);
    const long long p = cp2(cm, J, I);
    const T b = (comp == 0 ? L.bu : L.bv)[p];
    (comp == 0 ? L.xu : L.xv)[p] = (D != (T)0.0) ? mdiv(b - S, D) : (T)0.0;
  }
}

// Fused sweeps of a coarse level, one launch each way.  A tile (IMAU_TI x
// IMAU_TJ) plus a halo of H cells is held in LDS; the four colour phases update
// shrinking regions (after phase p the values are exact up to H - 1 - p cells
// beyond the tile, because every row couples only neighbours at distance one).
//   k_cdown: the pre-smoothing sweep from zero (H = 5: exact one cell beyond the
//     tile), the residual of the tile and its restriction to the next level;
//   k_cup: the iterate plus the prolonged next level, staged as the sum, and
//     the reversed sweep (H = 4), written to the second buffer.
// The results equal one launch per colour, k_crestrict and k_cprolong.
//
// Coarse levels are bound by the latency of their loads, not by bytes: a level
// of a 401 x 41 grid is a handful of workgroups.  So each thread owns at most
// two rows of a colour (CTH threads cover a colour's region, the first one in
// two steps), the rows' coefficients are loaded into registers for all four
// phases at once before the first barrier, and the phases touch only LDS.
// Neighbours outside the level read the LDS halo, which is zero there, with a
// zero coefficient (the Galerkin sums put nothing into such slots), so no row
// tests its neighbours.  Measured on the 401 x 41 channel (FP64, one V-cycle
// has three such levels): a sweep and a restriction kernel, 13.9 + 20.5 us,
// became k_cdown, 6.6 us; a prolongation and a sweep kernel, 4.6 + 13.9 us,
// became k_cup, 6.9 us (12 ice caps of 96-512 cells a side, FP32: 17 + 29 ->
// 8.1 us down, 4.7 + 17 -> 7.9 us up).
#define CTH 512
static_assert((IMAU_TI + 6) * (IMAU_TJ / 2 + 3) <= CTH && (IMAU_TI + 8) * (IMAU_TJ / 2 + 4) <= 2 * CTH,
              "a colour phase has at most one row per thread, the first of k_cdown two");
template <class T>
struct CRow {
  T cf[9], b;
  int l;     // LDS index of the cell, -1: no row
  bool in;   // the cell lies in the tile
};

// row of phase region cell q (region half-width r around the tile, halo H)
template <class T, int H, int R, int COLOR>
__device__ __forceinline__ void crow_load(const CLevelT<T> &L, const CMember &cm, const Tile &t, int q, CRow<T> &row) {
  constexpr int RH = IMAU_TJ / 2 + R, N = (IMAU_TI + 2 * R) * RH, CRJ = IMAU_TJ + 2 * H, COMP = COLOR >> 1;
  row.l = -1;
  row.in = false;
  if (q >= N) return;
  const int Ib = t.i0 - H, Jb = t.j0 - H;
  const int li = H - R + q / RH;
  const int lj = H - R + 2 * (q % RH) + ((COLOR ^ (Ib + li + Jb + H - R)) & 1);
  const int I = Ib + li, J = Jb + lj;
  if (!cvalid(cm, COMP, J, I)) return;
  const long long p = cp2(cm, J, I);
  const T *cf = COMP == 0 ? L.cu : L.cv;
#pragma unroll
  for (int k = 0; k < 9; ++k) row.cf[k] = cf[k * L.na + p];
  row.b = (COMP == 0 ? L.bu : L.bv)[p];
  row.l = li * CRJ + lj;
  row.in = li >= H && li < H + IMAU_TI && lj >= H && lj < H + IMAU_TJ;
}

// off-diagonal sum of a row from the LDS iterate (su, sv)
template <class T, int COMP, int CRJ>
__device__ __forceinline__ T crow_sum(const CRow<T> &row, const T *su, const T *sv) {
  T S = (T)0.0;
#pragma unroll
  for (int k = 1; k < 9; ++k) {
    int cc, dj, di;
    slot_pos(COMP, k, 0, 0, cc, dj, di);
    S += row.cf[k] * (cc == 0 ? su : sv)[row.l + di * CRJ + dj];
  }
  return S;
}

template <class T, int COMP, int CRJ>
__device__ __forceinline__ void crow_gs(const CRow<T> &row, T *su, T *sv) {
  if (row.l < 0) return;
  const T S = crow_sum<T, COMP, CRJ>(row, su, sv);
  (COMP == 0 ? su : sv)[row.l] = (row.cf[0] != (T)0.0) ? mdiv(row.b - S, row.cf[0]) : (T)0.0;
}

template <class T>
__global__ void __launch_bounds__(CTH) k_cdown(CLevelT<T> L, CLevelT<T> N, const int *__restrict__ active) {
  constexpr int H = 5, CRI = IMAU_TI + 2 * H, CRJ = IMAU_TJ + 2 * H;
  __shared__ T su[CRI * CRJ], sv[CRI * CRJ], sr[2][IMAU_TI * IMAU_TJ];
  const Tile t = L.tiles[imau_xcd_tile()];
  if (!active[t.g] || L.depth[t.g] <= L.lev) return;
  const CMember cm = L.mem[t.g];
  const int tid = threadIdx.x;
  CRow<T> r0, r0b, r1, r2, r3;
  crow_load<T, H, 4, 0>(L, cm, t, tid, r0);
  crow_load<T, H, 4, 0>(L, cm, t, tid + CTH, r0b);
  crow_load<T, H, 3, 1>(L, cm, t, tid, r1);
  crow_load<T, H, 2, 2>(L, cm, t, tid, r2);
  crow_load<T, H, 1, 3>(L, cm, t, tid, r3);
  for (int q = tid; q < CRI * CRJ; q += CTH) {
    su[q] = (T)0.0;
    sv[q] = (T)0.0;
  }
  for (int q = tid; q < IMAU_TI * IMAU_TJ; q += CTH) {
    sr[0][q] = (T)0.0;
    sr[1][q] = (T)0.0;
  }
  __syncthreads();
  crow_gs<T, 0, CRJ>(r0, su, sv);
  crow_gs<T, 0, CRJ>(r0b, su, sv);
  __syncthreads();
  crow_gs<T, 0, CRJ>(r1, su, sv);
  __syncthreads();
  crow_gs<T, 1, CRJ>(r2, su, sv);
  __syncthreads();
  crow_gs<T, 1, CRJ>(r3, su, sv);
  __syncthreads();
  // residual of the tile's rows
  auto res = [&](const CRow<T> &row, T S, const T *x, T *out) {
    const int li = row.l / CRJ - H, lj = row.l % CRJ - H;
    out[li * IMAU_TJ + lj] = row.b - S - row.cf[0] * x[row.l];
  };
  if (r0.in) res(r0, crow_sum<T, 0, CRJ>(r0, su, sv), su, sr[0]);
  if (r0b.in) res(r0b, crow_sum<T, 0, CRJ>(r0b, su, sv), su, sr[0]);
  if (r1.in) res(r1, crow_sum<T, 0, CRJ>(r1, su, sv), su, sr[0]);
  if (r2.in) res(r2, crow_sum<T, 1, CRJ>(r2, su, sv), sv, sr[1]);
  if (r3.in) res(r3, crow_sum<T, 1, CRJ>(r3, su, sv), sv, sr[1]);
  for (int q = tid; q < IMAU_TI * IMAU_TJ; q += CTH) {
    const int li = q / IMAU_TJ, lj = q % IMAU_TJ, I = t.i0 + li, J = t.j0 + lj;
    if (cvalid(cm, 0, J, I)) L.xu[cp2(cm, J, I)] = su[(li + H) * CRJ + lj + H];
    if (cvalid(cm, 1, J, I)) L.xv[cp2(cm, J, I)] = sv[(li + H) * CRJ + lj + H];
  }
  __syncthreads();
  const CMember nm = N.mem[t.g];
  for (int q = tid; q < 2 * (IMAU_TI / 2) * (IMAU_TJ / 2); q += CTH) {
    const int comp = q / ((IMAU_TI / 2) * (IMAU_TJ / 2)), c = q % ((IMAU_TI / 2) * (IMAU_TJ / 2));
    const int li = c / (IMAU_TJ / 2), lj = c % (IMAU_TJ / 2), I = t.i0 / 2 + li, J = t.j0 / 2 + lj;
    if (!cvalid(nm, comp, J, I)) continue;
    const T *s = sr[comp] + 2 * li * IMAU_TJ + 2 * lj;
    (comp == 0 ? N.bu : N.bv)[cp2(nm, J, I)] = (((s[0] + s[IMAU_TJ]) + s[1]) + s[IMAU_TJ + 1]);
  }
}

// L.xu / L.xv: the pre-smoothed iterate; N.xu / N.xv: the next level's result;
// the post-smoothed iterate goes to (xou, xov)
template <class T>
__global__ void __launch_bounds__(CTH) k_cup(CLevelT<T> L, CLevelT<T> N, T *__restrict__ xou, T *__restrict__ xov,
                                            const int *__restrict__ active) {
  constexpr int H = 4, CRI = IMAU_TI + 2 * H, CRJ = IMAU_TJ + 2 * H;
  __shared__ T su[CRI * CRJ], sv[CRI * CRJ];
  const Tile t = L.tiles[imau_xcd_tile()];
  if (!active[t.g] || L.depth[t.g] <= L.lev) return;
  const CMember cm = L.mem[t.g], nm = N.mem[t.g];
  const int tid = threadIdx.x;
  CRow<T> r0, r1, r2, r3;
  crow_load<T, H, 3, 3>(L, cm, t, tid, r0);
  crow_load<T, H, 2, 2>(L, cm, t, tid, r1);
  crow_load<T, H, 1, 1>(L, cm, t, tid, r2);
  crow_load<T, H, 0, 0>(L, cm, t, tid, r3);
  for (int q = tid; q < CRI * CRJ; q += CTH) {
    const int I = t.i0 - H + q / CRJ, J = t.j0 - H + q % CRJ;
    T a = (T)0.0, b = (T)0.0;
    if (cvalid(cm, 0, J, I)) a = L.xu[cp2(cm, J, I)] + N.xu[cp2(nm, J >> 1, I >> 1)];
    if (cvalid(cm, 1, J, I)) b = L.xv[cp2(cm, J, I)] + N.xv[cp2(nm, J >> 1, I >> 1)];
    su[q] = a;
    sv[q] = b;
  }
  __syncthreads();
  crow_gs<T, 1, CRJ>(r0, su, sv);
  __syncthreads();
  crow_gs<T, 1, CRJ>(r1, su, sv);
  __syncthreads();
  crow_gs<T, 0, CRJ>(r2, su, sv);
  __syncthreads();
  crow_gs<T, 0, CRJ>(r3, su, sv);
  __syncthreads();
  for (int q = tid; q < IMAU_TI * IMAU_TJ; q += CTH) {
    const int li = q / IMAU_TJ, lj = q % IMAU_TJ, I = t.i0 + li, J = t.j0 + lj;
    if (cvalid(cm, 0, J, I)) xou[cp2(cm, J, I)] = su[(li + H) * CRJ + lj + H];
    if (cvalid(cm, 1, J, I)) xov[cp2(cm, J, I)] = sv[(li + H) * CRJ + lj + H];
  }
}

// b(l+1) = R (b - A x)(l); one thread per coarse cell
template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_crestrict(CLevelT<T> Fl, CLevelT<T> L, const int *__restrict__ active) {
  CTILE_SETUP
  if (J >= cm.ny || !active[t.g] || Fl.depth[t.g] <= Fl.lev) return;
  const CMember fm = Fl.mem[t.g];
  FOR_TILE_ROWS {
    const int I = t.i0 + ii;
    if (I >= cm.nx) break;
    for (int comp = 0; comp < 2; ++comp) {
      if (!cvalid(cm, comp, J, I)) continue;
      T s = (T)0.0;
      for (int dj = 0; dj < 2; ++dj)
        for (int di = 0; di < 2; ++di) {
          const int j = 2 * J + dj, i = 2 * I + di;
          if (!cvalid(fm, comp, j, i)) continue;
          T S, D;
          crow(Fl, fm, comp, j, i, Fl.xu, Fl.xv, S, D);
          const long long pf = cp2(fm, j, i);
          s += (comp == 0 ? Fl.bu : Fl.bv)[pf] - S - D * (comp == 0 ? Fl.xu : Fl.xv)[pf];
        }
      (comp == 0 ? L.bu : L.bv)[cp2(cm, J, I)] = s;
    }
  }
}

// x(l) += P x(l+1); one thread per fine cell
template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_cprolong(CLevelT<T> Fl, CLevelT<T> L, const int *__restrict__ active) {
  const Tile t = Fl.tiles[imau_xcd_tile()];
  const CMember fm = Fl.mem[t.g];
  const int j = t.j0 + (int)threadIdx.x;
  if (j >= fm.ny || !active[t.g] || Fl.depth[t.g] <= Fl.lev) return;
  const CMember cm = L.mem[t.g];
  FOR_TILE_ROWS {
    const int i = t.i0 + ii;
    if (i >= fm.nx) break;
    const long long pf = cp2(fm, j, i), pc = cp2(cm, j >> 1, i >> 1);
    if (cvalid(fm, 0, j, i)) Fl.xu[pf] += L.xu[pc];
    if (cvalid(fm, 1, j, i)) Fl.xv[pf] += L.xv[pc];
  }
}

// the coarsest level of each member: one workgroup, nsweeps symmetric
// four-colour Gauss-Seidel sweeps from zero with the iterate in LDS.
// Bound by the latency of its chain of colour phases (LDS reads, the row's sum,
// a write, a barrier), so there are as few and as short phases as possible:
//   - thread q owns the q-th red and the q-th black cell (u and v rows, in
//     registers), so all lanes work in every phase and half as many waves meet
//     at its barrier; the launch has only the threads that the level's largest
//     member needs;
//   - a colour updated twice in a row (the turning points of the symmetric
//     sweeps) keeps its values, so it is updated once: 6 nsweeps + 1 phases for 8 nsweeps;
//   - in FP32 the rows are divided by their diagonal beforehand and summed in
//     two halves (in FP64 that would change the rounding of the solves, which a
//     time loop can amplify), and a halo of zeros in LDS replaces the bounds tests.
// 401 x 41 channel (26 x 3 cells, FP64): 19.8 -> 14.7 us (9.7 with divided
// rows); 12 caps of 96-512
// cells (up to 32 x 32, FP32): 18.9 -> 12.2 us.
constexpr int CL = IMAU_CMAX + 2;  // LDS row length, one-cell halo

// FP32: a row divided by its diagonal, x = b - sum_k cf[k] x_k (zero where the
// diagonal is); FP64: the row itself, x = (b - sum_k cf[k] x_k) / D, summed and
// divided as the other smoothers do
template <class T>
struct CoarseRow {
  T cf[8], b, D;  // D: FP64 rows only
  int l;       // LDS index, -1: no row
  long long p;
};

template <class T, int COMP>
__device__ __forceinline__ void coarse_row_load(const CLevelT<T> &L, const CMember &m, int J, int I, bool in,
                                                CoarseRow<T> &r) {
  r.l = -1;
  if (!in || !cvalid(m, COMP, J, I)) return;
  r.p = cp2(m, J, I);
  const T *src = COMP == 0 ? L.cu : L.cv;
  const T D = src[r.p];
  const T inv = sizeof(T) == 8 ? (T)1.0 : D != (T)0.0 ? (T)__builtin_amdgcn_rcpf((float)D) : (T)0.0;
#pragma unroll
  for (int k = 0; k < 8; ++k) r.cf[k] = src[(k + 1) * L.na + r.p] * inv;
  r.b = (COMP == 0 ? L.bu : L.bv)[r.p] * inv;
  r.D = D;
  r.l = (I + 1) * CL + J + 1;
}

template <class T, int COMP>
__device__ __forceinline__ void coarse_row_gs(const CoarseRow<T> &r, T *su, T *sv) {
  if (r.l < 0) return;
  if constexpr (sizeof(T) == 8) {
    T S = (T)0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      int cc, dj, di;
      slot_pos(COMP, k + 1, 0, 0, cc, dj, di);
      S += r.cf[k] * (cc == 0 ? su : sv)[r.l + di * CL + dj];
    }
    (COMP == 0 ? su : sv)[r.l] = (r.D != (T)0.0) ? mdiv(r.b - S, r.D) : (T)0.0;
    return;
  }
  T s[2] = {r.b, (T)0.0};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    int cc, dj, di;
    slot_pos(COMP, k + 1, 0, 0, cc, dj, di);
    s[k & 1] -= r.cf[k] * (cc == 0 ? su : sv)[r.l + di * CL + dj];
  }
  (COMP == 0 ? su : sv)[r.l] = s[0] + s[1];
}

template <class T>
__global__ void __launch_bounds__(IMAU_CMAX *IMAU_CMAX / 2) k_coarsest(CLevelT<T> L, const int *__restrict__ active,
                                                                      int nsweeps) {
  __shared__ T su[CL * CL], sv[CL * CL];
  const int g = blockIdx.x;
  if (!active[g] || L.depth[g] != L.lev) return;
  const CMember cm = L.mem[g];
  const int q = threadIdx.x, half = (cm.ny + 1) / 2, I = q / half, m = 2 * (q - I * half);
  const bool in = I < cm.nx;
  const int J0 = m + (I & 1), J1 = m + ((I + 1) & 1);  // red: I + J even
  CoarseRow<T> u0, u1, v0, v1;
  coarse_row_load<T, 0>(L, cm, J0, I, in, u0);
  coarse_row_load<T, 0>(L, cm, J1, I, in, u1);
  coarse_row_load<T, 1>(L, cm, J0, I, in, v0);
  coarse_row_load<T, 1>(L, cm, J1, I, in, v1);
  for (int k = q; k < CL * CL; k += blockDim.x) {
    su[k] = (T)0.0;
    sv[k] = (T)0.0;
  }
  __syncthreads();
  coarse_row_gs<T, 0>(u0, su, sv);
  __syncthreads();
  for (int sw = 0; sw < nsweeps; ++sw) {
    coarse_row_gs<T, 0>(u1, su, sv);
    __syncthreads();
    coarse_row_gs<T, 1>(v0, su, sv);
    __syncthreads();
    coarse_row_gs<T, 1>(v1, su, sv);
    __syncthreads();
    coarse_row_gs<T, 1>(v0, su, sv);
    __syncthreads();
    coarse_row_gs<T, 0>(u1, su, sv);
    __syncthreads();
    coarse_row_gs<T, 0>(u0, su, sv);
    __syncthreads();
  }
  if (u0.l >= 0) L.xu[u0.p] = su[u0.l];
  if (u1.l >= 0) L.xu[u1.p] = su[u1.l];
  if (v0.l >= 0) L.xv[v0.p] = sv[v0.l];
  if (v1.l >= 0) L.xv[v1.p] = sv[v1.l];
}

// ---------------------------------------------------------------------------
// level 0 (matrix-free fine operator)
// ---------------------------------------------------------------------------
// one colour of Gauss-Seidel on A z = y (colour 4: the domain-boundary rows)
template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_smooth0(const Member *__restrict__ mem, const Tile *__restrict__ tiles,
                                                     const KP kp, const CoefT<T> c, VecT<T> x, CVecT<T> y, int color,
                                                     const int *__restrict__ active) {
  TILE_SETUP
  if (j >= m.ny || !active[t.g]) return;
  const GAccT<T> U{x.u, m}, V{x.v, m};
  const int nx = m.nx, ny = m.ny;
  FOR_TILE_ROWS {
    const int i = t.i0 + ii;
    if (i >= nx) break;
    const long long p = p2(m, j, i);
    if (color < 4) {
      const bool isu = color < 2;
      if (((i + j) & 1) != (color & 1)) continue;
      if (isu && i >= nx - 1) continue;
      if (!isu && j >= ny - 1) continue;
      const uint8_t rt = isu ? c.rt_u[p] : c.rt_v[p];
      if (is_bnd(rt)) continue;
      T S, D;
      if (isu) u_sd<T>(m, kp, c, j, i, rt, U, V, S, D);
      else v_sd<T>(m, kp, c, j, i, rt, U, V, S, D);
      (isu ? x.u : x.v)[p] = mdiv((isu ? y.u : y.v)[p] - S, D);
    } else {
      if (i < nx - 1 && is_bnd(c.rt_u[p])) {
        const uint8_t rt = c.rt_u[p];
        T val = y.u[p];
        if (rt != RT_BND_ZERO) {
          int jo, io;
          bnd_src(rt, i, j, nx - 2, ny - 1, jo, io);
          val += x.u[p2(m, jo, io)];
        }
        x.u[p] = val;
      }
      if (j < ny - 1 && is_bnd(c.rt_v[p])) {
        const uint8_t rt = c.rt_v[p];
        T val = y.v[p];
        if (rt != RT_BND_ZERO) {
          int jo, io;
          bnd_src(rt, i, j, nx - 1, ny - 2, jo, io);
          val += x.v[p2(m, jo, io)];
        }
        x.v[p] = val;
      }
    }
  }
}

// Fused fine-level sweeps, one launch each way.  A tile (IMAU_FTI x IMAU_FTJ)
// plus a halo of H cells is held in LDS; the four colour phases (u red, u black,
// v red, v black; reversed on the way up) update shrinking regions -- every row
// couples only neighbours at distance one -- and then the 'infinite' and 'zero'
// domain-boundary rows are set from their sources.
//   k_fine_down: the sweep from zero (H = 6: exact two cells beyond the tile
//     before the boundary rows, one after them), then the residual of the tile
//     and its restriction to level 1;
//   k_fine_up: the iterate plus the prolonged level 1, staged as the sum, and
//     the reversed sweep (H = 5); the result in the working precision, or
//     (TO = double) in FP64 for the Krylov solver.
// The right-hand side is read in the Krylov solver's FP64.  The results equal
// one launch per colour, k_restrict0 and k_prolong0.  Periodic boundary rows,
// whose sources lie across the domain, are completed by a colour-4 pass of
// k_smooth0, and the restriction then runs on its own (RESTRICT = false).
//
// Bound by load latency at small sizes and by the fine coefficients at large
// ones.  A thread owns at most one row of every colour (FTH threads cover the
// largest region), so the coefficients of its four rows are loaded at once
// before the first barrier and the phases touch only LDS.  401 x 41 channel
// (FP64): sweep 17.1 + restriction 11.5 us -> k_fine_down 10.9 us, prolongation
// 4.6 + sweep 17.1 us -> k_fine_up 10.6 us; 12 caps of 96-512 cells (FP32):
// conversion 8.0 + sweep 30.3 + restriction 23.5 -> 31.7 us, prolongation 10.8 +
// sweep 30.3 + conversion 6.8 -> 34.1 us.
#define FTH 1024

// the coefficients of one fine row held in registers, with the accessors the
// rows of stencil.h read them through; (j, i) is the row's own position
template <class T, int COMP, int CROSS>
struct FRow {
  T n0, n1, nb0, nbm, beta, ns;  // N_a on both sides, N_b on both sides, beta_eff, N on the row's own grid
  T y;
  int j, i, l;                   // l: LDS index of the cell, -1: no row
  uint8_t rt;
  bool in;                       // the cell lies in the tile
  __device__ __forceinline__ T na(const Member &, int jj, int ii) const {
    return (COMP == 0 ? ii == i : jj == j) ? n0 : n1;
  }
  __device__ __forceinline__ T nb(const Member &, int jj, int ii) const {
    return (COMP == 0 ? jj == j : ii == i) ? nb0 : nbm;
  }
  __device__ __forceinline__ T bx(const Member &, int, int) const { return beta; }
  __device__ __forceinline__ T by(const Member &, int, int) const { return beta; }
  __device__ __forceinline__ T ncx(const Member &, int, int) const { return ns; }
  __device__ __forceinline__ T ncy(const Member &, int, int) const { return ns; }
};

// row of phase region cell q (region half-width R around the tile, halo H)
template <class T, int H, int R, int COLOR, int CROSS, class TY>
__device__ __forceinline__ void frow_load(const Member &m, const CoefT<T> &c, const CVecT<TY> &y, const Tile &t, int q,
                                          FRow<T, (COLOR >> 1), CROSS> &r) {
  constexpr int RH = IMAU_FTJ / 2 + R, N = (IMAU_FTI + 2 * R) * RH, RJ = IMAU_FTJ + 2 * H, COMP = COLOR >> 1;
  static_assert(N <= FTH, "one row of every colour per thread");
  r.l = -1;
  r.in = false;
  if (q >= N) return;
  const int ib = t.i0 - H, jb = t.j0 - H;
  const int li = H - R + q / RH;
  const int lj = H - R + 2 * (q % RH) + ((COLOR ^ (ib + li + jb + H - R)) & 1);
  const int i = ib + li, j = jb + lj;
  if (i < 0 || j < 0 || i >= m.nx - (COMP == 0) || j >= m.ny - (COMP == 1)) return;
  const long long p = p2(m, j, i);
  r.j = j;
  r.i = i;
  r.rt = COMP == 0 ? c.rt_u[p] : c.rt_v[p];
  r.y = (T)(COMP == 0 ? y.u : y.v)[p];
  r.n0 = c.Na[p];
  r.n1 = c.Na[COMP == 0 ? p + m.ny : p + 1];
  r.beta = (COMP == 0 ? c.bcx : c.bcy)[p];
  if (CROSS) {
    // the row of the domain's first line is a boundary row: its N_b is not used
    r.nb0 = c.Nb[p];
    r.nbm = c.Nb[COMP == 0 ? p - (j > 0) : p - (i > 0 ? m.ny : 0)];
  } else {
    r.ns = (COMP == 0 ? c.Ncx : c.Ncy)[p];
  }
  if (is_bnd(r.rt)) return;
  r.l = li * RJ + lj;
  r.in = li >= H && li < H + IMAU_FTI && lj >= H && lj < H + IMAU_FTJ;
}

template <class T, int RJ>
struct LAccT {
  const T *base;  // LDS region, element (0,0) at global (ib, jb)
  int ib, jb;
  __device__ __forceinline__ T operator()(int jj, int ii) const { return base[(ii - ib) * RJ + (jj - jb)]; }
};

// the row's off-diagonal sum S and diagonal D at the LDS iterate
template <class T, int COMP, int CROSS, class A>
__device__ __forceinline__ void frow_sd(const Member &m, const KP &kp, const FRow<T, COMP, CROSS> &r, const A &U,
                                        const A &V, T &S, T &D) {
  if (COMP == 0) u_sd_x<CROSS, T>(m, kp, r, r.j, r.i, r.rt, U, V, S, D);
  else v_sd_x<CROSS, T>(m, kp, r, r.j, r.i, r.rt, U, V, S, D);
}
template <class T, int COMP, int CROSS, class A>
__device__ __forceinline__ void frow_gs(const Member &m, const KP &kp, const FRow<T, COMP, CROSS> &r, const A &U,
                                        const A &V, T *x) {
  if (r.l < 0) return;
  T S, D;
  frow_sd<T, COMP, CROSS>(m, kp, r, U, V, S, D);
  x[r.l] = mdiv(r.y - S, D);
}

// 'infinite' and 'zero' domain-boundary rows of the tile and E cells beyond it
template <class T, int H, int E, class TY, class A>
__device__ __forceinline__ void fine_boundary(const Member &m, const CoefT<T> &c, const CVecT<TY> &y, const Tile &t,
                                              int tid, const A &U, const A &V, T *su, T *sv) {
  constexpr int RJ = IMAU_FTJ + 2 * H, BJ = IMAU_FTJ + 2 * E, BI = IMAU_FTI + 2 * E;
  for (int q = tid; q < BI * BJ; q += FTH) {
    const int li = H - E + q / BJ, lj = H - E + q % BJ;
    const int i = t.i0 - H + li, j = t.j0 - H + lj;
    if (i < 0 || j < 0 || i >= m.nx || j >= m.ny) continue;
    // rows of the domain's edges only (u: i = 0, nx-2, j = 0, ny-1; v likewise)
    if (i > 0 && j > 0 && i < m.nx - 2 && j < m.ny - 2) continue;
    const long long p = p2(m, j, i);
    int jo, io;
    if (i < m.nx - 1) {
      const uint8_t rt = c.rt_u[p];
      if (rt == RT_BND_ZERO || rt == RT_BND_INF) {
        T val = (T)y.u[p];
        if (rt == RT_BND_INF) {
          bnd_src(rt, i, j, m.nx - 2, m.ny - 1, jo, io);
          val += U(jo, io);
        }
        su[li * RJ + lj] = val;
      }
    }
    if (j < m.ny - 1) {
      const uint8_t rt = c.rt_v[p];
      if (rt == RT_BND_ZERO || rt == RT_BND_INF) {
        T val = (T)y.v[p];
        if (rt == RT_BND_INF) {
          bnd_src(rt, i, j, m.nx - 1, m.ny - 2, jo, io);
          val += V(jo, io);
        }
        sv[li * RJ + lj] = val;
      }
    }
  }
}
// whether the tile and E cells beyond it reach the domain's edges
__device__ __forceinline__ bool at_edge(const Member &m, const Tile &t, int E) {
  return t.i0 <= E || t.j0 <= E || t.i0 + IMAU_FTI + E > m.nx - 2 || t.j0 + IMAU_FTJ + E > m.ny - 2;
}

template <class T, int CROSS, bool RESTRICT, class TY>
__global__ void __launch_bounds__(FTH) k_fine_down(const Member *__restrict__ mem, const Tile *__restrict__ ftiles,
                                                   const KP kp, const CoefT<T> c, CVecT<TY> y, VecT<T> zout,
                                                   CLevelT<T> N, const int *__restrict__ active) {
  constexpr int H = 6, RI = IMAU_FTI + 2 * H, RJ = IMAU_FTJ + 2 * H;
  __shared__ T su[RI * RJ], sv[RI * RJ], sr[2][IMAU_FTI * IMAU_FTJ];
  const Tile t = ftiles[imau_xcd_tile()];
  if (!active[t.g]) return;
  const Member m = mem[t.g];
  const int tid = threadIdx.x;
  FRow<T, 0, CROSS> r0, r1;
  FRow<T, 1, CROSS> r2, r3;
  frow_load<T, H, 5, 0, CROSS>(m, c, y, t, tid, r0);
  frow_load<T, H, 4, 1, CROSS>(m, c, y, t, tid, r1);
  frow_load<T, H, 3, 2, CROSS>(m, c, y, t, tid, r2);
  frow_load<T, H, 2, 3, CROSS>(m, c, y, t, tid, r3);
  for (int q = tid; q < RI * RJ; q += FTH) {
    su[q] = (T)0.0;
    sv[q] = (T)0.0;
  }
  sr[0][tid] = (T)0.0;
  sr[1][tid] = (T)0.0;
  static_assert(IMAU_FTI * IMAU_FTJ == FTH, "one tile cell per thread");
  __syncthreads();
  const LAccT<T, RJ> U{su, t.i0 - H, t.j0 - H}, V{sv, t.i0 - H, t.j0 - H};
  frow_gs<T, 0, CROSS>(m, kp, r0, U, V, su);
  __syncthreads();
  frow_gs<T, 0, CROSS>(m, kp, r1, U, V, su);
  __syncthreads();
  frow_gs<T, 1, CROSS>(m, kp, r2, U, V, sv);
  __syncthreads();
  frow_gs<T, 1, CROSS>(m, kp, r3, U, V, sv);
  __syncthreads();
  if (at_edge(m, t, 1)) {  // the same for the whole workgroup
    fine_boundary<T, H, 1>(m, c, y, t, tid, U, V, su, sv);
    __syncthreads();
  }
  {
    const int li = tid / IMAU_FTJ, lj = tid % IMAU_FTJ, i = t.i0 + li, j = t.j0 + lj;
    if (i < m.nx && j < m.ny) {
      const long long p = p2(m, j, i);
      if (i < m.nx - 1) zout.u[p] = su[(li + H) * RJ + lj + H];
      if (j < m.ny - 1) zout.v[p] = sv[(li + H) * RJ + lj + H];
    }
  }
  if (!RESTRICT) return;
  auto res = [&](const auto &r, const T *x, T *out) {
    if (!r.in || !in_row(r.rt)) return;
    T S, D;
    frow_sd(m, kp, r, U, V, S, D);
    out[(r.i - t.i0) * IMAU_FTJ + r.j - t.j0] = r.y - S - D * x[r.l];
  };
  res(r0, su, sr[0]);
  res(r1, su, sr[0]);
  res(r2, sv, sr[1]);
  res(r3, sv, sr[1]);
  __syncthreads();
  const CMember nm = N.mem[t.g];
  if (tid < 2 * (IMAU_FTI / 2) * (IMAU_FTJ / 2)) {
    const int comp = tid / ((IMAU_FTI / 2) * (IMAU_FTJ / 2)), q = tid % ((IMAU_FTI / 2) * (IMAU_FTJ / 2));
    const int li = q / (IMAU_FTJ / 2), lj = q % (IMAU_FTJ / 2), I = t.i0 / 2 + li, J = t.j0 / 2 + lj;
    if (cvalid(nm, comp, J, I)) {
      const T *s = sr[comp] + 2 * li * IMAU_FTJ + 2 * lj;
      (comp == 0 ? N.bu : N.bv)[cp2(nm, J, I)] = (((s[0] + s[IMAU_FTJ]) + s[1]) + s[IMAU_FTJ + 1]);
    }
  }
}

// za: the pre-smoothed iterate; N.xu / N.xv: level 1's result
template <class T, int CROSS, class TY, class TO>
__global__ void __launch_bounds__(FTH) k_fine_up(const Member *__restrict__ mem, const Tile *__restrict__ ftiles,
                                                 const KP kp, const CoefT<T> c, CVecT<TY> y, CVecT<T> za, VecT<TO> zout,
                                                 CLevelT<T> N, const int *__restrict__ active) {
  constexpr int H = 5, RI = IMAU_FTI + 2 * H, RJ = IMAU_FTJ + 2 * H;
  __shared__ T su[RI * RJ], sv[RI * RJ];
  const Tile t = ftiles[imau_xcd_tile()];
  if (!active[t.g]) return;
  const Member m = mem[t.g];
  const CMember nm = N.mem[t.g];
  const int tid = threadIdx.x;
  FRow<T, 1, CROSS> r0, r1;
  FRow<T, 0, CROSS> r2, r3;
  frow_load<T, H, 4, 3, CROSS>(m, c, y, t, tid, r0);
  frow_load<T, H, 3, 2, CROSS>(m, c, y, t, tid, r1);
  frow_load<T, H, 2, 1, CROSS>(m, c, y, t, tid, r2);
  frow_load<T, H, 1, 0, CROSS>(m, c, y, t, tid, r3);
  for (int q = tid; q < RI * RJ; q += FTH) {
    const int i = t.i0 - H + q / RJ, j = t.j0 - H + q % RJ;
    T u = (T)0.0, v = (T)0.0;
    if (i >= 0 && j >= 0 && i < m.nx && j < m.ny) {
      const long long p = p2(m, j, i);
      int Jc, Ic;
      if (i < m.nx - 1) {
        u = za.u[p];
        if (fine_agg(m, c.rt_u, c.rt_v, 0, j, i, Jc, Ic)) u += N.xu[cp2(nm, Jc, Ic)];
      }
      if (j < m.ny - 1) {
        v = za.v[p];
        if (fine_agg(m, c.rt_u, c.rt_v, 1, j, i, Jc, Ic)) v += N.xv[cp2(nm, Jc, Ic)];
      }
    }
    su[q] = u;
    sv[q] = v;
  }
  __syncthreads();
  const LAccT<T, RJ> U{su, t.i0 - H, t.j0 - H}, V{sv, t.i0 - H, t.j0 - H};
  frow_gs<T, 1, CROSS>(m, kp, r0, U, V, sv);
  __syncthreads();
  frow_gs<T, 1, CROSS>(m, kp, r1, U, V, sv);
  __syncthreads();
  frow_gs<T, 0, CROSS>(m, kp, r2, U, V, su);
  __syncthreads();
  frow_gs<T, 0, CROSS>(m, kp, r3, U, V, su);
  __syncthreads();
  if (at_edge(m, t, 0)) {  // the same for the whole workgroup
    fine_boundary<T, H, 0>(m, c, y, t, tid, U, V, su, sv);
    __syncthreads();
  }
  const int li = tid / IMAU_FTJ, lj = tid % IMAU_FTJ, i = t.i0 + li, j = t.j0 + lj;
  if (i < m.nx && j < m.ny) {
    const long long p = p2(m, j, i);
    if (i < m.nx - 1) zout.u[p] = (TO)su[(li + H) * RJ + lj + H];
    if (j < m.ny - 1) zout.v[p] = (TO)sv[(li + H) * RJ + lj + H];
  }
}

// level-1 right-hand side: R (y - A z) over the interior and calving-front rows
template <class T, int CROSS>
__global__ void __launch_bounds__(IMAU_WG) k_restrict0(const Member *__restrict__ mem, const KP kp, const CoefT<T> c,
                                                       CVecT<T> y, CVecT<T> z, CLevelT<T> L,
                                                       const int *__restrict__ active) {
  CTILE_SETUP
  if (J >= cm.ny || !active[t.g]) return;
  const Member m = mem[t.g];
  const GAccT<T> U{z.u, m}, V{z.v, m};
  FOR_TILE_ROWS {
    const int I = t.i0 + ii;
    if (I >= cm.nx) break;
    for (int comp = 0; comp < 2; ++comp) {
      if (!cvalid(cm, comp, J, I)) continue;
      T s = (T)0.0;
      for (int dj = 0; dj < 2; ++dj)
        for (int di = 0; di < 2; ++di) {
          const int j = 2 * J + dj, i = 2 * I + di;
          if (!fine_valid(m, comp, j, i)) continue;
          const long long p = p2(m, j, i);
          const uint8_t rt = comp == 0 ? c.rt_u[p] : c.rt_v[p];
          if (!in_row(rt)) continue;
          T S, D;
          if (comp == 0) {
            u_sd_x<CROSS, T>(m, kp, c, j, i, rt, U, V, S, D);
            s += y.u[p] - S - D * z.u[p];
          } else {
            v_sd_x<CROSS, T>(m, kp, c, j, i, rt, U, V, S, D);
            s += y.v[p] - S - D * z.v[p];
          }
        }
      (comp == 0 ? L.bu : L.bv)[cp2(cm, J, I)] = s;
    }
  }
}

// z += P x(1) on the interior, calving-front and 'infinite' boundary unknowns
template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_prolong0(const Member *__restrict__ mem, const Tile *__restrict__ tiles,
                                                      const uint8_t *__restrict__ rt_u, const uint8_t *__restrict__ rt_v,
                                                      VecT<T> z, CLevelT<T> L, const int *__restrict__ active) {
  TILE_SETUP
  if (j >= m.ny || !active[t.g]) return;
  const CMember cm = L.mem[t.g];
  FOR_TILE_ROWS {
    const int i = t.i0 + ii;
    if (i >= m.nx) break;
    const long long p = p2(m, j, i);
    int Jc, Ic;
    if (i < m.nx - 1 && fine_agg(m, rt_u, rt_v, 0, j, i, Jc, Ic)) z.u[p] += L.xu[cp2(cm, Jc, Ic)];
    if (j < m.ny - 1 && fine_agg(m, rt_u, rt_v, 1, j, i, Jc, Ic)) z.v[p] += L.xv[cp2(cm, Jc, Ic)];
  }
}

// z = 0 (and, for FP32, y32 = y) on every cell of the active members
template <class T>
__global__ void __launch_bounds__(IMAU_WG) k_prep(const Member *__restrict__ mem, const Tile *__restrict__ tiles,
                                                  CVecT<double> y64, VecT<T> y, VecT<T> z,
                                                  const int *__restrict__ active) {
  TILE_SETUP
  if (j >= m.ny || !active[t.g]) return;
  FOR_TILE_ROWS {
    const int i = t.i0 + ii;
    if (i >= m.nx) break;
    const long long p = p2(m, j, i);
    z.u[p] = (T)0.0;
    z.v[p] = (T)0.0;
    if constexpr (!std::is_same<T, double>::value) {
      y.u[p] = (T)y64.u[p];
      y.v[p] = (T)y64.v[p];
    }
  }
}

// FP64 result of the FP32 cycle
__global__ void __launch_bounds__(IMAU_WG) k_fin(const Member *__restrict__ mem, const Tile *__restrict__ tiles,
                                                 CVecT<float> z32, VecT<double> z, const int *__restrict__ active) {
  TILE_SETUP
  if (j >= m.ny || !active[t.g]) return;
  FOR_TILE_ROWS {
    const int i = t.i0 + ii;
    if (i >= m.nx) break;
    const long long p = p2(m, j, i);
    z.u[p] = (double)z32.u[p];
    z.v[p] = (double)z32.v[p];
  }
}

// FP32 copies of the fine coefficients the smoother reads
__global__ void __launch_bounds__(IMAU_WG) k_coef32(const Member *__restrict__ mem, const Tile *__restrict__ tiles,
                                                    const CoefT<double> c, imau::MGFine32 o, int sans,
                                                    const int *__restrict__ active) {
  TILE_SETUP
  if (j >= m.ny || !active[t.g]) return;
  FOR_TILE_ROWS {
    const int i = t.i0 + ii;
    if (i >= m.nx) break;
    const long long p = p2(m, j, i);
    o.Na[p] = (float)c.Na[p];
    o.Nb[p] = (float)c.Nb[p];
    o.bcx[p] = (float)c.bcx[p];
    o.bcy[p] = (float)c.bcy[p];
    if (sans) {
      o.Ncx[p] = (float)c.Ncx[p];
      o.Ncy[p] = (float)c.Ncy[p];
    }
  }
}

template <class T>
__global__ void k_fill(T *p, long long n) {
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x)
    p[q] = (T)0.0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
inline dim3 wg() { return dim3(IMAU_TJ, IMAU_WG_I, 1); }

inline CoefT<double> coef64(const imau::Coef &c) {
  return CoefT<double>{c.Na, c.Nb, c.Ncx, c.Ncy, c.bcx, c.bcy, c.taudx, c.taudy, c.frhs, c.rt_u, c.rt_v};
}
inline CoefT<float> coef32(const imau::MGFine32 &f, const imau::Coef &c) {
  return CoefT<float>{f.Na, f.Nb, f.Ncx, f.Ncy, f.bcx, f.bcy, nullptr, nullptr, nullptr, c.rt_u, c.rt_v};
}

template <class T>
CLevelT<T> view(const imau::MGPlan &P, int l) {
  const imau::MGLevelDev &d = P.levels[l];
  CLevelT<T> L{};
  L.mem = d.mem;
  L.tiles = d.tiles;
  L.depth = P.depth;
  L.lev = d.lev;
  L.ntiles = d.ntiles;
  L.na = d.na;
  L.cu = (T *)d.data;
  L.cv = L.cu + 9 * d.na;
  L.xu = L.cv + 9 * d.na;
  L.xv = L.xu + d.na;
  L.bu = L.xv + d.na;
  L.bv = L.bu + d.na;
  return L;
}

// the level with its iterate pointers on the second buffer (after the fused post-smoothing)
template <class T>
CLevelT<T> view2(const imau::MGPlan &P, int l) {
  CLevelT<T> L = view<T>(P, l);
  L.xu = L.bv + L.na;
  L.xv = L.xu + L.na;
  return L;
}

template <class T>
void fill(hipStream_t s, T *p, long long n) {
  int blocks = (int)std::min<long long>((n + 255) / 256, 4096);
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(k_fill<T>, dim3(blocks), dim3(256), 0, s, p, n);
}

template <class T>
void setup_t(const imau::Launch &F, const KP &kp, const imau::Coef &c, const imau::MGPlan &P, const int *act) {
  const CLevelT<T> L1 = view<T>(P, 0);
  auto kp0 = kp.cross ? k_gal0_plain<T, 1> : k_gal0_plain<T, 0>;
  hipLaunchKernelGGL(kp0, dim3(L1.ntiles), wg(), 0, F.s, F.mem, kp, coef64(c), L1, act, P.plain);
  if (P.nlist > 0) {
    auto kg = kp.cross ? k_gal0_list<T, 1> : k_gal0_list<T, 0>;
    hipLaunchKernelGGL(kg, dim3((8 * P.nlist + 255) / 256), dim3(256), 0, F.s, F.mem, kp, coef64(c), L1, act, P.plain,
                       P.list, P.nlist);
  }
  for (size_t l = 1; l < P.levels.size(); ++l) {
    const CLevelT<T> Fl = view<T>(P, (int)l - 1), L = view<T>(P, (int)l);
    hipLaunchKernelGGL(k_galc<T>, dim3(2 * L.ntiles), wg(), 0, F.s, Fl, L, act);
  }
}

// coarse part of the cycle: b(1) is set; x(1) is returned
template <class T>
void coarse_t(hipStream_t s, const imau::MGPlan &P, const int *act) {
  const int nl = (int)P.levels.size();
  for (int l = 0; l < nl; ++l) {
    const CLevelT<T> C = view<T>(P, l);
    fill<T>(s, C.xu, 2 * C.na);
    if (P.levels[l].ends)
      hipLaunchKernelGGL(k_coarsest<T>, dim3(P.ngrids), dim3(P.levels[l].cthreads), 0, s, C, act, P.coarsest_sweeps);
    if (l + 1 == nl) break;
    for (int col = 0; col < 4; ++col) hipLaunchKernelGGL(k_cgs<T>, dim3(C.ntiles), wg(), 0, s, C, col, act);
    const CLevelT<T> N = view<T>(P, l + 1);
    hipLaunchKernelGGL(k_crestrict<T>, dim3(N.ntiles), wg(), 0, s, C, N, act);
  }
  for (int l = nl - 2; l >= 0; --l) {
    const CLevelT<T> C = view<T>(P, l), N = view<T>(P, l + 1);
    hipLaunchKernelGGL(k_cprolong<T>, dim3(C.ntiles), wg(), 0, s, C, N, act);
    for (int col = 3; col >= 0; --col) hipLaunchKernelGGL(k_cgs<T>, dim3(C.ntiles), wg(), 0, s, C, col, act);
  }
}

// coarse part with fused sweeps: pre-smoothing from zero into x, the post-smoothed
// (or coarsest-level) result of every level in the second buffer x2
template <class T>
void coarse_fused_t(hipStream_t s, const imau::MGPlan &P, const int *act) {
  const int nl = (int)P.levels.size();
  for (int l = 0; l < nl; ++l) {
    const CLevelT<T> C = view<T>(P, l), C2 = view2<T>(P, l);
    if (P.levels[l].ends)
      hipLaunchKernelGGL(k_coarsest<T>, dim3(P.ngrids), dim3(P.levels[l].cthreads), 0, s, C2, act,
                         P.coarsest_sweeps);
    if (l + 1 == nl) break;
    hipLaunchKernelGGL(k_cdown<T>, dim3(C.ntiles), dim3(CTH), 0, s, C, view<T>(P, l + 1), act);
  }
  for (int l = nl - 2; l >= 0; --l) {
    const CLevelT<T> C = view<T>(P, l);
    hipLaunchKernelGGL(k_cup<T>, dim3(C.ntiles), dim3(CTH), 0, s, C, view2<T>(P, l + 1), C.bv + C.na,
                       C.bv + 2 * C.na, act);
  }
}

// one launch per colour; the cycle runs in place on z (zeroed by the caller)
template <class T>
void vcycle_t(const imau::Launch &F, const KP &kp, const CoefT<T> &cf, const imau::MGPlan &P, CVecT<T> y, VecT<T> z,
              const int *act, imau::MGMark mark, void *mctx) {
  hipStream_t s = F.s;
  if (mark) mark(mctx, 0);
  for (int col = 0; col < 5; ++col)
    hipLaunchKernelGGL(k_smooth0<T>, dim3(F.ntiles), wg(), 0, s, F.mem, F.tiles, kp, cf, z, y, col, act);
  if (mark) mark(mctx, 1);
  const CLevelT<T> L1 = view<T>(P, 0);
  auto kr = kp.cross ? k_restrict0<T, 1> : k_restrict0<T, 0>;
  hipLaunchKernelGGL(kr, dim3(L1.ntiles), wg(), 0, s, F.mem, kp, cf, y, CVecT<T>{z.u, z.v}, L1, act);
  coarse_t<T>(s, P, act);
  hipLaunchKernelGGL(k_prolong0<T>, dim3(F.ntiles), wg(), 0, s, F.mem, F.tiles, cf.rt_u, cf.rt_v, z, L1, act);
  for (int col = 3; col >= 0; --col)
    hipLaunchKernelGGL(k_smooth0<T>, dim3(F.ntiles), wg(), 0, s, F.mem, F.tiles, kp, cf, z, y, col, act);
  hipLaunchKernelGGL(k_smooth0<T>, dim3(F.ntiles), wg(), 0, s, F.mem, F.tiles, kp, cf, z, y, 4, act);
}

// fused sweeps: pre-smoothing from zero into za, post-smoothing from za into
// z (FP64).  With periodic boundaries, whose rows need a pass of their own on
// the working-precision iterate, the restriction runs on its own and the
// post-smoothed iterate goes through zb; yt is then the right-hand side in
// the working precision (null otherwise).
template <class T, int CROSS>
void vcycle_fused_t(const imau::Launch &F, const KP &kp, const CoefT<T> &cf, const imau::MGPlan &P, CVecT<double> y,
                    CVecT<T> yt, VecT<T> za, VecT<T> zb, VecT<double> z, const int *act, imau::MGMark mark, void *mctx) {
  hipStream_t s = F.s;
  const CLevelT<T> L1 = view<T>(P, 0);
  const CVecT<T> zac{za.u, za.v};
  if (mark) mark(mctx, 0);
  if (!P.periodic) {
    hipLaunchKernelGGL((k_fine_down<T, CROSS, true, double>), dim3(P.nftiles), dim3(FTH), 0, s, F.mem, P.ftiles, kp, cf,
                       y, za, L1, act);
    if (mark) mark(mctx, 1);
    coarse_fused_t<T>(s, P, act);
    hipLaunchKernelGGL((k_fine_up<T, CROSS, double, double>), dim3(P.nftiles), dim3(FTH), 0, s, F.mem, P.ftiles, kp, cf,
                       y, zac, z, view2<T>(P, 0), act);
    return;
  }
  hipLaunchKernelGGL((k_fine_down<T, CROSS, false, double>), dim3(P.nftiles), dim3(FTH), 0, s, F.mem, P.ftiles, kp, cf, y,
                     za, L1, act);
  hipLaunchKernelGGL(k_smooth0<T>, dim3(F.ntiles), wg(), 0, s, F.mem, F.tiles, kp, cf, za, yt, 4, act);
  if (mark) mark(mctx, 1);
  hipLaunchKernelGGL((k_restrict0<T, CROSS>), dim3(L1.ntiles), wg(), 0, s, F.mem, kp, cf, yt, zac, L1, act);
  coarse_fused_t<T>(s, P, act);
  hipLaunchKernelGGL((k_fine_up<T, CROSS, double, T>), dim3(P.nftiles), dim3(FTH), 0, s, F.mem, P.ftiles, kp, cf, y, zac,
                     zb, view2<T>(P, 0), act);
  hipLaunchKernelGGL(k_smooth0<T>, dim3(F.ntiles), wg(), 0, s, F.mem, F.tiles, kp, cf, zb, yt, 4, act);
}

}  // namespace

namespace imau {

void mg_plain_flags(const Launch &F, const uint8_t *rt_u, const uint8_t *rt_v, const MGPlan &P) {
  if (P.levels.empty()) return;
  const CLevelT<float> L1 = view<float>(P, 0);
  fill_i32(F.s, P.nlist_d, 1, 0);
  hipLaunchKernelGGL(k_gal_plain_flags, dim3(L1.ntiles), wg(), 0, F.s, F.mem, rt_u, rt_v, L1, P.plain, P.list,
                     P.nlist_d);
}

void mg_setup(const Launch &F, const KP &kp, const Coef &c, const MGPlan &P, bool fp32, bool galerkin,
              const int *active) {
  if (fp32) {
    hipLaunchKernelGGL(k_coef32, dim3(F.ntiles), wg(), 0, F.s, F.mem, F.tiles, coef64(c), P.f32, kp.cross ? 0 : 1,
                       active);
    if (galerkin) setup_t<float>(F, kp, c, P, active);
  } else if (galerkin) {
    setup_t<double>(F, kp, c, P, active);
  }
}

void mg_vcycle(const Launch &F, const KP &kp, const Coef &c, const MGPlan &P, bool fp32, const double *yu,
               const double *yv, double *zu, double *zv, const int *active, MGMark mark, void *mark_ctx) {
  const CVecT<double> y{yu, yv};
  const VecT<double> z{zu, zv};
  if (fp32) {
    const VecT<float> y32{P.f32.yu, P.f32.yv}, z32{P.f32.zu, P.f32.zv}, z32b{P.f32.zu2, P.f32.zv2};
    const CVecT<float> y32c{y32.u, y32.v};
    const CoefT<float> cf = coef32(P.f32, c);
    const bool own = !P.fused || P.periodic;  // paths on an FP32 right-hand side and result
    if (own)
      hipLaunchKernelGGL(k_prep<float>, dim3(F.ntiles), wg(), 0, F.s, F.mem, F.tiles, y, y32, z32, active);
    if (P.fused) {
      auto run = kp.cross ? vcycle_fused_t<float, 1> : vcycle_fused_t<float, 0>;
      run(F, kp, cf, P, y, y32c, z32, z32b, z, active, mark, mark_ctx);
    } else {
      vcycle_t<float>(F, kp, cf, P, y32c, z32, active, mark, mark_ctx);
    }
    if (own) {
      const VecT<float> r = P.fused ? z32b : z32;
      hipLaunchKernelGGL(k_fin, dim3(F.ntiles), wg(), 0, F.s, F.mem, F.tiles, CVecT<float>{r.u, r.v}, z, active);
    }
  } else if (P.fused) {
    auto run = kp.cross ? vcycle_fused_t<double, 1> : vcycle_fused_t<double, 0>;
    run(F, kp, coef64(c), P, y, y, VecT<double>{P.zu64, P.zv64}, z, z, active, mark, mark_ctx);
  } else {
    hipLaunchKernelGGL(k_prep<double>, dim3(F.ntiles), wg(), 0, F.s, F.mem, F.tiles, y, VecT<double>{nullptr, nullptr}, z,
                       active);
    vcycle_t<double>(F, kp, coef64(c), P, y, z, active, mark, mark_ctx);
  }
}

}  // namespace imau
