// k_push2d.hip -- Buneman-Boris push (2d/common/particle.f90:48-179) and
// Esirkepov charge-conserving deposit (2d/common/field.f90:189-316) on tiles.
//
// One workgroup owns a tile of cells.  It stages the cell-centred fields of
// the tile plus a one-cell halo in LDS (computed from uf as particle.f90:70-83
// does) and, in fast mode, a current accumulator for the tile plus a two-cell
// halo; lane groups walk one cell at a time (particles of a cell are
// contiguous, sorted by cell), see k_push_deposit_fast.
//
// Parity mode: one lane per cell accumulates in the reference's slot order and
// writes its 5x5x3 block to a per-cell buffer; k_gather_pj then adds the
// blocks in the reference's (j, i) cell order, reproducing uj bit for bit.
//
// All arithmetic is written in the reference's evaluation order and the
// library is built with -ffp-contract=off, so the push is bit-identical to
// the reference at any thread count.
#include "k_push2d.h"

namespace wpic {

struct PushArgs {
  Grid2D g;
  Parts A, B;
  const int* rowbase;
  const int* cumcnt;
  const int* ap;  // A's slot -> record (null: identity)
  const double* uf;
  double* uj;
  double* pjbuf;
  int* code;
  int* err;
  int ntx, nty;
  int tw;   // columns of cells a workgroup takes (the fused fast kernel)
  int vay;  // the Vay kick instead of Buneman-Boris (particle__solv_vay)
};

// register layout of one cell's current block:
//   [0,20)  pjx(ip,jp), ip = -1..2, jp = -2..2  -> (jp+2)*4 + ip+1
//   [20,40) pjy(ip,jp), ip = -2..2, jp = -1..2  -> 20 + (jp+1)*5 + ip+2
//   [40,65) pjz(ip,jp)                          -> 40 + (jp+2)*5 + ip+2
// pjx(-2,.) and pjy(.,-2) are identically +0 in the reference and adding +0
// to a never-negative-zero sum is the identity, so they are not carried.
constexpr int NPJ = 65;

// Esirkepov shape arrays of one particle (field.f90:223-268): s0 at the old
// position relative to cell (i, j), ds = (shifted new shape) - s0
__device__ inline void esirkepov_shapes(const Grid2D& g, double x, double y, double nxp, double nyp, int i, int j,
                                        double s0x[5], double s0y[5], double dsx[5], double dsy[5]) {
  double t0, t1, t2;
  shape3(x - 0.5 - i, t0, t1, t2);
  s0x[0] = 0.0; s0x[1] = t0; s0x[2] = t1; s0x[3] = t2; s0x[4] = 0.0;
  shape3(y - 0.5 - j, t0, t1, t2);
  s0y[0] = 0.0; s0y[1] = t0; s0y[2] = t1; s0y[3] = t2; s0y[4] = 0.0;
#pragma unroll
  for (int d = 0; d < 2; d++) {
    const double gp = d == 0 ? nxp : nyp;
    const int cell = d == 0 ? i : j;
    const int i2 = (int)gp;
    const double dh = gp - 0.5 - i2;
    const int inc = i2 - cell;
    const double s1_1 = 0.5 * (0.5 - dh) * (0.5 - dh);
    const double s1_2 = 0.75 - dh * dh;
    const double s1_3 = 0.5 * (0.5 + dh) * (0.5 + dh);
    // smo_1 = -(inc-abs(inc))*0.5+0 etc. (field.f90:244-246): whole numbers,
    // never -0; |inc| = 1 at most except where a reflecting wall moves a
    // particle by more, and then the same formula applies
    const double smo_1 = inc < 0 ? (double)(-inc) : 0.0;
    const double smo_2 = (double)(-abs(inc) + 1);
    const double smo_3 = inc > 0 ? (double)inc : 0.0;
    double* ds = d == 0 ? dsx : dsy;
    const double* s0 = d == 0 ? s0x : s0y;
    ds[0] = s1_1 * smo_1;
    ds[1] = s1_1 * smo_2 + s1_2 * smo_1;
    ds[2] = s1_2 * smo_2 + s1_3 * smo_1 + s1_1 * smo_3;
    ds[3] = s1_3 * smo_2 + s1_2 * smo_3;
    ds[4] = s1_3 * smo_3;
#pragma unroll
    for (int k = 0; k < 5; k++) ds[k] = ds[k] - s0[k];
  }
}

// The shapes of a particle that stays in cell (i, j): inc = 0 makes smo =
// (0, 1, 0), so ds(-2) = ds(2) = 0 and ds(k) = s1(k) - s0(k) for k = -1..1,
// the values esirkepov_shapes gives there (x * 1 and + 0 are exact), with
// three of its ten live at a time
__device__ inline void stayer_shapes(double x, double y, double nxp, double nyp, int i, int j,
                                     double s0x[3], double s0y[3], double dsx[3], double dsy[3]) {
  shape3(x - 0.5 - i, s0x[0], s0x[1], s0x[2]);
  shape3(y - 0.5 - j, s0y[0], s0y[1], s0y[2]);
  double t0, t1, t2;
  shape3(nxp - 0.5 - i, t0, t1, t2);
  dsx[0] = t0 - s0x[0]; dsx[1] = t1 - s0x[1]; dsx[2] = t2 - s0x[2];
  shape3(nyp - 0.5 - j, t0, t1, t2);
  dsy[0] = t0 - s0y[0]; dsy[1] = t1 - s0y[1]; dsy[2] = t2 - s0y[2];
}

// One cell's N accumulators to the cell's block at offset OFF
template <int N, int OFF>
__device__ inline void store_block(double (&v)[N], double* pjbuf, int cellidx) {
  double* dst = pjbuf + (size_t)cellidx * NPJ + OFF;
#pragma unroll
  for (int k = 0; k < N; k++) dst[k] = v[k];
}

// boundary_periodic__particle_x (:74-88, x wrap under round-down, periodic
// only) and particle_y's row test and y wrap (:120-154) for a particle of row
// j; returns the exchange code (new x cell << 2 | row step + 1).
template <int BC>
__device__ inline int wrap_code(const Grid2D& g, double& nxp, double& nyp, int j, int* err) {
  if (BC == WPIC_BC_PERIODIC) {
    const int ipos = cell_of(nxp);
    if (ipos < g.nxgs)
      nxp = rd_add(nxp, g.spanx);
    else if (ipos >= g.nxge + 1)
      nxp = rd_add(nxp, -g.spanx);
  }
  const int jpos = cell_of(nyp);
  if (jpos != j) {
    if (jpos <= g.nygs - 1)
      nyp = rd_add(nyp, g.spany);
    else if (jpos >= g.nyge + 1)
      nyp = rd_add(nyp, -g.spany);
  }
  int ni = (int)nxp, dy = jpos - j;
  if (ni < g.nxgs || ni > g.nxge || dy < -1 || dy > 1) {
    atomicOr(err, ERR_DOMAIN);
    ni = ni < g.nxgs ? g.nxgs : (ni > g.nxge ? g.nxge : ni);
    dy = dy < -1 ? -1 : (dy > 1 ? 1 : dy);
  }
  return ((ni - g.nxgs) << 2) | (dy + 1);
}

// One pass over a cell's particles accumulating the current components
// selected by DZ/DX/DY from the old (A) and new (B) positions, then storing
// them.  With WRAP it also applies boundary_periodic__particle_x/_y's
// round-down wraps (:74-88, :124-154) and writes the exchange code.
template <bool DZ, bool DX, bool DY, bool WRAP, int BC>
__device__ inline void deposit_pass(const PushArgs& a, int i, int j, int cellidx) {
  const Grid2D& g = a.g;
  const double cc2 = g.c * g.c;
  const bool unit_c = cc2 == 1.0;
  const double fac = 1.0 / 3.0;
  double az[DZ ? 25 : 1], ax[DX ? 20 : 1], ay[DY ? 20 : 1];
#pragma unroll
  for (int k = 0; k < (DZ ? 25 : 1); k++) az[k] = 0.0;
#pragma unroll
  for (int k = 0; k < (DX ? 20 : 1); k++) ax[k] = 0.0;
#pragma unroll
  for (int k = 0; k < (DY ? 20 : 1); k++) ay[k] = 0.0;
  for (int s = 0; s < g.nsp; s++) {
    const int rw = s * g.ny + (j - g.nys);
    const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
    const int base = a.rowbase[rw];
    const int pbeg = base + cr[i - g.nxgs], pend = base + cr[i - g.nxgs + 1];
    const double q = g.q[s];
    const double qk = q * g.delx * g.d_delt;
    for (int pi = pbeg; pi < pend; pi++) {
      double nxp = a.B.x[pi], nyp = a.B.y[pi];
      const int ia = a.ap ? a.ap[pi] : pi;
      double s0x[5], s0y[5], dsx[5], dsy[5];
      esirkepov_shapes(g, a.A.x[ia], a.A.y[ia], nxp, nyp, i, j, s0x, s0y, dsx, dsy);
      if (DZ) {
        const double g3 = a.B.ux[pi], g4 = a.B.uy[pi], g5 = a.B.uz[pi];
        const double u2 = +g3 * g3 + g4 * g4 + g5 * g5;
        const double gvz = g5 / sqrt(1. + (unit_c ? u2 : u2 / cc2));
        const double qgvz = q * gvz;
#pragma unroll
        for (int jp = 0; jp < 5; jp++)
#pragma unroll
          for (int ip = 0; ip < 5; ip++)
            az[jp * 5 + ip] = az[jp * 5 + ip] + qgvz * (+s0x[ip] * s0y[jp] + 0.5 * dsx[ip] * s0y[jp] +
                                                         0.5 * s0x[ip] * dsy[jp] + fac * dsx[ip] * dsy[jp]);
      }
      if (DX) {
#pragma unroll
        for (int jp = 0; jp < 5; jp++) {
          const double wy = s0y[jp] + 0.5 * dsy[jp];
          double run = 0.0;
#pragma unroll
          for (int ip = 0; ip < 4; ip++) {
            run = run - qk * dsx[ip] * wy;
            ax[jp * 4 + ip] = ax[jp * 4 + ip] + run;
          }
        }
      }
      if (DY) {
#pragma unroll
        for (int ip = 0; ip < 5; ip++) {
          const double wx = s0x[ip] + 0.5 * dsx[ip];
          double run = 0.0;
#pragma unroll
          for (int jp = 0; jp < 4; jp++) {
            run = run - qk * dsy[jp] * wx;
            ay[jp * 5 + ip] = ay[jp * 5 + ip] + run;
          }
        }
      }
      if (WRAP) {
        const int code = wrap_code<BC>(g, nxp, nyp, j, a.err);
        a.B.x[pi] = nxp;
        a.B.y[pi] = nyp;
        a.code[pi] = code;
      }
    }
  }
  if constexpr (DZ) store_block<25, 40>(az, a.pjbuf, cellidx);
  if constexpr (DX) store_block<20, 0>(ax, a.pjbuf, cellidx);
  if constexpr (DY) store_block<20, 20>(ay, a.pjbuf, cellidx);
}

// Parity mode, one lane per cell in the reference's slot order: the push with
// its walls, wraps and exchange code and the deposit (PUSH: the fused step),
// or the deposit alone.  Passes over a cell's particles keep few values live
// at once: push and reflecting walls, gp stored;  Jz;  Jx;  Jy, then the
// periodic wraps and the exchange code.
template <bool PUSH, int BC>
__global__ __launch_bounds__(NT) void k_push_deposit_parity(PushArgs a) {
  __shared__ FieldPair sf[PUSH ? 3 : 1][SFW * SFH];
  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * TX;
  const int j0 = g.nys + (tile / a.ntx) * TY;
  if constexpr (PUSH) {
    stage_fields(g, a.uf, sf, i0, j0);
    __syncthreads();
  }
  const double delt = g.delt, c = g.c;
  const bool unit_c = c * c == 1.0;  // x/(c*c) == x exactly: skip the division
  for (int cc = threadIdx.x; cc < TX * TY; cc += NT) {
    const int li = cc % TX, lj = cc / TX;
    const int i = i0 + li, j = j0 + lj;
    if (i > g.nxge || j > g.nye) continue;
    const int cellidx = cidx(g, i, j);
    if constexpr (PUSH) {
      for (int s = 0; s < g.nsp; s++) {
        const int rw = s * g.ny + (j - g.nys);
        const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
        const int base = a.rowbase[rw];
        const int pbeg = base + cr[i - g.nxgs], pend = base + cr[i - g.nxgs + 1];
        const double q = g.q[s], rm = g.r[s];
        const double fac1 = q / rm * 0.5 * delt;
        const double txxx = fac1 * fac1;
        const double fac2 = q * delt / rm;
        for (int pi = pbeg; pi < pend; pi++) {
          const Rec p = load_rec(a.A, a.ap ? a.ap[pi] : pi);
          double nxp, nyp, g3, g4, g5, gmv;
          if (a.vay)
            vay_push(sf, li, lj, i, j, delt, c, fac1, fac2, p.x, p.y, p.ux, p.uy, p.uz, nxp, nyp, g3, g4, g5, gmv);
          else
            boris_push(sf, li, lj, i, j, delt, c, unit_c, fac1, txxx, fac2, p.x, p.y, p.ux, p.uy, p.uz, nxp, nyp, g3,
                       g4, g5, gmv);
          // reflecting walls act before the deposit in the reconnection order
          // (2d/proj/reconnection/app.f90:101-103; boundary_reconnection.f90:79-91)
          reflect_x<BC>(g, nxp, g3, g4, g5);
          store_rec(a.B, pi, Rec{nxp, nyp, g3, g4, g5, p.id});  // particle.f90:173-177
        }
      }
    }
    // Jz (field.f90:292-298), Jx (:274-281), Jy (:283-290)
    deposit_pass<true, false, false, false, BC>(a, i, j, cellidx);
    deposit_pass<false, true, false, false, BC>(a, i, j, cellidx);
    deposit_pass<false, false, true, PUSH, BC>(a, i, j, cellidx);
  }
}

// Current of one particle as the full 5x5 Esirkepov block in the factored
// form below, added to the LDS tile at cell (li, lj) with atomics (zeros
// skipped): the path of a particle that changes cell.
__device__ inline void deposit2_full(double (*acc)[ACW * ACH], int li, int lj, const double s0x[5], const double s0y[5],
                                     const double dsx[5], const double dsy[5], double qk, double qvz) {
  double cx = 0.0, cy = 0.0;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    cx -= dsx[m];
    cy -= dsy[m];
#pragma unroll
    for (int n = 0; n < 5; n++) {
      const double vx = cx * (qk * fma(0.5, dsy[n], s0y[n]));  // x face m - 1, y node n - 2
      const double vy = cy * (qk * fma(0.5, dsx[n], s0x[n]));  // x node n - 2, y face m - 1
      if (vx != 0.0) atomicAdd(&acc[0][(lj + n) * ACW + (li + 1 + m)], vx);
      if (vy != 0.0) atomicAdd(&acc[1][(lj + 1 + m) * ACW + (li + n)], vy);
    }
  }
#pragma unroll
  for (int jp = 0; jp < 5; jp++) {
    const double A = qvz * fma(0.5, dsy[jp], s0y[jp]), B = qvz * fma(1.0 / 3.0, dsy[jp], 0.5 * s0y[jp]);
#pragma unroll
    for (int ip = 0; ip < 5; ip++) {
      double v = dsx[ip] * B;
      if (ip >= 1 && ip <= 3) v = fma(s0x[ip], A, v);
      if (v != 0.0) atomicAdd(&acc[2][(lj + jp) * ACW + (li + ip)], v);
    }
  }
}

// The same current on the 4-node window [lo, lo + 3] of the 5 nodes -2..2 per
// axis, lo = 0 for a step to the left and 1 otherwise, which holds every
// non-zero s0 and ds: 12 + 12 + 16 values instead of 65.  The new shape at its
// nodes carries the reference's weights (field.f90:244-266), |inc| moved by one
// node and 1 - |inc| unmoved: a plain shift for a step of one cell (where the
// products are exact), and what the reference does where a particle near c
// rounds across two faces (c delt = delx allows that in x).
__device__ inline void shapes_window(double old, double nw, int cell, double S0[4], double DS[4], int& lo) {
  double t0, t1, t2, u0, u1, u2;
  shape3(old - 0.5 - cell, t0, t1, t2);
  const int c2 = (int)nw, inc = c2 - cell;
  shape3(nw - 0.5 - c2, u0, u1, u2);
  const bool left = inc < 0;
  lo = left ? 0 : 1;
  const double far = (double)abs(inc), near = 1.0 - far;
  const double p = left ? far : near, q = left ? near : far;
  // old shape on window nodes 1..3 (left) or 0..2; of the new one p on 0..2 and
  // q on 1..3
  S0[0] = left ? 0.0 : t0;
  S0[1] = left ? t0 : t1;
  S0[2] = left ? t1 : t2;
  S0[3] = left ? t2 : 0.0;
  DS[0] = p * u0 - S0[0];
  DS[1] = p * u1 + q * u0 - S0[1];
  DS[2] = p * u2 + q * u1 - S0[2];
  DS[3] = q * u2 - S0[3];
}

__device__ inline void deposit2_window(double (*acc)[ACW * ACH], int li, int lj, int i, int j, double x, double y,
                                       double nxp, double nyp, double qk, double qvz) {
  double S0x[4], DSx[4], S0y[4], DSy[4];
  int lox, loy;
  shapes_window(x, nxp, i, S0x, DSx, lox);
  shapes_window(y, nyp, j, S0y, DSy, loy);
  const bool mx = (int)nxp != i, my = (int)nyp != j;
  double* const o = &acc[0][(lj + loy) * ACW + (li + lox)];  // window node (0, 0)
  // row by row (the barriers keep the compiler from forming all the products
  // first, which costs the caller's registers): Jx and Jz of node row n, then
  // Jy of face row m.  The fourth node of an axis along which the particle
  // keeps its cell carries nothing, and that axis' third face only rounding.
  const double cx0 = 0.0 - DSx[0], cx1 = cx0 - DSx[1], cx2 = cx1 - DSx[2];
#pragma unroll
  for (int n = 0; n < 4; n++) {
    if (n == 3 && !my) break;
    const double ay = fma(0.5, DSy[n], S0y[n]);
    const double wy = qk * ay, A = qvz * ay, B = qvz * fma(1.0 / 3.0, DSy[n], 0.5 * S0y[n]);
    double* const r = o + n * ACW;
    double* const z = r + 2 * ACW * ACH;
    atomicAdd(r + 1, cx0 * wy);
    atomicAdd(r + 2, cx1 * wy);
    atomicAdd(z, fma(S0x[0], A, DSx[0] * B));
    atomicAdd(z + 1, fma(S0x[1], A, DSx[1] * B));
    atomicAdd(z + 2, fma(S0x[2], A, DSx[2] * B));
    if (mx) {
      atomicAdd(r + 3, cx2 * wy);
      atomicAdd(z + 3, fma(S0x[3], A, DSx[3] * B));
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  double wx[4];
#pragma unroll
  for (int n = 0; n < 4; n++) wx[n] = qk * fma(0.5, DSx[n], S0x[n]);
  double cy = 0.0;
#pragma unroll
  for (int m = 0; m < 3; m++) {
    if (m == 2 && !my) break;
    cy -= DSy[m];
    double* const r = o + ACW * ACH + (m + 1) * ACW;
    atomicAdd(r, cy * wx[0]);
    atomicAdd(r + 1, cy * wx[1]);
    atomicAdd(r + 2, cy * wx[2]);
    if (mx) atomicAdd(r + 3, cy * wx[3]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Push of one particle of cell (i, j) and, with reflecting walls, the
// reflection that precedes the deposit in the reconnection order
// (2d/proj/reconnection/app.f90:101-103; boundary_reconnection.f90:79-91).
template <int BC, bool VAY>
__device__ inline void push_reflect(const Grid2D& g, const FieldPair (*sf)[SFW * SFH], int li, int lj, int i, int j,
                                    bool unit_c, const double* kc, double x, double y, double ux, double uy, double uz,
                                    double& nxp, double& nyp, double& g3, double& g4, double& g5, double& gmv) {
  if (VAY)
    vay_push(sf, li, lj, i, j, g.delt, g.c, kc[0], kc[2], x, y, ux, uy, uz, nxp, nyp, g3, g4, g5, gmv);
  else
    boris_push(sf, li, lj, i, j, g.delt, g.c, unit_c, kc[0], kc[1], kc[2], x, y, ux, uy, uz, nxp, nyp, g3,
               g4, g5, gmv);
  reflect_x<BC>(g, nxp, g3, g4, g5);
  // the injection edge sends ux to 2 u0 - ux, which changes gamma: vz of the
  // deposit comes from the momenta after the boundary (field.f90:270-272)
  if (BC == WPIC_BC_SHOCK) {
    const double u2 = +g3 * g3 + g4 * g4 + g5 * g5;
    gmv = 1.0 / sqrt(1.0 + (unit_c ? u2 : u2 / (g.c * g.c)));
  }
}

// The fast kernel, in one pass over each particle: push, deposit, wraps and
// exchange code (FUSED, the step), the push alone (PUSH: particle__solv, in
// every mode) or the deposit alone from the old and new positions (DEPOSIT:
// field__fdtd_i in fast mode).  The push is the shared bit-exact boris_push; the current is the same Esirkepov weights in a
// factored form that reorders the reference's sums (so uj agrees to rounding,
// not bit for bit):
//   Jx(ip, jp) += cx(ip) * wy(jp),  cx(m) = -sum_{k<=m} dsx(k),  wy = qk (s0y + ds_y/2)
//   Jy(ip, jp) += cy(jp) * wx(ip),  likewise with x and y exchanged
//   Jz(ip, jp) += s0x(ip) * A(jp) + dsx(ip) * B(jp),
//                 A = q vz (s0y + dsy/2),  B = q vz (s0y/2 + dsy/3)
// which expands to field.f90:274-298 term by term.  A particle that stays in
// its cell has ds = 0 on the outer nodes and cx = 0 on the outer faces (the
// last up to rounding), so its current lives on 6 + 6 + 9 nodes: each lane
// accumulates those 21 values in registers over the particles of the cell it
// handles and the group reduces them once per cell.  A particle that changes
// cell (about one in eight here) is queued in its wave's LDS queue with what
// its current needs (old and unwrapped new position, q vz); whenever 64 have
// gathered, over as many passes and cells as that takes, all the wave's lanes
// add one particle's window each (deposit2_window; with walls, which may
// reflect by more than one cell, the full block, deposit2_full).  The queues
// are per wave, so no barrier stops the workgroup between the staging and the
// final flush.
//
// Work mapping: wave w walks row w of the tile of a.tw x 4 cells, 64 / G
// x-adjacent cells per round (one per G-lane group), so a cell's x-neighbours
// share its wave and its y-neighbours run in the sibling waves at about the
// same time: the records of particles that crossed a cell or row boundary are
// read while the lines they share with their old neighbours are still in L2.
// Each lane walks its cell's particles (all species as one list) with a
// two-deep software pipeline: the permutation entry of element t + 2G and the
// record of element t + G are in flight while element t is pushed.  The push
// alone keeps the unwrapped positions, as particle__solv leaves them.
//
// What bounds it (1024x1024, 64 ppc): 16.1 GB of traffic (14.0 algorithmic:
// the record each way, its permutation entry and exchange code) in 4.15 ms,
// 3.9 TB/s where a plain copy reaches 4.8, at 2 waves a SIMD (254 registers)
// with VALU issue in 57 % of the cycles.  With one array per field it moved 22
// GB in 5.3 ms: 48-byte records, 16-byte loads and stores took 0.5 ms off, the
// full drains and windows 0.25, the shared root and halving reduction 0.2, the
// straight-line pass 0.15.
constexpr int QW = 128;  // queued cell-changing particles per wave: 63 left over and 64 of a pass at most
enum { FUSED, PUSH, DEPOSIT };
template <int G, int WHAT, int BC, bool VAY>
__global__ __launch_bounds__(NT, 2) void k_push_deposit_fast(PushArgs a) {
  constexpr bool PUSHES = WHAT != DEPOSIT, DEPOSITS = WHAT != PUSH;
  constexpr int NW = NT / 64;
  static_assert(NW == TY && 8 % (64 / G) == 0, "one wave per tile row, whole rounds of any tile width");
  __shared__ FieldPair sf[PUSHES ? 3 : 1][SFW * SFH];
  __shared__ double acc[3][ACW * ACH];
  __shared__ double spc[WPIC_MAXSP][5];  // fac1, txxx, fac2, qk, q
  __shared__ double xqd[NW][5][QW];      // x, y, unwrapped new x, y, q vz
  __shared__ int xqc[NW][QW];            // cell in the tile | species << 8

  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * a.tw;
  const int j0 = g.nys + (tile / a.ntx) * TY;
  const int tid = threadIdx.x;

  if constexpr (PUSHES) stage_fields(g, a.uf, sf, i0, j0, a.tw);
  if constexpr (DEPOSITS)
    for (int k = tid; k < 3 * ACW * ACH; k += NT) (&acc[0][0])[k] = 0.0;
  // per-species constants (particle.f90:92-94, field.f90:274)
#pragma unroll
  for (int s = 0; s < WPIC_MAXSP; s++) {
    if (tid == s && s < g.nsp) {
      const double q = g.q[s], rm = g.r[s];
      const double fac1 = q / rm * 0.5 * g.delt;
      spc[s][0] = fac1;
      spc[s][1] = fac1 * fac1;
      spc[s][2] = q * g.delt / rm;
      spc[s][3] = q * g.delx * g.d_delt;
      spc[s][4] = q;
    }
  }
  __syncthreads();

  constexpr int RX = 64 / G;  // cells per wave round
  const int w = tid >> 6, lane = tid & 63;
  const int lg = lane % G;
  const int lj = w, j = j0 + lj;
  const bool unit_c = g.c * g.c == 1.0;
  int nq = 0;  // queued particles, the same in all lanes

  // where this lane's sums of a cell's stayers go: the index in acc of cell
  // (0, lj)'s node
  constexpr int NRES = group_left(21, G);
  int node[NRES];
#pragma unroll
  for (int f = 0; f < NRES; f++) {
    const int q = group_index<21, G>(f, lane);
    const int m = q < 12 ? q % 6 / 3 : (q - 12) / 3, u = q % 3 - 1;
    const int xo = q < 6 ? m : u, yo = q < 6 ? u : (q < 12 ? m : m - 1);
    const int comp = q < 6 ? 0 : (q < 12 ? 1 : 2);
    node[f] = q < 0 ? -1 : comp * (ACW * ACH) + (lj + 2 + yo) * ACW + 2 + xo;
  }

  // the currents of the last (at most 64) queued particles
  auto drain = [&]() {
    // written by this wave's own lanes: LDS operations of one wave complete in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int n0 = nq > 64 ? nq - 64 : 0, q = n0 + lane;
    if (q < nq) {
      const int e = xqc[w][q];
      const int qli = (e & 255) % TX, qlj = (e & 255) / TX, s = e >> 8;
      const double x = xqd[w][0][q], y = xqd[w][1][q], nxp = xqd[w][2][q], nyp = xqd[w][3][q], qvz = xqd[w][4][q];
      // (gp's own boundaries may have acted on it before a separate deposit)
      if (WHAT == FUSED && BC == WPIC_BC_PERIODIC) {
        deposit2_window(acc, qli, qlj, i0 + qli, j0 + qlj, x, y, nxp, nyp, spc[s][3], qvz);
      } else {
        double s0x[5], s0y[5], dsx[5], dsy[5];
        esirkepov_shapes(g, x, y, nxp, nyp, i0 + qli, j0 + qlj, s0x, s0y, dsx, dsy);
        deposit2_full(acc, qli, qlj, s0x, s0y, dsx, dsy, spc[s][3], qvz);
      }
    }
    nq = n0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  for (int l0 = 0; l0 < a.tw; l0 += RX) {
    const int li = l0 + lane / G;
    const int i = i0 + li;
    const bool live = i <= g.nxge && j <= g.nye;  // uniform within a group
    // stayers: sx[m][u] Jx at x face m, y node u - 1; sy[m][u] Jy at y face
    // m, x node u - 1; sz[v][u] Jz at x node u - 1, y node v - 1
    double sx[2][3], sy[2][3], sz[3][3];
#pragma unroll
    for (int u = 0; u < 3; u++) {
      sx[0][u] = sx[1][u] = sy[0][u] = sy[1][u] = 0.0;
      sz[0][u] = sz[1][u] = sz[2][u] = 0.0;
    }

    // the cell's particles over all species as one list
    CellList cl;
    int tot = 0;
#pragma unroll
    for (int s = 0; s < WPIC_MAXSP; s++) {
      if (s < g.nsp) {
        int c0 = 0, c1 = 0, rb = 0;
        if (live) {
          const int rw = s * g.ny + (j - g.nys);
          const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1) + (i - g.nxgs);
          c0 = cr[0];
          c1 = cr[1];
          rb = a.rowbase[rw];
        }
        cl.set(s, rb + c0, tot);
        tot += c1 - c0;
      } else {
        cl.set(s, 0, 0x7fffffff);
      }
    }
    int ia_nn = 0;
    // (a cell's surplus lanes push a particle at rest at its centre)
    Rec pr = {i + 0.5, j + 0.5, 0.0, 0.0, 0.0, 0};
    {
      int s_, p_;
      int ia_n = 0;
      if (lg < tot) {
        cl.slot(g.nsp, lg, s_, p_);
        ia_n = a.ap ? a.ap[p_] : p_;
      }
      if (lg + G < tot) {
        cl.slot(g.nsp, lg + G, s_, p_);
        ia_nn = a.ap ? a.ap[p_] : p_;
      }
      if (lg < tot) {
        pr = load_rec(a.A, ia_n);
      }
    }
    // Every lane of the wave runs the passes of the wave's fullest cell, so
    // that the queue's length is one number for the wave, and the body is one
    // straight line: a lane past its cell's last particle repeats that one with
    // zero charge and stores nothing.  (With the body inside a branch the
    // compiler copied the 21 sums and the gather's values at every join: 75
    // 64-bit moves of the pass's 600 instructions.)
    for (int t = lg; __any(t < tot); t += G) {
      const bool act = t < tot;
      int s, pi;
      cl.slot(g.nsp, t, s, pi);
      const Rec cur = pr;
      if (t + G < tot) pr = load_rec(a.A, ia_nn);
      if (t + 2 * G < tot) {
        int s_, p_;
        cl.slot(g.nsp, t + 2 * G, s_, p_);
        ia_nn = a.ap ? a.ap[p_] : p_;
      }
      const double* kc = spc[s];
      const double x = cur.x, y = cur.y;
      double nxp, nyp, g3, g4, g5, gmv;
      if constexpr (PUSHES) {
        push_reflect<WHAT == FUSED ? BC : WPIC_BC_PERIODIC, VAY>(g, sf, li, lj, i, j, unit_c, kc, x, y, cur.ux, cur.uy,
                                                                 cur.uz, nxp, nyp, g3, g4, g5, gmv);
      } else {
        Rec gp = {x, y, 0.0, 0.0, 0.0, 0};
        if (act) gp = load_rec(a.B, pi);
        nxp = gp.x, nyp = gp.y, g3 = gp.ux, g4 = gp.uy, g5 = gp.uz;
        const double u2 = +g3 * g3 + g4 * g4 + g5 * g5;
        gmv = 1.0 / sqrt(1.0 + (unit_c ? u2 : u2 / (g.c * g.c)));
      }
      if constexpr (WHAT == PUSH) {
        if (act) store_rec(a.B, pi, Rec{nxp, nyp, g3, g4, g5, cur.id});  // the id travels along (particle.f90:173-177)
      } else {
      const double qvz = kc[4] * (g5 * gmv);
      const int i2 = cell_of(nxp), j2 = cell_of(nyp);
      const bool stays = i2 == i && j2 == j;
      const bool mover = act && !stays;
      if (WHAT == FUSED && act) {
        // the exchange code, and the wraps of the few that leave the box
        double wxp = nxp, wyp = nyp;
        int code = ((i2 - g.nxgs) << 2) | (j2 - j + 1);
        if ((unsigned)(i2 - g.nxgs) >= (unsigned)g.nx || (unsigned)(j2 - g.nys) >= (unsigned)g.ny ||
            (unsigned)(j2 - j + 1) > 2u)
          code = wrap_code<BC>(g, wxp, wyp, j, a.err);
        a.code[pi] = code;
        store_rec(a.B, pi, Rec{wxp, wyp, g3, g4, g5, cur.id});
      }
      {
        const double qk = act && stays ? kc[3] : 0.0, qz = act && stays ? qvz : 0.0;
        double s0x[3], s0y[3], dsx[3], dsy[3];
        stayer_shapes(x, y, nxp, nyp, i, j, s0x, s0y, dsx, dsy);
        const double cx1 = 0.0 - dsx[0], cx2 = cx1 - dsx[1];
        const double cy1 = 0.0 - dsy[0], cy2 = cy1 - dsy[1];
#pragma unroll
        for (int u = 0; u < 3; u++) {
          const double ay = fma(0.5, dsy[u], s0y[u]);
          const double wy = qk * ay, wx = qk * fma(0.5, dsx[u], s0x[u]);
          sx[0][u] = fma(cx1, wy, sx[0][u]);
          sx[1][u] = fma(cx2, wy, sx[1][u]);
          sy[0][u] = fma(cy1, wx, sy[0][u]);
          sy[1][u] = fma(cy2, wx, sy[1][u]);
          const double A = qz * ay, B = qz * fma(1.0 / 3.0, dsy[u], 0.5 * s0y[u]);
#pragma unroll
          for (int k = 0; k < 3; k++) sz[u][k] = fma(s0x[k], A, fma(dsx[k], B, sz[u][k]));
        }
      }
      const uint64_t mm = __ballot(mover);
      if (mm) {
        if (mover) {
          const int slot = nq + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mm >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mm, 0));
          xqd[w][0][slot] = x;
          xqd[w][1][slot] = y;
          xqd[w][2][slot] = nxp;
          xqd[w][3][slot] = nyp;
          xqd[w][4][slot] = qvz;
          xqc[w][slot] = (lj * TX + li) | (s << 8);
        }
        nq += __popcll(mm);
        if (nq >= 64) drain();
      }
      }
    }
    if constexpr (DEPOSITS) {
    // the stayers' 21 sums over the group, spread over its lanes (a cell without
    // particles adds nothing: its fields may be any, and 0 * NaN is not 0)
    double v[21];
#pragma unroll
    for (int u = 0; u < 3; u++) {
      v[u] = sx[0][u];
      v[3 + u] = sx[1][u];
      v[6 + u] = sy[0][u];
      v[9 + u] = sy[1][u];
      v[12 + u] = sz[0][u];
      v[15 + u] = sz[1][u];
      v[18 + u] = sz[2][u];
    }
    group_reduce<21, G>(v, lane);
#pragma unroll
    for (int f = 0; f < NRES; f++)
      if (tot > 0 && node[f] >= 0 && v[f] != 0.0) atomicAdd(&acc[0][0] + (node[f] + li), v[f]);
    }
  }
  if constexpr (DEPOSITS) {
  if (nq) drain();

  __syncthreads();
  const size_t pl = (size_t)g.fw * g.fh;
  const int aw = a.tw + 4, an = aw * ACH;
  for (int k = tid; k < 3 * an; k += NT) {
    const int comp = k / an, rem = k - comp * an;
    const int r = rem / aw, q = rem - r * aw;
    const double v = acc[comp][r * ACW + q];
    if (v == 0.0) continue;
    const int I = i0 - 2 + q, J = j0 - 2 + r;
    if (I > g.nxge + 2 || J > g.nye + 2) continue;
    unsafeAtomicAdd(a.uj + pl * comp + fidx(g, I, J), v);
  }
  }
}

// uj(c, I, J) = sum over source cells in the reference's (j, i) loop order of
// their block entry (field.f90:212-310 at one thread), starting from +0.
__global__ __launch_bounds__(256) void k_gather_pj(Grid2D g, const double* __restrict__ pjbuf,
                                                  double* __restrict__ uj) {
  const int n = g.fw * g.fh;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int I = g.nxgs - 2 + k % g.fw, J = g.nys - 2 + k / g.fw;
  const size_t pl = (size_t)g.fw * g.fh;
  double sx = 0.0, sy = 0.0, sz = 0.0;
  const int jlo = J - 2 > g.nys ? J - 2 : g.nys, jhi = J + 2 < g.nye ? J + 2 : g.nye;
  const int ilo = I - 2 > g.nxgs ? I - 2 : g.nxgs, ihi = I + 2 < g.nxge ? I + 2 : g.nxge;
  for (int j = jlo; j <= jhi; j++)
    for (int i = ilo; i <= ihi; i++) {
      const int ip = I - i, jp = J - j;
      const double* b = pjbuf + (size_t)cidx(g, i, j) * NPJ;
      if (ip >= -1) sx = sx + b[(jp + 2) * 4 + ip + 1];
      if (jp >= -1) sy = sy + b[20 + (jp + 1) * 5 + ip + 2];
      sz = sz + b[40 + (jp + 2) * 5 + ip + 2];
    }
  const int f = fidx(g, I, J);
  uj[f] = sx;
  uj[pl + f] = sy;
  uj[2 * pl + f] = sz;
}

template <int G>
static void launch_fast(wpic_ctx* c, const PushArgs& a, int nb, bool push, bool deposit) {
  const bool vay = a.vay;
#define L(WHAT, BC, V) hipLaunchKernelGGL((k_push_deposit_fast<G, WHAT, BC, V>), dim3(nb), dim3(NT), 0, c->st, a)
#define LV(WHAT, BC)      \
  {                       \
    if (vay)              \
      L(WHAT, BC, true);  \
    else                  \
      L(WHAT, BC, false); \
  }
  if (!push)
    L(DEPOSIT, WPIC_BC_PERIODIC, false);
  else if (!deposit)
    LV(PUSH, WPIC_BC_PERIODIC)
  else if (c->g.bc == WPIC_BC_SHOCK)
    LV(FUSED, WPIC_BC_SHOCK)
  else if (c->g.bc == WPIC_BC_WALLX)
    LV(FUSED, WPIC_BC_WALLX)
  else
    LV(FUSED, WPIC_BC_PERIODIC)
#undef LV
#undef L
}

template <int BC>
static void launch_parity(wpic_ctx* c, const PushArgs& a, int nb, bool push) {
  if (push)
    hipLaunchKernelGGL((k_push_deposit_parity<true, BC>), dim3(nb), dim3(NT), 0, c->st, a);
  else
    hipLaunchKernelGGL((k_push_deposit_parity<false, BC>), dim3(nb), dim3(NT), 0, c->st, a);
}

// push and deposit: the fused step; otherwise one of the two alone
hipError_t launch_push_deposit(wpic_ctx* c, bool push, bool deposit) {
  PushArgs a;
  a.g = c->g;
  a.A = c->A;
  a.B = c->B;
  a.rowbase = c->rowbaseA;
  a.cumcnt = c->cumcnt;
  a.ap = c->aperm;
  a.uf = c->uf;
  a.uj = c->uj;
  a.pjbuf = c->pjbuf;
  a.code = c->code;
  a.err = c->err;
  a.nty = (c->g.ny + TY - 1) / TY;
  a.vay = c->pusher == WPIC_PUSHER_VAY;
  if (c->mode == WPIC_MODE_PARITY && deposit) {
    a.tw = TX;
    a.ntx = (c->g.nx + TX - 1) / TX;
    const int nb = xcd_grid(a.ntx * a.nty);
    if (c->g.bc == WPIC_BC_SHOCK)
      launch_parity<WPIC_BC_SHOCK>(c, a, nb, push);
    else if (c->g.bc == WPIC_BC_WALLX)
      launch_parity<WPIC_BC_WALLX>(c, a, nb, push);
    else
      launch_parity<WPIC_BC_PERIODIC>(c, a, nb, push);
    return hipGetLastError();
  }
  // 16 lanes a cell for well filled cells, 8 for the others: fewer idle lanes
  // and fewer cells reduced one after another.  Push+deposit with 16 and 8
  // lanes: 4.28 and 4.44 ms at 128 particles a cell (1024x1024); 125 and 114
  // us at 48 (250x187); 1.86 and 1.58 ms at 12 (Harris, 1024x2048).
  a.tw = tile_width(c->g);
  a.ntx = (c->g.nx + a.tw - 1) / a.tw;
  const int nb = xcd_grid(a.ntx * a.nty);
  if (c->npart >= 96ll * c->g.nx * c->g.ny)
    launch_fast<16>(c, a, nb, push, deposit);
  else
    launch_fast<8>(c, a, nb, push, deposit);
  return hipGetLastError();
}

hipError_t launch_gather_pj(wpic_ctx* c) {
  const int n = c->g.fw * c->g.fh;
  hipLaunchKernelGGL(k_gather_pj, dim3((n + 255) / 256), dim3(256), 0, c->st, c->g, c->pjbuf, c->uj);
  return hipGetLastError();
}

}  // namespace wpic
