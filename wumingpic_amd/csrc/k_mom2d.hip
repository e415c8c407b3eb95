// k_mom2d.hip -- velocity moments of the 2D particles (2d/common/mom_calc.f90)
// and their boundary folds (boundary_periodic.f90:571-636,
// 2d/proj/reconnection/boundary_reconnection.f90:582-650).
//
// mom(7, nxgs-1:nxge+1, nys-1:nye+1, nsp) is kept in the reference's own
// layout (the seven moments of a node contiguous), so transfers are plain
// copies.  Three deposits:
//   k_mom_tile<KICK>  fast: one workgroup per tile of cells sums a cell's
//                     particles in registers, the tile's nodes (one-node
//                     halo) in LDS, and adds those to HBM once per node and
//                     species; with KICK it applies
//                     mom_calc__accl's half-step kick on the fly (the fused
//                     accl + nvt of the app's output sequence) and never
//                     writes gp;
//   k_mom_any         fast, for a gp in any slot order: HBM atomics;
//   k_mom_parity      one thread per node sums its particles in the
//                     reference's (j, ii) order: bit-identical to
//                     mom_calc__nvt at one thread.
#include "k_push2d.h"

namespace wpic {

struct MomArgs {
  Grid2D g;
  Parts A, B;  // A: up (sorted, read through ap), B: gp
  const int *rowbaseA, *np2A, *rowbaseB, *np2B;
  const int* cumcnt;
  const int* ap;
  const double* uf;
  double* mom;
  int* err;
  int ntx, nty;
  double fac1[WPIC_MAXSP], txxx[WPIC_MAXSP], fac2[WPIC_MAXSP];  // mom_calc.f90:90-92 with delt/2
};

// the seven moments of one particle times the CIC weight wx*wy, in the
// reference's product order (mom_calc.f90:203-243)
struct MomTerms {
  double u[3], gam;
  __device__ void set(double ux, double uy, double uz, double c) {
    u[0] = ux;
    u[1] = uy;
    u[2] = uz;
    gam = 1. / sqrt(1.0 + (+ux * ux + uy * uy + uz * uz) / (c * c));
  }
  __device__ double term(int k, double wx, double wy) const {
    if (k == 0) return wx * wy;
    if (k < 4) return u[k - 1] * gam * wx * wy;
    return u[k - 4] * u[k - 4] * gam * wx * wy;
  }
};

// ---------------------------------------------------------------------------
// mom_calc__accl: gp(1:2) = up(1:2), gp(3:5) = up(3:5) kicked over delt/2
// (mom_calc.f90:131-155); gp is slot-aligned with up, the id travels along.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(NT) void k_mom_accl(MomArgs a) {
  __shared__ FieldTile sf;
  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * TX;
  const int j0 = g.nys + (tile / a.ntx) * TY;
  stage_fields(g, a.uf, sf, i0, j0);
  __syncthreads();
  constexpr int G = 16, NGRP = NT / G;
  const int grp = threadIdx.x / G, lg = threadIdx.x % G;
  const double hdelt = g.delt * 0.5;
  for (int cc = grp; cc < TX * TY; cc += NGRP) {
    const int li = cc % TX, lj = cc / TX;
    const int i = i0 + li, j = j0 + lj;
    if (i > g.nxge || j > g.nye) continue;
    for (int s = 0; s < g.nsp; s++) {
      const int rw = s * g.ny + (j - g.nys);
      const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
      const int base = a.rowbaseA[rw];
      const int pend = base + cr[i - g.nxgs + 1];
      for (int pi = base + cr[i - g.nxgs] + lg; pi < pend; pi += G) {
        const int ia = a.ap ? a.ap[pi] : pi;
        const Rec p = load_rec(a.A, ia);
        double nxp, nyp, g3, g4, g5, gmv;
        boris_push(sf, li, lj, i, j, hdelt, g.c, true, a.fac1[s], a.txxx[s], a.fac2[s], p.x, p.y, p.ux, p.uy, p.uz,
                   nxp, nyp, g3, g4, g5, gmv);
        store_rec(a.B, pi, Rec{p.x, p.y, g3, g4, g5, p.id});
      }
    }
  }
}

// ---------------------------------------------------------------------------
// fast deposit over tiles: particles of the tile (A kicked on the fly, or B
// in A's rows) into an LDS node tile, then one HBM atomic per node.  The node
// tile covers i0-1 .. i0+TX and j0-1 .. j0+TY: a particle of cell i has its
// lower node int(x/dx - 1/2) in {i-1, i}.  A gp particle that is not in the
// cell its slot belongs to (gp not sorted by cell) is added to HBM directly.
// ---------------------------------------------------------------------------
constexpr int MTW = TX + 2, MTH = TY + 2;
// A particle of cell (i, j) adds to two of the nodes i-1, i, i+1 per axis, so a
// cell's particles meet on 9 nodes: every lane sums those 9 x 7 values for the
// particles it handles, the 8 lanes of the cell add up by halving exchanges
// and each adds 8 of the 63 sums to the LDS tile.  Up to KP passes kick their
// particles and leave dx, dy and the moments in registers, then the sums are
// formed from those (next to the gather's reads in flight they would not fit).
// A gp particle that left its cell is added to the tile by itself, or to HBM
// when its node lies off it.
//
// What bounds it (1024x1024, 2 species of 64 ppc, with the kick): VALU issue,
// half of it the kick, in 3.4 ms; the reads alone take 1.5.  28 LDS atomics a
// particle, on planes rotated by the lane, took 3.8.
template <bool KICK>
__global__ __launch_bounds__(NT, 2) void k_mom_tile(MomArgs a) {
  constexpr int G = 8, KP = 4, RX = 64 / G;
  static_assert(NT / 64 == TY, "one wave per tile row");
  __shared__ FieldPair sf[KICK ? 3 : 1][SFW * SFH];
  __shared__ double mt[7][MTW * MTH];
  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * TX;
  const int j0 = g.nys + (tile / a.ntx) * TY;
  const int ncx = min(TX, g.nxge + 1 - i0);
  const int tid = threadIdx.x;
  if constexpr (KICK) stage_fields(g, a.uf, sf, i0, j0);
  const double hdelt = g.delt * 0.5, c = g.c;
  const bool unit_c = c * c == 1.0;
  const int lane = tid & 63, lg = lane % G;
  const int lj = __builtin_amdgcn_readfirstlane(tid >> 6), j = j0 + lj;

  for (int s = 0; s < g.nsp; s++) {
    for (int k = tid; k < 7 * MTW * MTH; k += NT) (&mt[0][0])[k] = 0.0;
    __syncthreads();
    const int rw = s * g.ny + (j - g.nys);
    for (int l0 = 0; l0 < ncx && j <= g.nye; l0 += RX) {
      const int li = l0 + lane / G, i = i0 + li;
      int pe = 0, t = lg;
      if (i <= g.nxge) {  // uniform within a group
        const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1) + (i - g.nxgs);
        const int base = a.rowbaseA[rw];
        t = base + cr[0] + lg;
        pe = base + cr[1];
      }
      // (a cell's surplus lanes kick a particle at rest at its centre)
      Rec pr = {i + 0.5, j + 0.5, 0.0, 0.0, 0.0, 0};
      int ia_n = t + G;
      if (KICK && a.ap) ia_n = t + G < pe ? a.ap[t + G] : 0;
      if (t < pe) pr = KICK ? load_rec(a.A, a.ap ? a.ap[t] : t) : load_rec(a.B, t);
      while (__any(t < pe)) {
        double q[KP][8];  // dx, dy and the six moments u/gamma, u^2/gamma of the last KP passes, the latest first
        int at[KP];       // node of dx, dy: bit 0 x, bit 1 y (0: i-1, j-1); -1: nothing to add
#pragma unroll
        for (int h = 0; h < KP; h++) {
          at[h] = -1;
#pragma unroll
          for (int k = 0; k < 8; k++) q[h][k] = 0.0;
        }
        for (int h = 0; h < KP && __any(t < pe); h++, t += G) {
          const Rec p = pr;
          if (t + G < pe) pr = KICK ? load_rec(a.A, ia_n) : load_rec(a.B, t + G);
          if (KICK) {
            ia_n = t + 2 * G;
            if (a.ap) ia_n = t + 2 * G < pe ? a.ap[t + 2 * G] : 0;
          }
          double u[3] = {p.ux, p.uy, p.uz};
          if constexpr (KICK) {
            double nxp, nyp, gmv;
            boris_push(sf, li, lj, i, j, hdelt, c, true, a.fac1[s], a.txxx[s], a.fac2[s], p.x, p.y, p.ux, p.uy, p.uz,
                       nxp, nyp, u[0], u[1], u[2], gmv);
          }
          const int ih = (int)(p.x - 0.5), jh = (int)(p.y - 0.5);
          const double u2 = +u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
          double root, gam;
          sqrt_and_inverse(1.0 + (unit_c ? u2 : u2 / (c * c)), root, gam);
#pragma unroll
          for (int r = KP - 1; r > 0; r--) {
            at[r] = at[r - 1];
#pragma unroll
            for (int k = 0; k < 8; k++) q[r][k] = q[r - 1][k];
          }
          const double dx = p.x - 0.5 - ih, dxm = 1. - dx, dy = p.y - 0.5 - jh, dym = 1. - dy;
          double m[7] = {1.0};
#pragma unroll
          for (int d = 0; d < 3; d++) {
            m[1 + d] = u[d] * gam;
            m[4 + d] = u[d] * u[d] * gam;
          }
          const bool act = t < pe, in_cell = (unsigned)(ih - i + 1) < 2u && (unsigned)(jh - j + 1) < 2u;
          const bool add = act && in_cell;
          at[0] = add ? (ih - i + 1) | (jh - j + 1) << 1 : -1;
          q[0][0] = dx;
          q[0][1] = dy;
#pragma unroll
          for (int k = 1; k < 7; k++) q[0][1 + k] = add ? m[k] : 0.0;
          if (act && !in_cell) {
            if (ih < g.nxgs - 1 || ih > g.nxge || jh < j - 1 || jh > j) {
              atomicOr(a.err, ERR_DOMAIN);
            } else {
              const int lx = ih - (i0 - 1), ly = jh - (j0 - 1);
              const bool tiled = lx >= 0 && lx <= ncx;
              double* const node = &mt[0][0] + (tiled ? ly * MTW + lx : 0);
              double* const far = a.mom + midx(g, ih, jh, s);
              const size_t up = (size_t)7 * (g.nx + 2);
#pragma unroll
              for (int k = 0; k < 7; k++) {
                const double v[4] = {m[k] * (dxm * dym), m[k] * (dx * dym), m[k] * (dxm * dy), m[k] * (dx * dy)};
                if (tiled) {
                  double* const o = node + k * (MTW * MTH);
                  atomicAdd(o, v[0]);
                  atomicAdd(o + 1, v[1]);
                  atomicAdd(o + MTW, v[2]);
                  atomicAdd(o + MTW + 1, v[3]);
                } else {
                  unsafeAtomicAdd(far + k, v[0]);
                  unsafeAtomicAdd(far + 7 + k, v[1]);
                  unsafeAtomicAdd(far + up + k, v[2]);
                  unsafeAtomicAdd(far + up + 7 + k, v[3]);
                }
              }
            }
          }
        }
        double v[63];  // [moment][y node][x node]
#pragma unroll
        for (int k = 0; k < 63; k++) v[k] = 0.0;
#pragma unroll
        for (int h = 0; h < KP; h++) {
          if (!__any(at[h] >= 0)) continue;
          const bool xr = at[h] & 1, yr = at[h] & 2;
          const bool add = at[h] >= 0;
          const double dx = add ? q[h][0] : 0.0, dxm = (add ? 1.0 : 0.0) - dx;
          const double dy = add ? q[h][1] : 0.0, dym = 1. - dy;
          const double wx[3] = {xr ? 0.0 : dxm, xr ? dxm : dx, xr ? dx : 0.0};
          const double wy[3] = {yr ? 0.0 : dym, yr ? dym : dy, yr ? dy : 0.0};
#pragma unroll
          for (int e = 0; e < 9; e++) {
            const double w = wx[e % 3] * wy[e / 3];
            v[e] += w;
#pragma unroll
            for (int k = 1; k < 7; k++) v[9 * k + e] = fma(q[h][1 + k], w, v[9 * k + e]);
          }
        }
        group_reduce<63, G>(v, lane);
        int ln = lane;
        asm volatile("" : "+v"(ln));  // (the places worked out here, not kept over the passes)
#pragma unroll
        for (int f = 0; f < group_left(63, G); f++) {
          const int e = group_index<63, G>(f, ln);
          if (i <= g.nxge && e >= 0 && v[f] != 0.0)
            atomicAdd(&mt[0][0] + ((e / 9) * (MTW * MTH) + (lj + e % 9 / 3) * MTW + li + e % 3), v[f]);
        }
      }
    }
    __syncthreads();
    for (int k = tid; k < 7 * MTW * MTH; k += NT) {
      const int node = k / 7, comp = k % 7;
      const double v = mt[comp][node];
      if (v == 0.0) continue;
      const int I = i0 - 1 + node % MTW, J = j0 - 1 + node / MTW;
      if (I > g.nxge + 1 || J > g.nye + 1) continue;
      unsafeAtomicAdd(a.mom + midx(g, I, J, s) + comp, v);
    }
    __syncthreads();
  }
}

// gp in any slot order (rows of B): one thread per particle, HBM atomics
__global__ __launch_bounds__(NT) void k_mom_any(MomArgs a) {
  const Grid2D& g = a.g;
  const int rw = blockIdx.y, s = rw / g.ny, j = g.nys + rw % g.ny;
  const int base = a.rowbaseB[rw], n = a.np2B[rw];
  for (int t = blockIdx.x * NT + threadIdx.x; t < n; t += gridDim.x * NT) {
    const int pi = base + t;
    const double x = a.B.x[pi], y = a.B.y[pi];
    const int ih = (int)(x * g.d_delx - 0.5), jh = (int)(y * g.d_delx - 0.5);
    if (ih < g.nxgs - 1 || ih > g.nxge || jh < j - 1 || jh > j) {
      atomicOr(a.err, ERR_DOMAIN);
      continue;
    }
    const double dx = x * g.d_delx - 0.5 - ih, dxm = 1. - dx;
    const double dy = y * g.d_delx - 0.5 - jh, dym = 1. - dy;
    MomTerms m;
    m.set(a.B.ux[pi], a.B.uy[pi], a.B.uz[pi], g.c);
    double* p00 = a.mom + midx(g, ih, jh, s);
    double* p10 = a.mom + midx(g, ih + 1, jh, s);
    double* p01 = a.mom + midx(g, ih, jh + 1, s);
    double* p11 = a.mom + midx(g, ih + 1, jh + 1, s);
#pragma unroll
    for (int k = 0; k < 7; k++) {
      unsafeAtomicAdd(p00 + k, m.term(k, dxm, dym));
      unsafeAtomicAdd(p10 + k, m.term(k, dx, dym));
      unsafeAtomicAdd(p01 + k, m.term(k, dxm, dy));
      unsafeAtomicAdd(p11 + k, m.term(k, dx, dy));
    }
  }
}

// ---------------------------------------------------------------------------
// parity: thread per node (n, m) and species.  The particles that reach node
// row m live in rows m-1..m+1 (lower node jh in {j-1, j}); with gp
// slot-aligned with the sorted up only cells n-1..n+1 of those rows can reach
// node n, a contiguous slot range.  Each node adds its terms in the
// reference's (j, ii) order, starting from +0 like the OMP REDUCTION copy.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(NT) void k_mom_parity(MomArgs a, int aligned) {
  const Grid2D& g = a.g;
  const int n = g.nxgs - 1 + blockIdx.x * NT + threadIdx.x;
  if (n > g.nxge + 1) return;
  const int mh = g.ny + 2;
  const int s = blockIdx.y / mh, m = g.nys - 1 + blockIdx.y % mh;
  double acc[7];
#pragma unroll
  for (int k = 0; k < 7; k++) acc[k] = 0.0;
  for (int j = max(g.nys, m - 1); j <= min(g.nye, m + 1); j++) {
    const int rw = s * g.ny + (j - g.nys);
    const int base = a.rowbaseB[rw];
    int pb = 0, pe = a.np2B[rw];
    if (aligned) {
      const int lo = max(g.nxgs, n - 1), hi = min(g.nxge, n + 1);
      const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
      pb = cr[lo - g.nxgs];
      pe = cr[hi + 1 - g.nxgs];
    }
    Rec next{};  // (the next record on its way while one is added)
    if (pb < pe) next = load_rec(a.B, base + pb);
    for (int p = pb; p < pe; p++) {
      const Rec r = next;
      if (p + 1 < pe) next = load_rec(a.B, base + p + 1);
      const double x = r.x, y = r.y;
      const int ih = (int)(x * g.d_delx - 0.5), jh = (int)(y * g.d_delx - 0.5);
      if (ih < g.nxgs - 1 || ih > g.nxge || jh < j - 1 || jh > j) {
        atomicOr(a.err, ERR_DOMAIN);
        continue;
      }
      double wx, wy;
      const double dx = x * g.d_delx - 0.5 - ih, dy = y * g.d_delx - 0.5 - jh;
      if (ih == n)
        wx = 1. - dx;
      else if (ih + 1 == n)
        wx = dx;
      else
        continue;
      if (jh == m)
        wy = 1. - dy;
      else if (jh + 1 == m)
        wy = dy;
      else
        continue;
      MomTerms t;
      t.set(r.ux, r.uy, r.uz, g.c);
#pragma unroll
      for (int k = 0; k < 7; k++) acc[k] = acc[k] + t.term(k, wx, wy);
    }
  }
  double* o = a.mom + midx(g, n, m, s);
#pragma unroll
  for (int k = 0; k < 7; k++) o[k] = acc[k];
}

// ---------------------------------------------------------------------------
// boundary folds at one rank: x over all node rows (periodic: nxge+1 onto
// nxgs, nxgs-1 onto nxge; walls: each ghost onto its own edge), then y
// (nys-1 onto nye, then nye+1 onto nys) over all x nodes.
// ---------------------------------------------------------------------------
__global__ void k_mom_bc_x(Grid2D g, double* mom) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int mh = g.ny + 2;
  if (t >= 7 * mh * g.nsp) return;
  const int k = t % 7, jj = (t / 7) % mh, s = t / (7 * mh);
  const int j = g.nys - 1 + jj;
  const bool wall = walls(g);
  const int xa = wall ? g.nxgs - 1 : g.nxge + 1, xb = wall ? g.nxge + 1 : g.nxgs - 1;
  mom[midx(g, g.nxgs, j, s) + k] = mom[midx(g, g.nxgs, j, s) + k] + mom[midx(g, xa, j, s) + k];
  mom[midx(g, g.nxge, j, s) + k] = mom[midx(g, g.nxge, j, s) + k] + mom[midx(g, xb, j, s) + k];
}

__global__ void k_mom_bc_y(Grid2D g, double* mom) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int mw = g.nx + 2;
  if (t >= 7 * mw * g.nsp) return;
  const int k = t % 7, ii = (t / 7) % mw, s = t / (7 * mw);
  const int i = g.nxgs - 1 + ii;
  mom[midx(g, i, g.nye, s) + k] = mom[midx(g, i, g.nye, s) + k] + mom[midx(g, i, g.nys - 1, s) + k];
  mom[midx(g, i, g.nys, s) + k] = mom[midx(g, i, g.nys, s) + k] + mom[midx(g, i, g.nye + 1, s) + k];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static MomArgs mom_args(wpic_ctx* c) {
  MomArgs a;
  a.g = c->g;
  a.A = c->A;
  a.B = c->B;
  a.rowbaseA = c->rowbaseA;
  a.np2A = c->np2A;
  a.rowbaseB = c->rowbaseB;
  a.np2B = c->np2B;
  a.cumcnt = c->cumcnt;
  a.ap = c->aperm;
  a.uf = c->uf;
  a.mom = c->mom;
  a.err = c->err;
  a.ntx = (c->g.nx + TX - 1) / TX;
  a.nty = (c->g.ny + TY - 1) / TY;
  // mom_calc__init halves delt (mom_calc.f90:34); fac1, txxx, fac2 as
  // mom_calc.f90:90-92
  const double delt = c->g.delt * 0.5;
  for (int s = 0; s < WPIC_MAXSP; s++) {
    const double q = c->g.q[s], r = c->g.r[s];
    a.fac1[s] = s < c->g.nsp ? q / r * 0.5 * delt : 0.0;
    a.txxx[s] = a.fac1[s] * a.fac1[s];
    a.fac2[s] = s < c->g.nsp ? q * delt / r : 0.0;
  }
  return a;
}

hipError_t launch_mom_accl(wpic_ctx* c) {
  MomArgs a = mom_args(c);
  hipLaunchKernelGGL(k_mom_accl, dim3(xcd_grid(a.ntx * a.nty)), dim3(NT), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_mom_deposit(wpic_ctx* c, int kind) {
  MomArgs a = mom_args(c);
  const size_t nm = (size_t)7 * (c->g.nx + 2) * (c->g.ny + 2) * c->g.nsp;
  if (kind != MOM_PARITY_ALIGNED && kind != MOM_PARITY_ANY) {
    hipError_t e = launch_zero(c, c->mom, nm);
    if (e != hipSuccess) return e;
  }
  switch (kind) {
    case MOM_TILE_KICK:
      hipLaunchKernelGGL(k_mom_tile<true>, dim3(xcd_grid(a.ntx * a.nty)), dim3(NT), 0, c->st, a);
      break;
    case MOM_TILE_GP:
      hipLaunchKernelGGL(k_mom_tile<false>, dim3(xcd_grid(a.ntx * a.nty)), dim3(NT), 0, c->st, a);
      break;
    case MOM_ANY:
      hipLaunchKernelGGL(k_mom_any, dim3(8, c->g.nsp * c->g.ny), dim3(NT), 0, c->st, a);
      break;
    default:
      hipLaunchKernelGGL(k_mom_parity, dim3((c->g.nx + 2 + NT - 1) / NT, c->g.nsp * (c->g.ny + 2)), dim3(NT), 0,
                         c->st, a, kind == MOM_PARITY_ALIGNED ? 1 : 0);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_mom_bc(wpic_ctx* c) {
  const Grid2D& g = c->g;
  const int nx_t = 7 * (g.ny + 2) * g.nsp, ny_t = 7 * (g.nx + 2) * g.nsp;
  hipLaunchKernelGGL(k_mom_bc_x, dim3((nx_t + 255) / 256), dim3(256), 0, c->st, g, c->mom);
  hipLaunchKernelGGL(k_mom_bc_y, dim3((ny_t + 255) / 256), dim3(256), 0, c->st, g, c->mom);
  return hipGetLastError();
}

}  // namespace wpic
