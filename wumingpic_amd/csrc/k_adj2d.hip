// k_adj2d.hip -- hand-written adjoint kernels of the 2D periodic step loop
// (FP64): the sort permutation, the implicit field update and the fused
// Buneman-Boris push + Esirkepov deposit.  No reference counterpart.
//
// Adjoint state: lamA / lamB hold dL/d(x, y, ux, uy, uz) per particle slot
// (5 planes over the particle capacity) of the sorted state and of gp; lamF
// holds dL/d(uf) on the interior nodes (6 planes of nx*ny; the ghost nodes are
// periodic images, so their adjoint is folded into the interior); lamJ holds
// dL/d(uj) after the current ghost fold (3 planes of nx*ny).
//
// Forward step (periodic):  gp = push(up, uf);  J = deposit(up, gp);
//   b_l = f5 gkl_l(uf, J);  dB_l = M^-1 b_l (M = f4 - 4-neighbour sum, SPD);
//   dE = E(dB, uf, J);  uf' = uf + (dB, dE);  up' = sort(wrap(gp)).
// Reverse step: lamB = lamA' through the sort permutation (wraps are shifts);
//   lamF, lamJ from the transposed field update (the three CG solves with the
//   symmetric M); lamA, and lamF through the gather, from the push/deposit
//   adjoint of each particle recomputed from its stored start state.
#include "wpic_internal.h"

namespace wpic {

namespace {

constexpr double kPiA = 3.141592653589793;

__device__ inline int wrapi(const Grid2D& g, int i) { return i < g.nxgs ? i + g.nx : (i > g.nxge ? i - g.nx : i); }
__device__ inline int wrapj(const Grid2D& g, int j) { return j < g.nys ? j + g.ny : (j > g.nye ? j - g.ny : j); }
// interior index of the periodic image of node (i, j), at most one period out
__device__ inline int pix(const Grid2D& g, int i, int j) { return cidx(g, wrapi(g, i), wrapj(g, j)); }

__device__ inline void shape_d(double dh, double s[3], double ds[3]) {
  s[0] = 0.5 * (0.5 - dh) * (0.5 - dh);
  s[1] = 0.75 - dh * dh;
  s[2] = 0.5 * (0.5 + dh) * (0.5 + dh);
  ds[0] = -(0.5 - dh);
  ds[1] = -2.0 * dh;
  ds[2] = 0.5 + dh;
}

__device__ inline double cell_field_a(const Grid2D& g, const double* uf, int c, int i, int j) {
  const size_t pl = (size_t)g.fw * g.fh;
  const double* u = uf + pl * c;
  switch (c) {
    case 0: return 0.5 * (u[fidx(g, i, j)] + u[fidx(g, i, j + 1)]);
    case 1: return 0.5 * (u[fidx(g, i, j)] + u[fidx(g, i + 1, j)]);
    case 2: return 0.25 * (u[fidx(g, i, j)] + u[fidx(g, i + 1, j)] + u[fidx(g, i, j + 1)] + u[fidx(g, i + 1, j + 1)]);
    case 3: return 0.5 * (u[fidx(g, i, j)] + u[fidx(g, i + 1, j)]);
    case 4: return 0.5 * (u[fidx(g, i, j)] + u[fidx(g, i, j + 1)]);
    default: return u[fidx(g, i, j)];
  }
}

__device__ inline void cross(const double a[3], const double b[3], double o[3]) {
  o[0] = a[1] * b[2] - a[2] * b[1];
  o[1] = a[2] * b[0] - a[0] * b[2];
  o[2] = a[0] * b[1] - a[1] * b[0];
}

}  // namespace

// ---------------------------------------------------------------------------
// sort permutation: lamB[perm[k]] = lamA[k] over the active slots of the
// post-step state (perm maps a sorted slot to the gp slot it was gathered from)
// ---------------------------------------------------------------------------
__global__ void k_adj_unsort(Grid2D g, const int* rowbase, const int* np2, const int* perm, const double* lamA,
                             double* lamB, size_t N) {
  const int rw = blockIdx.x;
  const int base = rowbase[rw], n = np2[rw];
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const int d = base + k, s = perm[d];
    if ((size_t)s >= N) continue;
    for (int c = 0; c < 5; c++) lamB[c * N + s] = lamA[c * N + d];
  }
}

// ---------------------------------------------------------------------------
// field update, transposed (2d/common/field.f90:125-184 in reverse)
// ---------------------------------------------------------------------------
// from the E update: lam(dB) into the CG right-hand sides, lam(uf) terms of
// the curl of B, lamJ = -4 pi dt lam(E)
__global__ void k_adj_field1(Grid2D g, const double* __restrict__ lamF, double* __restrict__ lamF2,
                             double* __restrict__ b, double* __restrict__ lamJ) {
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const double f1 = g.f1, gf = g.gfac, pdt = g.pi4dt;
  const double *LBx = lamF, *LBy = lamF + n, *LBz = lamF + 2 * n, *LEx = lamF + 3 * n, *LEy = lamF + 4 * n,
               *LEz = lamF + 5 * n;
  const double cz = (-LEx[k] + LEx[pix(g, i, j - 1)]) + (LEy[k] - LEy[pix(g, i - 1, j)]);
  const double cy = -LEz[k] + LEz[pix(g, i - 1, j)];
  const double cx = LEz[k] - LEz[pix(g, i, j - 1)];
  b[k] = LBx[k] + f1 * gf * cx;
  b[n + k] = LBy[k] + f1 * gf * cy;
  b[2 * n + k] = LBz[k] + f1 * gf * cz;
  lamF2[k] = LBx[k] + f1 * cx;
  lamF2[n + k] = LBy[k] + f1 * cy;
  lamF2[2 * n + k] = LBz[k] + f1 * cz;
  lamF2[3 * n + k] = LEx[k];
  lamF2[4 * n + k] = LEy[k];
  lamF2[5 * n + k] = LEz[k];
  lamJ[k] = -pdt * LEx[k];
  lamJ[n + k] = -pdt * LEy[k];
  lamJ[2 * n + k] = -pdt * LEz[k];
}

// warm start and |b|^2 partials for the transposed solves (the CG kernels of
// the forward then run unchanged on b and phi)
__global__ __launch_bounds__(256) void k_adj_cg_init(Grid2D g, double* phi, const double* b, double* r, double* pold,
                                                     double* part, int nb, int parity) {
  __shared__ double sh[4];
  const int n = g.nx * g.ny;
  double s[3] = {0.0, 0.0, 0.0};
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += nb * 256) {
#pragma unroll
    for (int l = 0; l < 3; l++) {
      const size_t q = (size_t)l * n + k;
      const double v = b[q];
      phi[q] = 0.0;
      r[q] = v;
      if (parity) pold[q] = v;
      s[l] = s[l] + v * v;
    }
  }
  if (parity) return;
  for (int l = 0; l < 3; l++) {
    double v = s[l];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      const double t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
      part[(l * 3 + 0) * NPB + blockIdx.x] = t;  // r.r
      part[(l * 3 + 2) * NPB + blockIdx.x] = t;  // b.b
    }
    __syncthreads();
  }
}

// from the right-hand side gkl: mu = M^-1 lam(dB) solved, lam(gkl) = f5 mu
__global__ void k_adj_field2(Grid2D g, const double* __restrict__ mu, double* __restrict__ lamF2,
                             double* __restrict__ lamJ) {
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const double f1 = g.f1, f2 = g.f2, f3 = g.f3, f5 = g.f5;
  const double *M1 = mu, *M2 = mu + n, *M3 = mu + 2 * n;
  const int kW = pix(g, i - 1, j), kE = pix(g, i + 1, j), kS = pix(g, i, j - 1), kN = pix(g, i, j + 1);
  const double g1 = f5 * M1[k], g2 = f5 * M2[k], g3 = f5 * M3[k];
  const double g1N = f5 * M1[kN], g2E = f5 * M2[kE], g3E = f5 * M3[kE], g3N = f5 * M3[kN];
  // the 5-point Laplacian is symmetric
  const double lap1 = f5 * (M1[kS] + M1[kW] - 4.0 * M1[k] + M1[kE] + M1[kN]);
  const double lap2 = f5 * (M2[kS] + M2[kW] - 4.0 * M2[k] + M2[kE] + M2[kN]);
  const double lap3 = f5 * (M3[kS] + M3[kW] - 4.0 * M3[k] + M3[kE] + M3[kN]);
  lamF2[k] += f2 * lap1;
  lamF2[n + k] += f2 * lap2;
  lamF2[2 * n + k] += f2 * lap3;
  lamF2[3 * n + k] += -f1 * (g3N - g3);
  lamF2[4 * n + k] += -f1 * (g3 - g3E);
  lamF2[5 * n + k] += -f1 * (g1 - g1N) + f1 * (g2 - g2E);
  lamJ[k] += f2 * f3 * (g3N - g3);
  lamJ[n + k] += f2 * f3 * (g3 - g3E);
  lamJ[2 * n + k] += f2 * f3 * (g1 - g1N) - f2 * f3 * (g2 - g2E);
}

// the gather's cell-centred fields, transposed onto the staggered nodes
// (particle.f90:70-83: 2- and 4-point averages)
__global__ void k_adj_t2f(Grid2D g, const double* __restrict__ lamT, double* __restrict__ lamF) {
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const int kW = pix(g, i - 1, j), kS = pix(g, i, j - 1), kSW = pix(g, i - 1, j - 1);
  const double *T1 = lamT, *T2 = lamT + n, *T3 = lamT + 2 * n, *T4 = lamT + 3 * n, *T5 = lamT + 4 * n,
               *T6 = lamT + 5 * n;
  lamF[k] += 0.5 * (T1[k] + T1[kS]);
  lamF[n + k] += 0.5 * (T2[k] + T2[kW]);
  lamF[2 * n + k] += 0.25 * (T3[k] + T3[kW] + T3[kS] + T3[kSW]);
  lamF[3 * n + k] += 0.5 * (T4[k] + T4[kW]);
  lamF[4 * n + k] += 0.5 * (T5[k] + T5[kS]);
  lamF[5 * n + k] += T6[k];
}

// ---------------------------------------------------------------------------
// push + deposit, per particle, recomputed from the stored start state
// ---------------------------------------------------------------------------
struct AdjPArgs {
  Grid2D g;
  Parts P;
  const int *rowbase, *cumcnt;
  const double* uf;
  const double* lamB;  // [5][N]
  const double* lamJ;  // [3][nx*ny]
  double* lamA;        // [5][N]
  double* lamT;        // [6][nx*ny]
  size_t N;
  int ntx, nty, tw;
};

// (a, b, c) at nodes 0..4 of five, shifted from 1..3 by inc in {-1, 0, 1} (a
// step over two faces, which only rounding makes, at c delt = delx, has no
// derivative and counts as one)
__device__ inline void spread5(const double a[3], int inc, double o[5]) {
  const bool l = inc < 0, r = inc > 0;
  o[0] = l ? a[0] : 0.0;
  o[1] = l ? a[1] : (r ? 0.0 : a[0]);
  o[2] = l ? a[2] : (r ? a[0] : a[1]);
  o[3] = l ? 0.0 : (r ? a[1] : a[2]);
  o[4] = r ? a[2] : 0.0;
}
// its transpose: the three values of five that spread5 fills (from scalars that
// the compiler cannot see through: it would index an array in scratch)
__device__ inline void pick3(const double v[5], int inc, double a[3]) {
  const bool l = inc < 0, r = inc > 0;
  double o0 = v[0], o1 = v[1], o2 = v[2], o3 = v[3], o4 = v[4];
  asm volatile("" : "+v"(o0), "+v"(o1), "+v"(o2), "+v"(o3), "+v"(o4));
  a[0] = l ? o0 : (r ? o2 : o1);
  a[1] = l ? o1 : (r ? o3 : o2);
  a[2] = l ? o2 : (r ? o4 : o3);
}

// One workgroup per tile of cells, as in the push: the tile's cell-centred
// fields (one-cell halo) and the current's adjoint (two-cell halo) are read
// from LDS, the fields' adjoint is summed there and added to HBM once per
// node.  Eight lanes share a cell, so their LDS reads are broadcasts, and the
// 54 terms a particle adds to the fields' adjoint are summed over the eight
// before they meet in LDS.
//
// Bound by its FP64 instructions at 2 waves a SIMD (256 registers).  One thread
// per particle with every field, current and atomic in HBM took 6.57 ms at
// 256x256, 16 ppc (54 field stencils, read twice, 65 current reads and 54
// atomics a particle, and arrays indexed by the cell step in scratch); this
// took 0.255 ms with 224 bytes of scratch a thread.  Now 72 bytes (the node
// table in LDS, lamB loaded where it is used, pick3 without an array): a pass of
// 40 steps back 37.5 -> 35.5 ms.  At 1 wave a SIMD, without spills, it takes 3 %
// of a whole backward pass longer.
__global__ __launch_bounds__(256, 2) void k_adj_particles(AdjPArgs a) {
  constexpr int TX = 32, TY = 4, NT = 256, G = 8;
  constexpr int SFW = TX + 2, SFH = TY + 2, ACW = TX + 4, ACH = TY + 4;
  __shared__ double sf[6][SFW * SFH], lt[6][SFW * SFH];
  __shared__ double lj_[3][ACW * ACH];
  __shared__ double spc[WPIC_MAXSP][5];  // fac1, txxx, fac2, q, qk
  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * a.tw, j0 = g.nys + (tile / a.ntx) * TY;
  const int tid = threadIdx.x, ncell = g.nx * g.ny;
  const int sw = a.tw + 2, aw = a.tw + 4;
  for (int k = tid; k < sw * SFH; k += NT) {
    const int r = k / sw, q = k - r * sw;
    const int i = i0 - 1 + q, j = j0 - 1 + r;
    const bool in = i <= g.nxge + 1 && j <= g.nye + 1;
#pragma unroll
    for (int c = 0; c < 6; c++) {
      sf[c][r * SFW + q] = in ? cell_field_a(g, a.uf, c, i, j) : 0.0;
      lt[c][r * SFW + q] = 0.0;
    }
  }
  for (int k = tid; k < aw * ACH; k += NT) {
    const int r = k / aw, q = k - r * aw;
    const int i = i0 - 2 + q, j = j0 - 2 + r;
    const bool in = i <= g.nxge + 2 && j <= g.nye + 2;
#pragma unroll
    for (int c = 0; c < 3; c++) lj_[c][r * ACW + q] = in ? a.lamJ[(size_t)c * ncell + pix(g, i, j)] : 0.0;
  }
#pragma unroll
  for (int s = 0; s < WPIC_MAXSP; s++)
    if (tid == s && s < g.nsp) {
      const double q = g.q[s], rm = g.r[s], fac1 = q / rm * 0.5 * g.delt;
      spc[s][0] = fac1;
      spc[s][1] = fac1 * fac1;
      spc[s][2] = q * g.delt / rm;
      spc[s][3] = q;
      spc[s][4] = q * g.delx * g.d_delt;
    }
  __syncthreads();

  const double delt = g.delt, c2 = g.c * g.c;
  const size_t N = a.N;
  const int lj = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lg = lane % G;
  const int j = j0 + lj;
  // where a lane's sums of two components' 18 terms go in lt, from the cell's
  // lower left neighbour
  constexpr int NRES = group_left(18, G);
  __shared__ int node[NRES][G];
  if (tid < NRES * G) {
    const int q = group_index<18, G>(tid / G, tid % G);
    node[tid / G][tid % G] = q < 0 ? -1 : (q / 9) * (SFW * SFH) + (q % 9 / 3) * SFW + q % 3;
  }
  __syncthreads();
  for (int l0 = 0; l0 < a.tw; l0 += 64 / G) {
    const int li = l0 + lane / G, i = i0 + li;
    const bool live = i <= g.nxge && j <= g.nye;  // uniform within a group
    CellList cl;
    int tot = 0;
#pragma unroll
    for (int s = 0; s < WPIC_MAXSP; s++) {
      if (s < g.nsp) {
        int b0 = 0, b1 = 0, rb = 0;
        if (live) {
          const int rw = s * g.ny + (j - g.nys);
          const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1) + (i - g.nxgs);
          b0 = cr[0];
          b1 = cr[1];
          rb = a.rowbase[rw];
        }
        cl.set(s, rb + b0, tot);
        tot += b1 - b0;
      } else {
        cl.set(s, 0, 0x7fffffff);
      }
    }
    const int so = lj * SFW + li;  // the cell's lower left neighbour in sf and lt
    const int ao = lj * ACW + li;  // node (-2, -2) in lj_
    for (int t = lg; __any(t < tot); t += G) {
      const bool act = t < tot;
      int s, p;
      cl.slot(g.nsp, t, s, p);
      Rec P = {i + 0.5, j + 0.5, 0.0, 0.0, 0.0, 0};
      double G_xn = 0.0, G_yn = 0.0, G_g[3] = {0.0, 0.0, 0.0};
      if (act) {
        P = load_rec(a.P, p);
      }
      const double x = P.x, y = P.y, u[3] = {P.ux, P.uy, P.uz};
      const double fac1 = spc[s][0], txxx = spc[s][1], fac2 = spc[s][2], q = spc[s][3], qk = spc[s][4];
      // ---- forward recomputation ----
      double sx[3], dsxdh[3], sy[3], dsydh[3];
      shape_d(x - 0.5 - i, sx, dsxdh);
      shape_d(y - 0.5 - j, sy, dsydh);
      double F[6];
#pragma unroll
      for (int cm = 0; cm < 6; cm++) {
        double f = 0.0;
#pragma unroll
        for (int b = 0; b < 3; b++) {
          const double* r = &sf[cm][so + b * SFW];
          f = fma(fma(r[2], sx[2], fma(r[1], sx[1], r[0] * sx[0])), sy[b], f);
        }
        F[cm] = f;
      }
      // (combined here, not where a later block uses them)
      asm volatile("" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]), "+v"(F[5]));
      const double B[3] = {F[0], F[1], F[2]}, E[3] = {F[3], F[4], F[5]};
      double uvm[3];
#pragma unroll
      for (int d = 0; d < 3; d++) uvm[d] = u[d] + fac1 * E[d];
      const double gam = sqrt(c2 + uvm[0] * uvm[0] + uvm[1] * uvm[1] + uvm[2] * uvm[2]);
      const double igam = 1.0 / gam;
      const double fac1r = fac1 * igam;
      const double B2 = B[0] * B[0] + B[1] * B[1] + B[2] * B[2];
      const double iD = 1.0 / (gam + txxx * B2 * igam);
      const double fac2r = fac2 * iD;
      double v2[3], tt[3], ww[3], gv[3];
      cross(uvm, B, v2);
#pragma unroll
      for (int d = 0; d < 3; d++) tt[d] = uvm[d] + fac1r * v2[d];
      cross(tt, B, ww);
#pragma unroll
      for (int d = 0; d < 3; d++) gv[d] = uvm[d] + fac2r * ww[d] + fac1 * E[d];
      const double g2 = gv[0] * gv[0] + gv[1] * gv[1] + gv[2] * gv[2];
      const double gmv = 1.0 / sqrt(1.0 + g2 / c2);
      const double xn = x + gv[0] * delt * gmv, yn = y + gv[1] * delt * gmv;
      // deposit shapes (fast-mode factored form of field.f90:274-298)
      const int i2 = (int)xn, j2 = (int)yn;
      const int incx = i2 - i, incy = j2 - j;
      double ds1x[3], ds1y[3];
      double s0x[5] = {0.0, sx[0], sx[1], sx[2], 0.0}, s0y[5] = {0.0, sy[0], sy[1], sy[2], 0.0};
      double dsx[5], dsy[5];
      {
        double s1[3];
        shape_d(xn - 0.5 - i2, s1, ds1x);
        spread5(s1, incx, dsx);
        shape_d(yn - 0.5 - j2, s1, ds1y);
        spread5(s1, incy, dsy);
      }
#pragma unroll
      for (int m = 0; m < 5; m++) {
        dsx[m] -= s0x[m];
        dsy[m] -= s0y[m];
      }
      const double qvz = q * (gv[2] * gmv);
      if (act) {
        G_xn = a.lamB[p];
        G_yn = a.lamB[N + p];
#pragma unroll
        for (int d = 0; d < 3; d++) G_g[d] = a.lamB[(2 + d) * N + p];
      }
      // (the phases one after another: interleaved, their values do not fit)
      // ---- reverse: deposit ----
      double G_dsx[5], G_dsy[5], G_s0x[5], G_s0y[5];
      {
        // Jx = cx(m) qk wy(n): cx(m) = -sum_{k<=m} dsx(k), wy = s0y + dsy/2
        double G_wy[5], G_cx[4] = {0.0, 0.0, 0.0, 0.0}, cx[4];
        cx[0] = -dsx[0];
#pragma unroll
        for (int m = 1; m < 4; m++) cx[m] = cx[m - 1] - dsx[m];
#pragma unroll
        for (int n = 0; n < 5; n++) {
          const double* r = &lj_[0][ao + n * ACW + 1];
          const double wy = fma(0.5, dsy[n], s0y[n]);
          double gw = 0.0;
#pragma unroll
          for (int m = 0; m < 4; m++) {
            G_cx[m] = fma(r[m], wy, G_cx[m]);
            gw = fma(r[m], cx[m], gw);
          }
          G_wy[n] = gw;
        }
        double run = 0.0;
        G_dsx[4] = 0.0;
#pragma unroll
        for (int m = 3; m >= 0; m--) {
          run -= G_cx[m];
          G_dsx[m] = qk * run;
        }
#pragma unroll
        for (int n = 0; n < 5; n++) {
          G_s0y[n] = qk * G_wy[n];
          G_dsy[n] = 0.5 * G_s0y[n];
        }
      }
      {
        double G_wx[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, G_cy[4], cy = 0.0;
        double wx[5];
#pragma unroll
        for (int n = 0; n < 5; n++) wx[n] = fma(0.5, dsx[n], s0x[n]);
#pragma unroll
        for (int m = 0; m < 4; m++) {
          cy -= dsy[m];
          const double* r = &lj_[1][ao + (m + 1) * ACW];
          double gc = 0.0;
#pragma unroll
          for (int n = 0; n < 5; n++) {
            gc = fma(r[n], wx[n], gc);
            G_wx[n] = fma(r[n], cy, G_wx[n]);
          }
          G_cy[m] = gc;
        }
        double run = 0.0;
#pragma unroll
        for (int m = 3; m >= 0; m--) {
          run -= G_cy[m];
          G_dsy[m] = fma(qk, run, G_dsy[m]);
        }
#pragma unroll
        for (int n = 0; n < 5; n++) {
          G_s0x[n] = qk * G_wx[n];
          G_dsx[n] = fma(0.5, G_s0x[n], G_dsx[n]);
        }
      }
      double G_qvz = 0.0;
#pragma unroll
      for (int n = 0; n < 5; n++) {
        // Jz = qvz (s0x(m) A(n) + dsx(m) B(n)), A = s0y + dsy/2, B = s0y/2 + dsy/3
        const double* r = &lj_[2][ao + n * ACW];
        const double A = fma(0.5, dsy[n], s0y[n]), Bn = fma(1.0 / 3.0, dsy[n], 0.5 * s0y[n]);
        double ga = 0.0, gb = 0.0;
#pragma unroll
        for (int m = 0; m < 5; m++) {
          const double L = r[m];
          G_s0x[m] = fma(qvz * L, A, G_s0x[m]);
          G_dsx[m] = fma(qvz * L, Bn, G_dsx[m]);
          ga = fma(L, s0x[m], ga);
          gb = fma(L, dsx[m], gb);
        }
        G_qvz = fma(ga, A, fma(gb, Bn, G_qvz));
        G_s0y[n] = fma(qvz, fma(0.5, gb, ga), G_s0y[n]);
        G_dsy[n] = fma(qvz, fma(0.5, ga, gb * (1.0 / 3.0)), G_dsy[n]);
      }
      double h[3];
      pick3(G_dsx, incx, h);
      G_xn += h[0] * ds1x[0] + h[1] * ds1x[1] + h[2] * ds1x[2];
      pick3(G_dsy, incy, h);
      G_yn += h[0] * ds1y[0] + h[1] * ds1y[1] + h[2] * ds1y[2];
      double G_sx[3], G_sy[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        G_sx[k] = G_s0x[k + 1] - G_dsx[k + 1];
        G_sy[k] = G_s0y[k + 1] - G_dsy[k + 1];
      }
      // ---- reverse: move, x' = x + g dt gmv ----
      double G_gmv = q * gv[2] * G_qvz + gv[0] * delt * G_xn + gv[1] * delt * G_yn;
      G_g[2] += q * gmv * G_qvz;
      G_g[0] += delt * gmv * G_xn;
      G_g[1] += delt * gmv * G_yn;
      const double dgmv = -gmv * gmv * gmv / c2;
#pragma unroll
      for (int d = 0; d < 3; d++) G_g[d] += G_gmv * dgmv * gv[d];
      double G_x = G_xn, G_y = G_yn;
      // ---- reverse: Boris ----
      double G_E[3], G_B[3], G_uvm[3], G_w[3], G_t[3], tmp[3], G_v2[3];
      const double G_fac2r = G_g[0] * ww[0] + G_g[1] * ww[1] + G_g[2] * ww[2];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        G_E[d] = fac1 * G_g[d];
        G_uvm[d] = G_g[d];
        G_w[d] = fac2r * G_g[d];
      }
      cross(B, G_w, G_t);   // d(t x B).v / dt = B x v
      cross(G_w, tt, G_B);  // d(t x B).v / dB = v x t
      const double G_fac1r = G_t[0] * v2[0] + G_t[1] * v2[1] + G_t[2] * v2[2];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        G_uvm[d] += G_t[d];
        G_v2[d] = fac1r * G_t[d];
      }
      cross(B, G_v2, tmp);
#pragma unroll
      for (int d = 0; d < 3; d++) G_uvm[d] += tmp[d];
      cross(G_v2, uvm, tmp);
#pragma unroll
      for (int d = 0; d < 3; d++) G_B[d] += tmp[d];
      // fac2r = fac2 / D, D = gam + txxx |B|^2 igam, fac1r = fac1 igam, igam = 1/gam
      const double G_D = -fac2r * iD * G_fac2r;
      const double G_igam = txxx * B2 * G_D + fac1 * G_fac1r;
      const double G_gam = G_D - igam * igam * G_igam;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        G_B[d] += 2.0 * txxx * igam * B[d] * G_D;
        G_uvm[d] += uvm[d] * igam * G_gam;
        G_E[d] += fac1 * G_uvm[d];  // uvm = u + fac1 E
      }
      // ---- reverse: gather F_c = sum T sx sy ----
      double G_F[6] = {G_B[0], G_B[1], G_B[2], G_E[0], G_E[1], G_E[2]};
#pragma unroll
      for (int cm = 0; cm < 6; cm++) {
#pragma unroll
        for (int b = 0; b < 3; b++) {
          const double* r = &sf[cm][so + b * SFW];
          const double gy = G_F[cm] * sy[b];
          G_sx[0] = fma(r[0], gy, G_sx[0]);
          G_sx[1] = fma(r[1], gy, G_sx[1]);
          G_sx[2] = fma(r[2], gy, G_sx[2]);
          G_sy[b] = fma(G_F[cm], fma(r[2], sx[2], fma(r[1], sx[1], r[0] * sx[0])), G_sy[b]);
        }
        if (!act) G_F[cm] = 0.0;
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        G_x += G_sx[k] * dsxdh[k];
        G_y += G_sy[k] * dsydh[k];
      }
      if (act) {
        a.lamA[p] = G_x;
        a.lamA[N + p] = G_y;
#pragma unroll
        for (int d = 0; d < 3; d++) a.lamA[(2 + d) * N + p] = G_uvm[d];
      }
#pragma unroll
      for (int cp = 0; cp < 6; cp += 2) {
        double v[18];
#pragma unroll
        for (int k = 0; k < 18; k++) v[k] = G_F[cp + k / 9] * sx[k % 3] * sy[k % 9 / 3];
        group_reduce<18, G>(v, lane);
#pragma unroll
        for (int f = 0; f < NRES; f++) {
          const int n = node[f][lg];
          if (live && n >= 0) atomicAdd(&lt[cp][0] + (n + so), v[f]);
        }
      }
    }
  }
  __syncthreads();
  for (int k = tid; k < sw * SFH; k += NT) {
    const int r = k / sw, q = k - r * sw;
    const int i = i0 - 1 + q, j = j0 - 1 + r;
    if (i > g.nxge + 1 || j > g.nye + 1) continue;
    const int n = pix(g, i, j);
#pragma unroll
    for (int c = 0; c < 6; c++) {
      const double v = lt[c][r * SFW + q];
      if (v != 0.0) unsafeAtomicAdd(&a.lamT[(size_t)c * ncell + n], v);
    }
  }
}

// ---------------------------------------------------------------------------
// objective and parameters
// ---------------------------------------------------------------------------
// lamF = dW_B/duf on the interior: B/(4 pi) for Bx, By, Bz, zero for E
__global__ void k_adj_seed(Grid2D g, const double* uf, double* lamF, double seed) {
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const size_t pl = (size_t)g.fw * g.fh;
  const int f = fidx(g, i, j);
  for (int c = 0; c < 3; c++) lamF[(size_t)c * n + k] = seed * uf[pl * c + f] / (4.0 * kPiA);
  for (int c = 3; c < 6; c++) lamF[(size_t)c * n + k] = 0.0;
}

// per-block partial sums of dL/d(udrift), dL/d(uth_e), dL/d(amp) from the
// initial state (electrons = the last species; the beam sign alternates by
// in-cell slot as the seeded state assigns it)
__global__ __launch_bounds__(256) void k_adj_params(Grid2D g, Parts P, const int* rowbase, const int* np2,
                                                    const double* lamA, size_t N, const double* lamF,
                                                    double udrift, double uth_e, int mode, int n_ppc, double* out) {
  __shared__ double sh[3][256];
  double sd = 0.0, st = 0.0, sa = 0.0;
  const int se = g.nsp - 1;
  for (int r = blockIdx.x; r < g.ny; r += gridDim.x) {
    const int rw = se * g.ny + r;
    const int base = rowbase[rw], n = np2[rw];
    for (int k = threadIdx.x; k < n; k += 256) {
      const int p = base + k;
      const long long pid = -(long long)P.id[p];
      const long long sl = (pid - 1) % n_ppc;
      const double sgn = (sl & 1) ? -1.0 : 1.0;
      const double lx = lamA[2 * N + p], ly = lamA[3 * N + p], lz = lamA[4 * N + p];
      sd += sgn * lx;
      if (uth_e != 0.0) st += (lx * (P.ux[p] - sgn * udrift) + ly * P.uy[p] + lz * P.uz[p]) / uth_e;
    }
  }
  const int n = g.nx * g.ny;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) {
    const int i = k % g.nx;
    sa += lamF[2 * (size_t)n + k] * sin(2.0 * kPiA * mode * i / g.nx);
  }
  sh[0][threadIdx.x] = sd;
  sh[1][threadIdx.x] = st;
  sh[2][threadIdx.x] = sa;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if (threadIdx.x < off)
      for (int c = 0; c < 3; c++) sh[c][threadIdx.x] += sh[c][threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; c++) out[blockIdx.x * 3 + c] = sh[c][0];
}

// Bz += amp sin(2 pi mode (i - nxgs) / nx) on every node (ghosts included)
__global__ void k_perturb_bz(Grid2D g, double* uf, double amp, int mode) {
  const int n = g.fw * g.fh;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs - 2 + k % g.fw;
  uf[2 * (size_t)n + k] += amp * sin(2.0 * kPiA * mode * (i - g.nxgs) / g.nx);
}

// adjoint of the initial state to the reference layouts (ghost nodes zero)
__global__ void k_adj_lamF_to_planes(Grid2D g, const double* lamF, double* planes) {
  const int n = g.nx * g.ny;
  const int npl = g.fw * g.fh;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npl) return;
  const int i = g.nxgs - 2 + k % g.fw, j = g.nys - 2 + k / g.fw;
  const bool in = i >= g.nxgs && i <= g.nxge && j >= g.nys && j <= g.nye;
  for (int c = 0; c < 6; c++) planes[(size_t)c * npl + k] = in ? lamF[(size_t)c * n + cidx(g, i, j)] : 0.0;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static unsigned cells_grid(const Grid2D& g) { return (unsigned)((g.nx * g.ny + 255) / 256); }

hipError_t launch_adj_unsort(wpic_ctx* c, const int* rows, const int* perm, const double* lamA, double* lamB,
                             size_t N) {
  const int nr = c->g.nsp * c->g.ny;
  hipLaunchKernelGGL(k_adj_unsort, dim3(nr), dim3(256), 0, c->st, c->g, rows, rows + nr, perm, lamA, lamB, N);
  return hipGetLastError();
}

hipError_t launch_adj_field1(wpic_ctx* c, const double* lamF, double* lamF2, double* lamJ) {
  hipLaunchKernelGGL(k_adj_field1, dim3(cells_grid(c->g)), dim3(256), 0, c->st, c->g, lamF, lamF2, c->bb, lamJ);
  const int nb = cg_blocks(c->g);
  hipLaunchKernelGGL(k_adj_cg_init, dim3(nb), dim3(256), 0, c->st, c->g, c->phi, c->bb, c->rr, c->pa, c->part, nb,
                     c->mode == WPIC_MODE_PARITY ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_adj_field2(wpic_ctx* c, double* lamF2, double* lamJ) {
  hipLaunchKernelGGL(k_adj_field2, dim3(cells_grid(c->g)), dim3(256), 0, c->st, c->g, c->phi, lamF2, lamJ);
  return hipGetLastError();
}

hipError_t launch_adj_particles(wpic_ctx* c, const Parts& P, const int* rows, const int* cumcnt, const double* uf,
                                const double* lamB, const double* lamJ, double* lamA, double* lamT, size_t N) {
  AdjPArgs a;
  a.g = c->g;
  a.P = P;
  a.rowbase = rows;
  a.cumcnt = cumcnt;
  a.uf = uf;
  a.lamB = lamB;
  a.lamJ = lamJ;
  a.lamA = lamA;
  a.lamT = lamT;
  a.N = N;
  a.tw = tile_width(c->g);
  a.ntx = (c->g.nx + a.tw - 1) / a.tw;
  a.nty = (c->g.ny + 3) / 4;
  hipLaunchKernelGGL(k_adj_particles, dim3(xcd_grid(a.ntx * a.nty)), dim3(256), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_adj_t2f(wpic_ctx* c, const double* lamT, double* lamF) {
  hipLaunchKernelGGL(k_adj_t2f, dim3(cells_grid(c->g)), dim3(256), 0, c->st, c->g, lamT, lamF);
  return hipGetLastError();
}

hipError_t launch_adj_seed(wpic_ctx* c, double* lamF, double seed) {
  hipLaunchKernelGGL(k_adj_seed, dim3(cells_grid(c->g)), dim3(256), 0, c->st, c->g, c->uf, lamF, seed);
  return hipGetLastError();
}

hipError_t launch_adj_params(wpic_ctx* c, const Parts& P, const int* rows, const double* lamA, size_t N,
                             const double* lamF, double udrift, double uth_e, int mode, int n_ppc,
                             double* out) {
  const int nr = c->g.nsp * c->g.ny;
  hipLaunchKernelGGL(k_adj_params, dim3(256), dim3(256), 0, c->st, c->g, P, rows, rows + nr, lamA, N, lamF,
                     udrift, uth_e, mode, n_ppc, out);
  return hipGetLastError();
}

hipError_t launch_perturb_bz(wpic_ctx* c, double amp, int mode) {
  const int n = c->g.fw * c->g.fh;
  hipLaunchKernelGGL(k_perturb_bz, dim3((n + 255) / 256), dim3(256), 0, c->st, c->g, c->uf, amp, mode);
  return hipGetLastError();
}

hipError_t launch_adj_lamF_to_planes(wpic_ctx* c, const double* lamF, double* planes) {
  const int n = c->g.fw * c->g.fh;
  hipLaunchKernelGGL(k_adj_lamF_to_planes, dim3((n + 255) / 256), dim3(256), 0, c->st, c->g, lamF, planes);
  return hipGetLastError();
}

}  // namespace wpic
