// k_push3d.hip -- 3D Buneman-Boris push (3d/common/particle.f90:52-233) and
// Esirkepov deposit (3d/common/field.f90:211-406) on tiles of cells.
//
// Push: one workgroup per TX x TY x TZ tile stages the cell-centred fields
// (tmpf, particle.f90:74-91) of the tile plus a one-cell halo in LDS; groups of
// G lanes walk one cell at a time and each lane pushes every G-th particle of
// the cell with the reference's operation order (27-point gather nested as
// ((x row) y) z, particle.f90:126-185), so gp is bit-identical to the
// reference's at any thread count.
//
// Deposit: each half-wave (32 lanes) owns one cell at a time.  Its lanes first
// compute the old/new shape arrays s0 and ds of up to 16 particles into LDS;
// then lane (jp, kp) (25 of the 32) walks those particles in slot order and
// accumulates the cell's pjx(:, jp, kp), pjy(:, jp, kp), pjz(:, jp, kp) with
// the reference's dstmp / running pjtmp arithmetic (field.f90:335-380) in
// parity mode, or in a factored form with FMA (the running sums of ds
// precomputed per particle) in fast mode.
// Parity mode writes the 300-entry block per cell; k_gather_pj3d then adds the
// blocks into uj in the reference's (k, j, i) cell order with the scatter
// permutation uj(2) += pjy(jp, ip, kp), uj(3) += pjz(kp, ip, jp) (:390-398),
// bit for bit.  Fast mode adds the blocks into an LDS tile accumulator and
// the tile into uj with atomics.
#include "k_push3d.h"

namespace wpic {

struct Push3Args {
  Grid3D g;
  Parts3 A, B;
  const int* colbase;
  const int* cumcnt;
  const int* ap;  // A's slot -> record in A's buffer (null: identity)
  const double* uf;
  double* uj;
  double* pjbuf;
  int ntx, nty, ntz;
  int vay;  // the Vay kick instead of Buneman-Boris (particle__solv_vay)
  int* code;  // fused fast kernel: the exchange codes of gp
  int* err;
};

__global__ __launch_bounds__(p3::NT) void k_push3d(Push3Args a) {
  using namespace p3;
  __shared__ FieldTile3 sf;
  const Grid3D& g = a.g;
  const int ntiles = a.ntx * a.nty * a.ntz;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  int i0, j0, k0;
  tile_origin(g, tile, a.ntx, a.nty, i0, j0, k0);
  const int tid = threadIdx.x;
  stage_fields3(g, a.uf, sf, i0, j0, k0);
  __syncthreads();

  const int grp = tid / G, lg = tid % G;
  constexpr int NGRP = NT / G;
  const double delt = g.delt, c = g.c;
  for (int cc = grp; cc < TX * TY * TZ; cc += NGRP) {
    const int li = cc % TX, lj = (cc / TX) % TY, lk = cc / (TX * TY);
    const int i = i0 + li, j = j0 + lj, k = k0 + lk;
    if (i > g.nxge || j > g.nye || k > g.nze) continue;  // uniform within a group
    const int col = (j - g.nys) + g.ny * (k - g.nzs);
    for (int s = 0; s < g.nsp; s++) {
      const int rw = s * g.ncol + col;
      const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
      const int base = a.colbase[rw];
      const int pbeg = base + cr[i - g.nxgs], pend = base + cr[i - g.nxgs + 1];
      const double q = g.q[s], rm = g.r[s];
      const double fac1 = q / rm * 5e-1 * delt;
      const double txxx = fac1 * fac1;
      const double fac2 = q * delt / rm;
      for (int pi = pbeg + lg; pi < pend; pi += G) {
        const int ia = a.ap ? a.ap[pi] : pi;
        const Rec3 p = load_rec(a.A, ia);
        double nxp, nyp, nzp, g4, g5, g6;
        const int so = (lk + 1) * (SW * SH) + (lj + 1) * SW + (li + 1);
        if (a.vay)
          vay_push3(sf, so, i, j, k, delt, c, fac1, fac2, p.x, p.y, p.z, p.ux, p.uy, p.uz, nxp, nyp, nzp, g4, g5, g6);
        else
          boris_push3(sf, so, i, j, k, delt, c, fac1, txxx, fac2, p.x, p.y, p.z, p.ux, p.uy, p.uz, nxp, nyp, nzp, g4,
                      g5, g6);
        store_rec(a.B, pi, Rec3{nxp, nyp, nzp, g4, g5, g6, p.id});  // particle.f90:227-231
      }
    }
  }
}

// s0 and ds of one particle (field.f90:253-329) for cell (i, j, k):
// v[0..4] s0x, [5..9] s0y, [10..14] s0z, [15..19] dsx, [20..24] dsy, [25..29] dsz
__device__ inline void shapes3(const Grid3D& g, const double old[3], const double nw[3], const int cell[3],
                               double* v) {
  const double d_delx = g.d_delx;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double s0m, s00, s0p;
    shape3(old[d] * d_delx - 5e-1 - cell[d], s0m, s00, s0p);
    const int i2 = (int)(nw[d] * d_delx);
    const double dh = nw[d] * d_delx - 5e-1 - i2;
    const int inc = i2 - cell[d];
    double s1_1, s1_2, s1_3;
    shape3(dh, s1_1, s1_2, s1_3);
    // smo_* = -(inc-abs(inc))*5d-1+0 etc.: whole numbers, never -0
    const double smo_1 = inc < 0 ? (double)(-inc) : 0.0;
    const double smo_2 = (double)(-abs(inc) + 1);
    const double smo_3 = inc > 0 ? (double)inc : 0.0;
    double* s0 = v + 5 * d;
    double* ds = v + 15 + 5 * d;
    s0[0] = 0e0;
    s0[1] = s0m;
    s0[2] = s00;
    s0[3] = s0p;
    s0[4] = 0e0;
    ds[0] = s1_1 * smo_1 - 0e0;
    ds[1] = s1_1 * smo_2 + s1_2 * smo_1 - s0m;
    ds[2] = s1_2 * smo_2 + s1_3 * smo_1 + s1_1 * smo_3 - s00;
    ds[3] = s1_3 * smo_2 + s1_2 * smo_3 - s0p;
    ds[4] = s1_3 * smo_3 - 0e0;
  }
}

template <bool PARITY>
__global__ __launch_bounds__(p3::NT) void k_deposit3d(Push3Args a) {
  using namespace p3;
  __shared__ double shp[NT / 32][NB][NSV];
  __shared__ double acc[PARITY ? 1 : 3][PARITY ? 1 : AN];
  const Grid3D& g = a.g;
  const int ntiles = a.ntx * a.nty * a.ntz;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  int i0, j0, k0;
  tile_origin(g, tile, a.ntx, a.nty, i0, j0, k0);
  const int tid = threadIdx.x;
  if (!PARITY) {
    for (int q = tid; q < 3 * AN; q += NT) (&acc[0][0])[q] = 0.0;
    __syncthreads();
  }
  const int hw = tid >> 5, hl = tid & 31;      // half-wave and its lane
  const int ja = hl % 5, kb = hl / 5;          // this lane's (jp, kp) + 2 when hl < 25
  const bool accl = hl < 25;
  const double fac = 1e0 / 3e0;
  double(*sh)[NSV] = shp[hw];

  for (int cc = hw; cc < TX * TY * TZ; cc += NT / 32) {
    const int li = cc % TX, lj = (cc / TX) % TY, lk = cc / (TX * TY);
    const int i = i0 + li, j = j0 + lj, k = k0 + lk;
    const bool live = i <= g.nxge && j <= g.nye && k <= g.nze;
    const int cell[3] = {i, j, k};
    const int col = (j - g.nys) + g.ny * (k - g.nzs);
    double px[4] = {0, 0, 0, 0}, py[4] = {0, 0, 0, 0}, pz[4] = {0, 0, 0, 0};
    for (int s = 0; s < g.nsp; s++) {
      int pbeg = 0, pend = 0;
      if (live) {
        const int rw = s * g.ncol + col;
        const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
        const int base = a.colbase[rw];
        pbeg = base + cr[i - g.nxgs];
        pend = base + cr[i - g.nxgs + 1];
      }
      const double qdxdt = g.q[s] * g.delx * g.d_delt;
      for (int b0 = pbeg; b0 < pend; b0 += NB) {
        const int nb = pend - b0 < NB ? pend - b0 : NB;
        if (hl < nb) {
          const int pi = b0 + hl;
          const int ia = a.ap ? a.ap[pi] : pi;
          const double old[3] = {a.A.x[ia], a.A.y[ia], a.A.z[ia]};
          const double nw[3] = {a.B.x[pi], a.B.y[pi], a.B.z[pi]};
          double v[NSV];
          shapes3(g, old, nw, cell, v);
          if (!PARITY) {
            // running sums c(m) = -sum_{k<=m} ds(k) of the factored form
#pragma unroll
            for (int d = 0; d < 3; d++) {
              double run = 0.0;
#pragma unroll
              for (int m = 0; m < 4; m++) {
                run -= v[15 + 5 * d + m];
                v[30 + 4 * d + m] = run;
              }
            }
          }
#pragma unroll
          for (int q = 0; q < (PARITY ? 30 : NSV); q++) sh[hl][q] = v[q];
        }
        // the shapes were written by other lanes of this wave
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (accl && !PARITY) {
          // fast mode: pj(m-1, jp, kp) += c(m) * w(jp, kp), the dstmp of the
          // reference written as w = (s0 + ds/2) s0' + (s0/2 + ds/3) ds' (FMA)
          for (int p = 0; p < nb; p++) {
            const double* v = sh[p];
            const double *s0x = v, *s0y = v + 5, *s0z = v + 10, *dsx = v + 15, *dsy = v + 20, *dsz = v + 25;
            const double *cxs = v + 30, *cys = v + 34, *czs = v + 38;
            const double axj = fma(0.5, dsx[ja], s0x[ja]), bxj = fma(fac, dsx[ja], 0.5 * s0x[ja]);
            const double ayj = fma(0.5, dsy[ja], s0y[ja]), byj = fma(fac, dsy[ja], 0.5 * s0y[ja]);
            const double wx = fma(ayj, s0z[kb], byj * dsz[kb]) * qdxdt;
            const double wy = fma(axj, s0z[kb], bxj * dsz[kb]) * qdxdt;
            const double wz = fma(axj, s0y[kb], bxj * dsy[kb]) * qdxdt;
#pragma unroll
            for (int m = 0; m < 4; m++) {
              px[m] = fma(cxs[m], wx, px[m]);
              py[m] = fma(cys[m], wy, py[m]);
              pz[m] = fma(czs[m], wz, pz[m]);
            }
          }
        }
        if (accl && PARITY) {
          for (int p = 0; p < nb; p++) {
            const double* v = sh[p];
            const double *s0x = v, *s0y = v + 5, *s0z = v + 10, *dsx = v + 15, *dsy = v + 20, *dsz = v + 25;
            double dstmp, pjtmp;
            // pjx(:, jp, kp)
            dstmp = ((s0y[ja] + 5e-1 * dsy[ja]) * s0z[kb] + (5e-1 * s0y[ja] + fac * dsy[ja]) * dsz[kb]) * qdxdt;
            pjtmp = -dsx[0] * dstmp;
            px[0] = px[0] + pjtmp;
            pjtmp = pjtmp - dsx[1] * dstmp;
            px[1] = px[1] + pjtmp;
            pjtmp = pjtmp - dsx[2] * dstmp;
            px[2] = px[2] + pjtmp;
            pjtmp = pjtmp - dsx[3] * dstmp;
            px[3] = px[3] + pjtmp;
            // pjy(:, jp, kp)
            dstmp = ((s0x[ja] + 5e-1 * dsx[ja]) * s0z[kb] + (5e-1 * s0x[ja] + fac * dsx[ja]) * dsz[kb]) * qdxdt;
            pjtmp = -dsy[0] * dstmp;
            py[0] = py[0] + pjtmp;
            pjtmp = pjtmp - dsy[1] * dstmp;
            py[1] = py[1] + pjtmp;
            pjtmp = pjtmp - dsy[2] * dstmp;
            py[2] = py[2] + pjtmp;
            pjtmp = pjtmp - dsy[3] * dstmp;
            py[3] = py[3] + pjtmp;
            // pjz(:, jp, kp)
            dstmp = ((s0x[ja] + 5e-1 * dsx[ja]) * s0y[kb] + (5e-1 * s0x[ja] + fac * dsx[ja]) * dsy[kb]) * qdxdt;
            pjtmp = -dsz[0] * dstmp;
            pz[0] = pz[0] + pjtmp;
            pjtmp = pjtmp - dsz[1] * dstmp;
            pz[1] = pz[1] + pjtmp;
            pjtmp = pjtmp - dsz[2] * dstmp;
            pz[2] = pz[2] + pjtmp;
            pjtmp = pjtmp - dsz[3] * dstmp;
            pz[3] = pz[3] + pjtmp;
          }
        }
        // before the next batch overwrites the shapes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
    if (!live || !accl) continue;
    if (PARITY) {
      double* b = a.pjbuf + cidx3(g, i, j, k) * 300 + hl * 4;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        b[m] = px[m];
        b[100 + m] = py[m];
        b[200 + m] = pz[m];
      }
    } else {
      // pjx(m-1, jp, kp) -> node (i+m-1, j+jp, k+kp); pjy -> (i+jp, j+m-1, k+kp);
      // pjz -> (i+jp, j+kp, k+m-1), with jp = ja-2, kp = kb-2
      const int bx = (li + 2), by = (lj + 2), bz = (lk + 2);
#pragma unroll
      for (int m = 0; m < 4; m++) {
        atomicAdd(&acc[0][((bz + kb - 2) * AH + (by + ja - 2)) * AW + (bx + m - 1)], px[m]);
        atomicAdd(&acc[1][((bz + kb - 2) * AH + (by + m - 1)) * AW + (bx + ja - 2)], py[m]);
        atomicAdd(&acc[2][((bz + m - 1) * AH + (by + kb - 2)) * AW + (bx + ja - 2)], pz[m]);
      }
    }
  }
  if (!PARITY) {
    __syncthreads();
    const size_t pl = plane3(g);
    for (int q = tid; q < 3 * AN; q += NT) {
      const int comp = q / AN, rem = q - comp * AN;
      const double v = acc[comp][rem];
      if (v == 0.0) continue;
      const int I = i0 - 2 + rem % AW, J = j0 - 2 + (rem / AW) % AH, K = k0 - 2 + rem / (AW * AH);
      if (I > g.nxge + 2 || J > g.nye + 2 || K > g.nze + 2) continue;
      unsafeAtomicAdd(a.uj + pl * comp + fidx3(g, I, J, K), v);
    }
  }
}

// uj(c, I, J, K) = sum over source cells in the reference's (k, j, i) order of
// their block entry, from +0 (field.f90:231-403 at one thread).  pjx(-2,.,.),
// pjy(-2,.,.) and pjz(-2,.,.) are structurally +0 and are skipped.
__global__ __launch_bounds__(256) void k_gather_pj3d(Grid3D g, const double* __restrict__ pjbuf,
                                                    double* __restrict__ uj) {
  const size_t n = plane3(g);
  const size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int I = g.nxgs - 2 + (int)(q % g.fw), J = g.nys - 2 + (int)((q / g.fw) % g.fh),
            K = g.nzs - 2 + (int)(q / ((size_t)g.fw * g.fh));
  double sx = 0.0, sy = 0.0, sz = 0.0;
  const int klo = K - 2 > g.nzs ? K - 2 : g.nzs, khi = K + 2 < g.nze ? K + 2 : g.nze;
  const int jlo = J - 2 > g.nys ? J - 2 : g.nys, jhi = J + 2 < g.nye ? J + 2 : g.nye;
  const int ilo = I - 2 > g.nxgs ? I - 2 : g.nxgs, ihi = I + 2 < g.nxge ? I + 2 : g.nxge;
  for (int k = klo; k <= khi; k++)
    for (int j = jlo; j <= jhi; j++)
      for (int i = ilo; i <= ihi; i++) {
        const int ox = I - i, oy = J - j, oz = K - k;
        const double* b = pjbuf + cidx3(g, i, j, k) * 300;
        // lane (ja, kb) = (a + 2, b + 2) holds pj(m - 1, a, b) at [lane*4 + m]
        if (ox >= -1) sx = sx + b[((oz + 2) * 5 + (oy + 2)) * 4 + ox + 1];
        if (oy >= -1) sy = sy + b[100 + ((oz + 2) * 5 + (ox + 2)) * 4 + oy + 1];
        if (oz >= -1) sz = sz + b[200 + ((oy + 2) * 5 + (ox + 2)) * 4 + oz + 1];
      }
  uj[q] = sx;
  uj[n + q] = sy;
  uj[2 * n + q] = sz;
}

// Current of one particle that changes cell, in the factored form of
// k_push_deposit3d_fast, from its old and new in-cell shape arguments
// (x - 0.5 - cell per axis, field.f90:253-266) and its cell increments, added
// to the LDS tile: o is the tile's Jx at the particle's cell.  The 4-node
// window [lo, lo + 3] of the 5 nodes -2..2 per axis, lo = 0 for a step to the
// left and 1 otherwise, holds every non-zero s0 and ds; the new shape carries
// the reference's weights there, |inc| moved by one node and 1 - |inc| unmoved
// (a plain shift for a step of one cell; a particle near c may round across two
// faces in x).  An axis along which the particle keeps its cell has nothing on
// its fourth node and only rounding on its third face, so a step along one axis
// costs 75 atomics and one along all three 144.
__device__ inline void deposit3_window(double* o, const double dh0[3], const double dh1[3], const int inc[3],
                                       double qd) {
  using namespace p3;
  constexpr int SY = AW, SZ = AW * AH;
  double S[3][4], D[3][4], cq[3][3];
  bool mv[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double t0, t1, t2, u0, u1, u2;
    shape3(dh0[d], t0, t1, t2);
    shape3(dh1[d], u0, u1, u2);
    const bool left = inc[d] < 0;
    mv[d] = inc[d] != 0;
    const double far = (double)abs(inc[d]), near = 1.0 - far;
    const double p = left ? far : near, q = left ? near : far;
    o += (left ? -2 : -1) * (d == 0 ? 1 : (d == 1 ? SY : SZ));  // window node 0 of the axis
    S[d][0] = left ? 0.0 : t0;
    S[d][1] = left ? t0 : t1;
    S[d][2] = left ? t1 : t2;
    S[d][3] = left ? t2 : 0.0;
    D[d][0] = p * u0 - S[d][0];
    D[d][1] = p * u1 + q * u0 - S[d][1];
    D[d][2] = p * u2 + q * u1 - S[d][2];
    D[d][3] = q * u2 - S[d][3];
    double run = 0.0;
#pragma unroll
    for (int m = 0; m < 3; m++) {
      run = run - D[d][m];
      cq[d][m] = run * qd;
    }
  }
  // face m lies between window nodes m and m + 1, at the offset of node m + 1
  // (the barriers keep the compiler from forming all the products first)
#pragma unroll
  for (int v = 0; v < 4; v++) {  // z node
    if (v == 3 && !mv[2]) break;
    const double Sz = S[2][v], Dz = D[2][v], az = fma(0.5, Dz, Sz), bz = fma(1.0 / 3.0, Dz, 0.5 * Sz);
    double* const r = o + v * SZ;
#pragma unroll
    for (int u = 0; u < 4; u++) {  // y node of Jx
      if (u == 3 && !mv[1]) break;
      const double w = fma(S[1][u], az, D[1][u] * bz);
      atomicAdd(r + u * SY + 1, cq[0][0] * w);
      atomicAdd(r + u * SY + 2, cq[0][1] * w);
      if (mv[0]) atomicAdd(r + u * SY + 3, cq[0][2] * w);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {  // x node of Jy
      if (u == 3 && !mv[0]) break;
      const double w = fma(S[0][u], az, D[0][u] * bz);
      atomicAdd(r + AN + u + SY, cq[1][0] * w);
      atomicAdd(r + AN + u + 2 * SY, cq[1][1] * w);
      if (mv[1]) atomicAdd(r + AN + u + 3 * SY, cq[1][2] * w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; v++) {  // y node of Jz
    if (v == 3 && !mv[1]) break;
    const double Sy = S[1][v], Dy = D[1][v], ay = fma(0.5, Dy, Sy), by = fma(1.0 / 3.0, Dy, 0.5 * Sy);
#pragma unroll
    for (int u = 0; u < 4; u++) {  // x node
      if (u == 3 && !mv[0]) break;
      const double w = fma(S[0][u], ay, D[0][u] * by);
      double* const r = o + 2 * AN + v * SY + u;
      atomicAdd(r + SZ, cq[2][0] * w);
      atomicAdd(r + 2 * SZ, cq[2][1] * w);
      if (mv[2]) atomicAdd(r + 3 * SZ, cq[2][2] * w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Fast mode, push and deposit in one kernel.  The push is the shared bit-exact
// boris_push3; the deposit uses the factored weights of k_deposit3d's fast path,
//   Jx(m, j, k) += cx(m) (s0y(j) az(k) + dsy(j) bz(k)),  cx(m) = -sum_{n<=m} dsx(n),
//   az = s0z + dsz/2,  bz = s0z/2 + dsz/3,
// and Jy, Jz with the axes permuted (field.f90:335-380 expanded term by term).
// A particle that stays in its cell along every axis has ds = 0 on the outer
// nodes and cx = 0 on the outer faces (the last one up to rounding), so its
// current lives on 2 x 3 x 3 nodes per component: every lane sums those 54
// values over the particles it handles and the lane group adds them up.  A
// particle that changes cell is queued in its wave's LDS queue; whenever 64
// have gathered, over as many passes and cells as that takes, all the wave's
// lanes add one particle's window each (deposit3_window) to the LDS tile.  The
// tile is added to uj with one HBM atomic per node.
//
// Work mapping: wave w walks row w of each of the tile's four layers, 8 cells
// of 8 lanes, each lane every eighth particle of its cell (all species as one
// list) with the two-deep load pipeline of the 2D kernel.  Up to KP passes
// push and leave their particles' six shape arguments in registers, then the
// 54 sums are formed from those: kept over the pushes themselves, next to the
// gather's 16-byte reads in flight, the sums spilled (10.0 ms, half of it
// scratch traffic).
//
// What bounds it (160x144x128, 2 species of 16 ppc, 94 M particles): VALU
// issue in 71 % of the cycles at 2 waves a SIMD; 12.9 GB of traffic (11.3
// algorithmic) in 6.1 ms.  One pass with the sums kept, one array per field,
// single LDS reads and per-round queues took 8.2 ms.  KP = 3, 4, 5, 6: 6.2,
// 6.2, 6.1, 6.2 ms.
namespace p3f {
constexpr int G = 8;     // lanes per cell
constexpr int KP = 5;    // passes between two deposits of what stays
constexpr int QW = 128;  // queued cell-changing particles per wave: 63 left over and 64 of a pass at most
}  // namespace p3f

template <bool VAY>
__global__ __launch_bounds__(p3::NT, 2) void k_push_deposit3d_fast(Push3Args a) {
  using namespace p3;
  constexpr int GF = p3f::G, NW = NT / 64;
  using p3f::QW;
  using p3f::KP;
  static_assert(64 / GF == TX && NW == TY, "a wave takes a row of the tile at a time");
  __shared__ FieldTile3 sf;
  __shared__ double acc[3][AN];
  __shared__ double spc[WPIC_MAXSP][4];  // fac1, txxx, fac2, q delx / delt
  // the waves' queued particles: old and new shape arguments per axis, and
  // cell in the tile | species << 7 | (inc + 4) per axis << 9, 12, 15
  __shared__ double xqd[NW][6][QW];
  __shared__ int xqc[NW][QW];
  const Grid3D& g = a.g;
  const int ntiles = a.ntx * a.nty * a.ntz;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  int i0, j0, k0;
  tile_origin(g, tile, a.ntx, a.nty, i0, j0, k0);
  const int tid = threadIdx.x;
  stage_fields3(g, a.uf, sf, i0, j0, k0);
  for (int q = tid; q < 3 * AN; q += NT) (&acc[0][0])[q] = 0.0;
#pragma unroll
  for (int s = 0; s < WPIC_MAXSP; s++) {
    if (tid == s && s < g.nsp) {
      const double q = g.q[s], rm = g.r[s];
      const double fac1 = q / rm * 5e-1 * g.delt;
      spc[s][0] = fac1;
      spc[s][1] = fac1 * fac1;
      spc[s][2] = q * g.delt / rm;
      spc[s][3] = q * g.delx * g.d_delt;
    }
  }
  __syncthreads();

  // (the wave's number, the same in its lanes, and with it j and k stay in
  // scalar registers)
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lg = lane % GF;
  const int li = lane / GF, lj = w;
  const int i = i0 + li, j = j0 + lj;
  int nq = 0;  // queued particles, the same in all lanes

  // the currents of the last (at most 64) queued particles
  auto drain = [&]() {
    // written by this wave's own lanes: LDS operations of one wave complete in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int n0 = nq > 64 ? nq - 64 : 0, q = n0 + lane;
    if (q < nq) {
      const int e = xqc[w][q];
      const int cc = e & 127, s = (e >> 7) & 3;
      const int inc[3] = {((e >> 9) & 7) - 4, ((e >> 12) & 7) - 4, ((e >> 15) & 7) - 4};
      const double dh0[3] = {xqd[w][0][q], xqd[w][1][q], xqd[w][2][q]};
      const double dh1[3] = {xqd[w][3][q], xqd[w][4][q], xqd[w][5][q]};
      deposit3_window(&acc[0][((cc / (TX * TY) + 2) * AH + (cc / TX % TY + 2)) * AW + (cc % TX + 2)], dh0, dh1, inc,
                      spc[s][3]);
    }
    nq = n0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  for (int lk = 0; lk < TZ; lk++) {
    const int k = k0 + lk;
    const bool live = i <= g.nxge && j <= g.nye && k <= g.nze;  // uniform within a group
    CellList cl;
    int tot = 0;
#pragma unroll
    for (int s = 0; s < WPIC_MAXSP; s++) {
      if (s < g.nsp) {
        int c0 = 0, c1 = 0, cb = 0;
        if (live) {
          const int rw = s * g.ncol + (j - g.nys) + g.ny * (k - g.nzs);
          const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1) + (i - g.nxgs);
          c0 = cr[0];
          c1 = cr[1];
          cb = a.colbase[rw];
        }
        cl.set(s, cb + c0, tot);
        tot += c1 - c0;
      } else {
        cl.set(s, 0, 0x7fffffff);
      }
    }
    const int so = (lk + 1) * (SW * SH) + (lj + 1) * SW + (li + 1);

    int ia_nn = 0;
    // (a cell's surplus lanes push a particle at rest at its centre)
    Rec3 pr = {i + 0.5, j + 0.5, k + 0.5, 0.0, 0.0, 0.0, 0};
    {
      int s_, p_, ia_n = 0;
      if (lg < tot) {
        cl.slot(g.nsp, lg, s_, p_);
        ia_n = a.ap ? a.ap[p_] : p_;
      }
      if (lg + GF < tot) {
        cl.slot(g.nsp, lg + GF, s_, p_);
        ia_nn = a.ap ? a.ap[p_] : p_;
      }
      if (lg < tot) pr = load_rec(a.A, ia_n);
    }
    // KP passes at a time: the pushes, one straight line for all lanes as in 2D
    // (a lane past its cell's last particle repeats one with zero charge and
    // stores nothing), then the current of those that stay
    int t = lg;
    while (__any(t < tot)) {
    double pd[KP][6];  // old and new shape arguments of the last KP passes, the latest first
    int ps[KP];    // species, or -1: no current from it
#pragma unroll
    for (int h = 0; h < KP; h++) {
      ps[h] = -1;
#pragma unroll
      for (int d = 0; d < 6; d++) pd[h][d] = 0.0;
    }
    for (int h = 0; h < KP && __any(t < tot); h++, t += GF) {
      const bool act = t < tot;
      int s, pi;
      cl.slot(g.nsp, t, s, pi);
      const Rec3 cur = pr;
      if (t + GF < tot) pr = load_rec(a.A, ia_nn);
      if (t + 2 * GF < tot) {
        int s_, p_;
        cl.slot(g.nsp, t + 2 * GF, s_, p_);
        ia_nn = a.ap ? a.ap[p_] : p_;
      }
      const double* kc = spc[s];
      const double x = cur.x, y = cur.y, z = cur.z;
      double nxp, nyp, nzp, g4, g5, g6;
      if (VAY)
        vay_push3(sf, so, i, j, k, g.delt, g.c, kc[0], kc[2], x, y, z, cur.ux, cur.uy, cur.uz, nxp, nyp, nzp, g4, g5,
                  g6);
      else
        boris_push3(sf, so, i, j, k, g.delt, g.c, kc[0], kc[1], kc[2], x, y, z, cur.ux, cur.uy, cur.uz, nxp, nyp, nzp,
                    g4, g5, g6);
      const int i2 = (int)nxp, j2 = (int)nyp, k2 = (int)nzp;
      const bool stays = i2 == i && j2 == j && k2 == k;
      const bool mover = act && !stays;
      if (act) {
        // the x wrap, the y-z wraps and the exchange code: particle_x and
        // particle_yz act on gp after the deposit, which uses the unwrapped
        // position
        double wx = nxp, wy = nyp, wz = nzp;
        int code = ((i2 - g.nxgs) << CODE_SHIFT3) | ((k2 - k + 1) * 3 + (j2 - j + 1));
        if ((unsigned)(i2 - g.nxgs) >= (unsigned)g.nx || (unsigned)(j2 - g.nys) >= (unsigned)g.ny ||
            (unsigned)(k2 - g.nzs) >= (unsigned)g.nz || (unsigned)(j2 - j + 1) > 2u || (unsigned)(k2 - k + 1) > 2u) {
          bool moved;
          code = wrap3_code<true>(g, wx, wy, wz, j, k, a.err, moved);
        }
        a.code[pi] = code;
        store_rec(a.B, pi, Rec3{wx, wy, wz, g4, g5, g6, cur.id});
      }
#pragma unroll
      for (int q = KP - 1; q > 0; q--) {
        ps[q] = ps[q - 1];
#pragma unroll
        for (int d = 0; d < 6; d++) pd[q][d] = pd[q - 1][d];
      }
      ps[0] = act && stays ? s : -1;
      pd[0][0] = x - 5e-1 - i;
      pd[0][1] = y - 5e-1 - j;
      pd[0][2] = z - 5e-1 - k;
      pd[0][3] = nxp - 5e-1 - i2;
      pd[0][4] = nyp - 5e-1 - j2;
      pd[0][5] = nzp - 5e-1 - k2;
      const uint64_t mm = __ballot(mover);
      if (mm) {
        if (mover) {
          const int slot = nq + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mm >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mm, 0));
#pragma unroll
          for (int d = 0; d < 6; d++) xqd[w][d][slot] = pd[0][d];
          xqc[w][slot] = ((lk * TY + lj) * TX + li) | (s << 7) | (((i2 - i + 4) & 7) << 9) |
                         (((j2 - j + 4) & 7) << 12) | (((k2 - k + 4) & 7) << 15);
        }
        nq += __popcll(mm);
        if (nq >= 64) drain();
      }
    }
    // the current of the particles that stay: sum 18 c + 9 m + 3 u + b of
    // component c, face m along its own axis, nodes u - 1, b - 1 of the other
    // two in the order x, y, z
    double v[54];
#pragma unroll
    for (int q = 0; q < 54; q++) v[q] = 0.0;
#pragma unroll
    for (int h = 0; h < KP; h++) {
      if (!__any(ps[h] >= 0)) continue;
      const double qd = ps[h] >= 0 ? spc[ps[h] & 3][3] : 0.0;
      double S[3][3], D[3][3], cq[3][2];  // s0, ds = s1 - s0, -sum ds
#pragma unroll
      for (int d = 0; d < 3; d++) {
        double t0, t1, t2;
        shape3(pd[h][d], S[d][0], S[d][1], S[d][2]);
        shape3(pd[h][3 + d], t0, t1, t2);
        D[d][0] = t0 - S[d][0];
        D[d][1] = t1 - S[d][1];
        D[d][2] = t2 - S[d][2];
        cq[d][0] = (0.0 - D[d][0]) * qd;
        cq[d][1] = ((0.0 - D[d][0]) - D[d][1]) * qd;
      }
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const double az = fma(0.5, D[2][b], S[2][b]), bz = fma(1.0 / 3.0, D[2][b], 0.5 * S[2][b]);
        const double ay = fma(0.5, D[1][b], S[1][b]), by = fma(1.0 / 3.0, D[1][b], 0.5 * S[1][b]);
#pragma unroll
        for (int u = 0; u < 3; u++) {
          const double wx = fma(S[1][u], az, D[1][u] * bz);  // y node u, z node b
          const double wy = fma(S[0][u], az, D[0][u] * bz);  // x node u, z node b
          const double wz = fma(S[0][u], ay, D[0][u] * by);  // x node u, y node b
#pragma unroll
          for (int m = 0; m < 2; m++) {
            const int q = 9 * m + 3 * u + b;
            v[q] = fma(cq[0][m], wx, v[q]);
            v[18 + q] = fma(cq[1][m], wy, v[18 + q]);
            v[36 + q] = fma(cq[2][m], wz, v[36 + q]);
          }
        }
      }
    }
    // over the group, spread over its lanes (a cell without particles adds
    // nothing: its fields may be any, and 0 * NaN is not 0)
    group_reduce<54, GF>(v, lane);
    // (the places are worked out here: kept over the passes they would spill)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    double* const o = &acc[0][0] + ((lk + 2) * AH + (lj + 2)) * AW + (li + 2);
#pragma unroll
    for (int f = 0; f < group_left(54, GF); f++) {
      const int q = group_index<54, GF>(f, ln);
      const int c = q / 18, m = q % 18 / 9, u = q % 9 / 3 - 1, b = q % 3 - 1;
      const int xo = c == 0 ? m : u, yo = c == 0 ? u : (c == 1 ? m : b), zo = c == 2 ? m : b;
      if (tot > 0 && q >= 0 && v[f] != 0.0) atomicAdd(o + (c * AN + (zo * AH + yo) * AW + xo), v[f]);
    }
    }
  }
  if (nq) drain();
  __syncthreads();
  const size_t pl = plane3(g);
  for (int q = tid; q < 3 * AN; q += NT) {
    const int comp = q / AN, rem = q - comp * AN;
    const double v = acc[comp][rem];
    if (v == 0.0) continue;
    const int I = i0 - 2 + rem % AW, J = j0 - 2 + (rem / AW) % AH, K = k0 - 2 + rem / (AW * AH);
    if (I > g.nxge + 2 || J > g.nye + 2 || K > g.nze + 2) continue;
    unsafeAtomicAdd(a.uj + pl * comp + fidx3(g, I, J, K), v);
  }
}

static Push3Args push_args(wpic_ctx3d* c) {
  Push3Args a;
  a.g = c->g;
  a.A = c->A;
  a.B = c->B;
  a.colbase = c->colbaseA;
  a.cumcnt = c->cumcnt;
  a.ap = c->aperm;
  a.uf = c->uf;
  a.uj = c->uj;
  a.pjbuf = c->pjbuf;
  a.ntx = (c->g.nx + p3::TX - 1) / p3::TX;
  a.nty = (c->g.ny + p3::TY - 1) / p3::TY;
  a.ntz = (c->g.nz + p3::TZ - 1) / p3::TZ;
  a.vay = c->pusher == WPIC_PUSHER_VAY;
  a.code = c->code;
  a.err = c->err;
  return a;
}

hipError_t launch_push3d(wpic_ctx3d* c) {
  Push3Args a = push_args(c);
  const int nblk = xcd_grid(a.ntx * a.nty * a.ntz);
  hipLaunchKernelGGL(k_push3d, dim3(nblk), dim3(p3::NT), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_deposit3d(wpic_ctx3d* c) {
  Push3Args a = push_args(c);
  const int nblk = xcd_grid(a.ntx * a.nty * a.ntz);
  if (c->mode == WPIC_MODE_PARITY)
    hipLaunchKernelGGL(k_deposit3d<true>, dim3(nblk), dim3(p3::NT), 0, c->st, a);
  else
    hipLaunchKernelGGL(k_deposit3d<false>, dim3(nblk), dim3(p3::NT), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_push_deposit3d(wpic_ctx3d* c) {
  Push3Args a = push_args(c);
  const int nblk = xcd_grid(a.ntx * a.nty * a.ntz);
  if (a.vay)
    hipLaunchKernelGGL(k_push_deposit3d_fast<true>, dim3(nblk), dim3(p3::NT), 0, c->st, a);
  else
    hipLaunchKernelGGL(k_push_deposit3d_fast<false>, dim3(nblk), dim3(p3::NT), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_gather_pj3d(wpic_ctx3d* c) {
  const size_t n = plane3(c->g);
  hipLaunchKernelGGL(k_gather_pj3d, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->st, c->g, c->pjbuf, c->uj);
  return hipGetLastError();
}

}  // namespace wpic
