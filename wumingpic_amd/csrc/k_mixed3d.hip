// k_mixed3d.hip -- the mixed-precision form of the 3D fused push + deposit +
// x wrap (the physics of 3d/common/particle.f90:52-233 and
// 3d/common/field.f90:211-406 followed by the particle boundaries).
//
// A particle is an int32 x cell plus FP32 offsets (x - ix, y - j, z - k) in
// [0, 1) and FP32 momenta, 36 B with the id: positions keep ~1e-7 of a cell
// everywhere in the box and the shape functions see offsets directly.  Push
// and deposit run in FP32 (FMA contraction on); each particle's current is
// formed in FP32 and accumulated in an FP64 LDS tile, the tile is added to
// the FP64 uj with FP64 atomics and the field solve is the FP64 one.  The work mapping is the FP64
// fused kernel's (k_push_deposit3d_fast): 8x4x4-cell tiles, 8 lanes per cell,
// the 54 current values of a particle that stays in its cell in registers, a
// particle that changes cell queued (per wave) with its offsets and added with
// its window when 64 have gathered.  The push writes the exchange code
// ((new x cell - nxgs) << 4 | y-z direction) itself: the x wrap is a cell
// wrap and the y-z offsets are already relative to the destination column.
#include "wpic_internal3d.h"

namespace wpic {
// the tile accumulates in FP64: LDS FP32 atomics serialize badly when the
// lanes of a wave add to the same node, FP64 ones do not
__device__ inline void tile_add(double* p, float v) { atomicAdd(p, (double)v); }

namespace m3 {
constexpr int TX = 8, TY = 4, TZ = 4, NT = 256, G = 8;
constexpr int SW = TX + 2, SH = TY + 2, SD = TZ + 2, SN = SW * SH * SD;  // staged tmpf
constexpr int AW = TX + 4, AH = TY + 4, AD = TZ + 4, AN = AW * AH * AD;  // current tile
constexpr int KP = 5;    // passes between two deposits of what stays
constexpr int QW = 128;  // queued cell-changing particles per wave: 63 left over and 64 of a pass at most
}  // namespace m3

struct Mix3Args {
  Grid3D g;
  PartsM3 A, B;
  const int* colbase;
  const int* cumcnt;
  const int* ap;  // A's slot -> record (null: identity)
  const double* uf;
  double* uj;
  int* code;
  int* err;
  int ntx, nty, ntz;
};

// tmpf(c, i, j, k) of particle.f90:74-91 in FP64, rounded to FP32 by the caller
__device__ inline double tmpf3m(const Grid3D& g, const double* uf, int c, int i, int j, int k) {
  const size_t pl = plane3(g);
  const double* u = uf + pl * c;
  const size_t o = fidx3(g, i, j, k);
  const size_t dx = 1, dy = (size_t)g.fw, dz = (size_t)g.fw * g.fh;
  switch (c) {
    case 0: return 0.25 * (u[o] + u[o + dy] + u[o + dz] + u[o + dy + dz]);
    case 1: return 0.25 * (u[o] + u[o + dx] + u[o + dz] + u[o + dx + dz]);
    case 2: return 0.25 * (u[o] + u[o + dx] + u[o + dy] + u[o + dx + dy]);
    case 3: return 0.5 * (u[o] + u[o + dx]);
    case 4: return 0.5 * (u[o] + u[o + dy]);
    default: return 0.5 * (u[o] + u[o + dz]);
  }
}

__device__ inline void shape3m(float dh, float& s0, float& s1, float& s2) {
  s0 = 0.5f * (0.5f - dh) * (0.5f - dh);
  s1 = 0.75f - dh * dh;
  s2 = 0.5f * (0.5f + dh) * (0.5f + dh);
}

// the staged fields of a cell: (Bx, By, Bz, Ex) in one 16-byte LDS read and
// (Ey, Ez) in one of 8
struct alignas(16) Field4M {
  float v[4];
};
struct alignas(8) Field2M {
  float v[2];
};

struct Mix3Const {
  float delt, ic2, cc2;  // dt, 1/c^2, c^2
};

// The push of one particle in FP32 (particle.f90:93-217 in the cell + offset
// form): old shape sh (x, y, z triplets), new offsets f and cell increments inc.
struct Mix3Push {
  float sh[9];
  float f[3];
  int inc[3];
  float g4, g5, g6, gmv;
};

__device__ inline Mix3Push mixed_push3(const Mix3Const& mc, const Field4M* fa, const Field2M* fb, int so,
                                       const float* kc, const RecM3& p) {
#pragma clang fp contract(fast)
  using namespace m3;
  const float fac1 = kc[0], txxx = kc[1], fac2 = kc[2];
  const float ux = p.ux, uy = p.uy, uz = p.uz;
  Mix3Push r;
  // the gather: nine rows of three cells, the next two rows' reads in flight
  // while one is combined
  constexpr int AHEAD = 2;
  int off = so - SW * SH - SW - 1;  // the cell's lowest neighbour
  asm volatile("" : "+v"(off));
  Field4M va[AHEAD + 1][3];
  Field2M vb[AHEAD + 1][3];
  auto load = [&](int q) {
#pragma unroll
    for (int e = 0; e < 3; e++) {
      const int o = off + (q / 3) * (SW * SH) + (q % 3) * SW + e;
      va[q % (AHEAD + 1)][e] = fa[o];
      vb[q % (AHEAD + 1)][e] = fb[o];
    }
  };
#pragma unroll
  for (int q = 0; q < AHEAD; q++) load(q);
  __builtin_amdgcn_sched_barrier(0);
  shape3m(p.ox - 0.5f, r.sh[0], r.sh[1], r.sh[2]);
  shape3m(p.oy - 0.5f, r.sh[3], r.sh[4], r.sh[5]);
  shape3m(p.oz - 0.5f, r.sh[6], r.sh[7], r.sh[8]);
  float fl[6], ya[6];
#pragma unroll
  for (int q = 0; q < 9; q++) {
    if (q + AHEAD < 9) load(q + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
    const Field4M* A = va[q % (AHEAD + 1)];
    const Field2M* B = vb[q % (AHEAD + 1)];
    const int n = q % 3, m = q / 3;
#pragma unroll
    for (int c = 0; c < 6; c++) {
      const float t = c < 4 ? A[0].v[c & 3] * r.sh[0] + A[1].v[c & 3] * r.sh[1] + A[2].v[c & 3] * r.sh[2]
                            : B[0].v[c & 1] * r.sh[0] + B[1].v[c & 1] * r.sh[1] + B[2].v[c & 1] * r.sh[2];
      ya[c] = n == 0 ? t * r.sh[3] : ya[c] + t * r.sh[3 + n];
      if (n == 2) fl[c] = m == 0 ? ya[c] * r.sh[6] : fl[c] + ya[c] * r.sh[6 + m];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // (combined here, not where a later block uses them)
  asm volatile("" : "+v"(fl[0]), "+v"(fl[1]), "+v"(fl[2]), "+v"(fl[3]), "+v"(fl[4]), "+v"(fl[5]));
  const float bpx = fl[0], bpy = fl[1], bpz = fl[2], epx = fl[3], epy = fl[4], epz = fl[5];
  float uvm1 = ux + fac1 * epx;
  float uvm2 = uy + fac1 * epy;
  float uvm3 = uz + fac1 * epz;
  const float gam = sqrtf(mc.cc2 + uvm1 * uvm1 + uvm2 * uvm2 + uvm3 * uvm3);
  const float igam = 1.0f / gam;
  const float fac1r = fac1 * igam;
  const float fac2r = fac2 / (gam + txxx * (bpx * bpx + bpy * bpy + bpz * bpz) * igam);
  const float uvm4 = uvm1 + fac1r * (uvm2 * bpz - uvm3 * bpy);
  const float uvm5 = uvm2 + fac1r * (uvm3 * bpx - uvm1 * bpz);
  const float uvm6 = uvm3 + fac1r * (uvm1 * bpy - uvm2 * bpx);
  uvm1 = uvm1 + fac2r * (uvm5 * bpz - uvm6 * bpy);
  uvm2 = uvm2 + fac2r * (uvm6 * bpx - uvm4 * bpz);
  uvm3 = uvm3 + fac2r * (uvm4 * bpy - uvm5 * bpx);
  r.g4 = uvm1 + fac1 * epx;
  r.g5 = uvm2 + fac1 * epy;
  r.g6 = uvm3 + fac1 * epz;
  r.gmv = 1.0f / sqrtf(1.0f + (r.g4 * r.g4 + r.g5 * r.g5 + r.g6 * r.g6) * mc.ic2);
  const float o[3] = {p.ox, p.oy, p.oz}, u[3] = {r.g4, r.g5, r.g6};
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const float np = o[d] + u[d] * mc.delt * r.gmv;
    const float fi = floorf(np);
    r.inc[d] = (int)fi;
    r.f[d] = np - fi;
    if (r.f[d] >= 1.0f) {
      r.f[d] -= 1.0f;
      r.inc[d] += 1;
    }
  }
  return r;
}

// Current of one particle that changes cell, added to the FP64 tile with the
// window of k_push_deposit3d_fast (|inc| <= 1; a longer step is reported): o is
// the tile's Jx at the particle's cell.
__device__ inline void deposit3_window_m(double* o, const float dh0[3], const float dh1[3], const int inc[3],
                                         float qd) {
#pragma clang fp contract(fast)
  using namespace m3;
  constexpr int SY = AW, SZ = AW * AH;
  float S[3][4], D[3][4], cq[3][3];
  bool mv[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    float t0, t1, t2, u0, u1, u2;
    shape3m(dh0[d], t0, t1, t2);
    shape3m(dh1[d], u0, u1, u2);
    const bool left = inc[d] < 0, right = inc[d] > 0;
    mv[d] = left || right;
    o += (left ? -2 : -1) * (d == 0 ? 1 : (d == 1 ? SY : SZ));  // window node 0 of the axis
    S[d][0] = left ? 0.0f : t0;
    S[d][1] = left ? t0 : t1;
    S[d][2] = left ? t1 : t2;
    S[d][3] = left ? t2 : 0.0f;
    D[d][0] = (right ? 0.0f : u0) - S[d][0];
    D[d][1] = (right ? u0 : u1) - S[d][1];
    D[d][2] = (right ? u1 : u2) - S[d][2];
    D[d][3] = (right ? u2 : 0.0f) - S[d][3];
    float run = 0.0f;
#pragma unroll
    for (int m = 0; m < 3; m++) {
      run -= D[d][m];
      cq[d][m] = run * qd;
    }
  }
  // face m lies between window nodes m and m + 1, at the offset of node m + 1
#pragma unroll
  for (int v = 0; v < 4; v++) {  // z node
    if (v == 3 && !mv[2]) break;
    const float Sz = S[2][v], Dz = D[2][v], az = Sz + 0.5f * Dz, bz = 0.5f * Sz + (1.0f / 3.0f) * Dz;
    double* const r = o + v * SZ;
#pragma unroll
    for (int u = 0; u < 4; u++) {  // y node of Jx
      if (u == 3 && !mv[1]) break;
      const float w = S[1][u] * az + D[1][u] * bz;
      tile_add(r + u * SY + 1, cq[0][0] * w);
      tile_add(r + u * SY + 2, cq[0][1] * w);
      if (mv[0]) tile_add(r + u * SY + 3, cq[0][2] * w);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {  // x node of Jy
      if (u == 3 && !mv[0]) break;
      const float w = S[0][u] * az + D[0][u] * bz;
      tile_add(r + AN + u + SY, cq[1][0] * w);
      tile_add(r + AN + u + 2 * SY, cq[1][1] * w);
      if (mv[1]) tile_add(r + AN + u + 3 * SY, cq[1][2] * w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; v++) {  // y node of Jz
    if (v == 3 && !mv[1]) break;
    const float Sy = S[1][v], Dy = D[1][v], ay = Sy + 0.5f * Dy, by = 0.5f * Sy + (1.0f / 3.0f) * Dy;
#pragma unroll
    for (int u = 0; u < 4; u++) {  // x node
      if (u == 3 && !mv[0]) break;
      const float w = S[0][u] * ay + D[0][u] * by;
      double* const r = o + 2 * AN + v * SY + u;
      tile_add(r + SZ, cq[2][0] * w);
      tile_add(r + 2 * SZ, cq[2][1] * w);
      if (mv[2]) tile_add(r + 3 * SZ, cq[2][2] * w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

__device__ inline void tile_origin_m(const Grid3D& g, int tile, int ntx, int nty, int& i0, int& j0, int& k0) {
  const int tx = tile % ntx, rest = tile / ntx;
  i0 = g.nxgs + tx * m3::TX;
  j0 = g.nys + (rest % nty) * m3::TY;
  k0 = g.nzs + (rest / nty) * m3::TZ;
}

// Its structure is that of k_push_deposit3d_fast.  What bounds it (256^3, 2
// species of 16 ppc, 537 M particles): VALU issue, 85 % of the SIMD cycles at 3
// waves; 53 GB of traffic (43 algorithmic) in 20.3 ms.  One pass with the sums
// kept, one array per field, single LDS reads and per-round queues took 28.5.
// KP = 3, 4, 5, 6: 22.0, 21.4, 20.4, 20.4 ms.
__global__ __launch_bounds__(m3::NT, 3) void k_push_deposit_mixed3d(Mix3Args a) {
#pragma clang fp contract(fast)
  using namespace m3;
  constexpr int NW = NT / 64;
  static_assert(64 / G == TX && NW == TY, "a wave takes a row of the tile at a time");
  __shared__ Field4M sfa[SN];
  __shared__ Field2M sfb[SN];
  __shared__ double acc[3][AN];
  __shared__ float spc[WPIC_MAXSP][4];  // fac1, txxx, fac2, q delx / delt
  // the waves' queued particles: old and new shape arguments, and cell in the
  // tile | species << 7 | (inc + 1) per axis << 9, 11, 13
  __shared__ float xqo[NW][6][QW];
  __shared__ int xqc[NW][QW];
  const Grid3D& g = a.g;
  const int ntiles = a.ntx * a.nty * a.ntz;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  int i0, j0, k0;
  tile_origin_m(g, tile, a.ntx, a.nty, i0, j0, k0);
  const int tid = threadIdx.x;
  for (int q = tid; q < 6 * SN; q += NT) {
    const int c = q / SN, rem = q - c * SN;
    const int i = i0 - 1 + rem % SW, j = j0 - 1 + (rem / SW) % SH, k = k0 - 1 + rem / (SW * SH);
    if (i <= g.nxge + 1 && j <= g.nye + 1 && k <= g.nze + 1) {
      const float v = (float)tmpf3m(g, a.uf, c, i, j, k);
      if (c < 4)
        sfa[rem].v[c] = v;
      else
        sfb[rem].v[c - 4] = v;
    }
  }
  for (int q = tid; q < 3 * AN; q += NT) (&acc[0][0])[q] = 0.0;
#pragma unroll
  for (int s = 0; s < WPIC_MAXSP; s++) {
    if (tid == s && s < g.nsp) {
      const float fac1 = (float)(g.q[s] / g.r[s] * 0.5 * g.delt);
      spc[s][0] = fac1;
      spc[s][1] = fac1 * fac1;
      spc[s][2] = (float)(g.q[s] * g.delt / g.r[s]);
      spc[s][3] = (float)(g.q[s] * g.delx * g.d_delt);
    }
  }
  __syncthreads();

  Mix3Const mc;
  mc.delt = (float)g.delt;
  mc.ic2 = (float)(1.0 / (g.c * g.c));
  mc.cc2 = (float)(g.c * g.c);
  // (the wave's number, the same in its lanes, and with it j and k stay in
  // scalar registers)
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lg = lane % G;
  const int li = lane / G, lj = w;
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
      const int inc[3] = {((e >> 9) & 3) - 1, ((e >> 11) & 3) - 1, ((e >> 13) & 3) - 1};
      const float o[3] = {xqo[w][0][q], xqo[w][1][q], xqo[w][2][q]};
      const float f[3] = {xqo[w][3][q], xqo[w][4][q], xqo[w][5][q]};
      deposit3_window_m(&acc[0][((cc / (TX * TY) + 2) * AH + (cc / TX % TY + 2)) * AW + (cc % TX + 2)], o, f, inc,
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
    RecM3 pr = {i, 0.5f, 0.5f, 0.5f, 0.0f, 0.0f, 0.0f, 0, 0};
    {
      int s_, p_, ia_n = 0;
      if (lg < tot) {
        cl.slot(g.nsp, lg, s_, p_);
        ia_n = a.ap ? a.ap[p_] : p_;
      }
      if (lg + G < tot) {
        cl.slot(g.nsp, lg + G, s_, p_);
        ia_nn = a.ap ? a.ap[p_] : p_;
      }
      if (lg < tot) pr = load_rec(a.A, ia_n);
    }
    // KP passes at a time: the pushes, one straight line for all lanes as in 2D
    // (a lane past its cell's last particle repeats one with zero charge and
    // stores nothing), then the current of those that stay
    int t = lg;
    while (__any(t < tot)) {
    float pd[KP][6];  // old and new shape arguments of the last KP passes, the latest first
    int ps[KP];    // species, or -1: no current from it
#pragma unroll
    for (int h = 0; h < KP; h++) {
      ps[h] = -1;
#pragma unroll
      for (int d = 0; d < 6; d++) pd[h][d] = 0.0f;
    }
    for (int h = 0; h < KP && __any(t < tot); h++, t += G) {
      const bool act = t < tot;
      int s, pi;
      cl.slot(g.nsp, t, s, pi);
      const RecM3 cur = pr;
      if (t + G < tot) pr = load_rec(a.A, ia_nn);
      if (t + 2 * G < tot) {
        int s_, p_;
        cl.slot(g.nsp, t + 2 * G, s_, p_);
        ia_nn = a.ap ? a.ap[p_] : p_;
      }
      const float* kc = spc[s];
      const Mix3Push r = mixed_push3(mc, sfa, sfb, so, kc, cur);
      const bool stays = (r.inc[0] | r.inc[1] | r.inc[2]) == 0;
      const bool mover = act && !stays;
      if (act) {
        // the x wrap is a cell wrap; the y-z step goes to the exchange
        int dj = r.inc[1], dk = r.inc[2];
        int cx = i + r.inc[0];
        if (cx < g.nxgs)
          cx += g.nx;
        else if (cx > g.nxge)
          cx -= g.nx;
        if ((unsigned)(r.inc[0] + 1) > 2u || (unsigned)(dj + 1) > 2u || (unsigned)(dk + 1) > 2u || cx < g.nxgs ||
            cx > g.nxge) {
          atomicOr(a.err, ERR_DOMAIN);
          dj = dj < -1 ? -1 : (dj > 1 ? 1 : dj);
          dk = dk < -1 ? -1 : (dk > 1 ? 1 : dk);
          cx = cx < g.nxgs ? g.nxgs : (cx > g.nxge ? g.nxge : cx);
        }
        a.code[pi] = ((cx - g.nxgs) << CODE_SHIFT3) | ((dk + 1) * 3 + (dj + 1));
        store_rec(a.B, pi, RecM3{cx, r.f[0], r.f[1], r.f[2], r.g4, r.g5, r.g6, cur.id0, cur.id1});
      }
#pragma unroll
      for (int q = KP - 1; q > 0; q--) {
        ps[q] = ps[q - 1];
#pragma unroll
        for (int d = 0; d < 6; d++) pd[q][d] = pd[q - 1][d];
      }
      ps[0] = act && stays ? s : -1;
      pd[0][0] = cur.ox - 0.5f;
      pd[0][1] = cur.oy - 0.5f;
      pd[0][2] = cur.oz - 0.5f;
#pragma unroll
      for (int d = 0; d < 3; d++) pd[0][3 + d] = r.f[d] - 0.5f;
      const uint64_t mm = __ballot(mover);
      if (mm) {
        if (mover) {
          const int slot = nq + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mm >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mm, 0));
#pragma unroll
          for (int d = 0; d < 6; d++) xqo[w][d][slot] = pd[0][d];
          xqc[w][slot] = ((lk * TY + lj) * TX + li) | (s << 7) | (((r.inc[0] + 1) & 3) << 9) |
                         (((r.inc[1] + 1) & 3) << 11) | (((r.inc[2] + 1) & 3) << 13);
        }
        nq += __popcll(mm);
        if (nq >= 64) drain();
      }
    }
    // the current of the particles that stay: sum 18 c + 9 m + 3 u + b of
    // component c, face m along its own axis, nodes u - 1, b - 1 of the other
    // two in the order x, y, z
    float v[54];
#pragma unroll
    for (int q = 0; q < 54; q++) v[q] = 0.0f;
#pragma unroll
    for (int h = 0; h < KP; h++) {
      if (!__any(ps[h] >= 0)) continue;
      const float qd = ps[h] >= 0 ? spc[ps[h] & 3][3] : 0.0f;
      float S[3][3], D[3][3], cq[3][2];  // s0, ds = s1 - s0, -sum ds
#pragma unroll
      for (int d = 0; d < 3; d++) {
        float t0, t1, t2;
        shape3m(pd[h][d], S[d][0], S[d][1], S[d][2]);
        shape3m(pd[h][3 + d], t0, t1, t2);
        D[d][0] = t0 - S[d][0];
        D[d][1] = t1 - S[d][1];
        D[d][2] = t2 - S[d][2];
        cq[d][0] = (0.0f - D[d][0]) * qd;
        cq[d][1] = ((0.0f - D[d][0]) - D[d][1]) * qd;
      }
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const float az = 0.5f * D[2][b] + S[2][b], bz = (1.0f / 3.0f) * D[2][b] + 0.5f * S[2][b];
        const float ay = 0.5f * D[1][b] + S[1][b], by = (1.0f / 3.0f) * D[1][b] + 0.5f * S[1][b];
#pragma unroll
        for (int u = 0; u < 3; u++) {
          const float wx = S[1][u] * az + D[1][u] * bz;  // y node u, z node b
          const float wy = S[0][u] * az + D[0][u] * bz;  // x node u, z node b
          const float wz = S[0][u] * ay + D[0][u] * by;  // x node u, y node b
#pragma unroll
          for (int m = 0; m < 2; m++) {
            const int q = 9 * m + 3 * u + b;
            v[q] = cq[0][m] * wx + v[q];
            v[18 + q] = cq[1][m] * wy + v[18 + q];
            v[36 + q] = cq[2][m] * wz + v[36 + q];
          }
        }
      }
    }
    // over the group, spread over its lanes (a cell without particles adds
    // nothing: its fields may be any, and 0 * NaN is not 0)
    group_reduce<54, G>(v, lane);
    // (the places are worked out here: kept over the passes they would spill)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    double* const o = &acc[0][0] + ((lk + 2) * AH + (lj + 2)) * AW + (li + 2);
#pragma unroll
    for (int f = 0; f < group_left(54, G); f++) {
      const int q = group_index<54, G>(f, ln);
      const int c = q / 18, m = q % 18 / 9, u = q % 9 / 3 - 1, b = q % 3 - 1;
      const int xo = c == 0 ? m : u, yo = c == 0 ? u : (c == 1 ? m : b), zo = c == 2 ? m : b;
      if (tot > 0 && q >= 0 && v[f] != 0.0f) tile_add(o + (c * AN + (zo * AH + yo) * AW + xo), v[f]);
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

hipError_t launch_push_deposit_mixed3d(wpic_ctx3d* c) {
  Mix3Args a;
  a.g = c->g;
  a.A = c->MA;
  a.B = c->MB;
  a.colbase = c->colbaseA;
  a.cumcnt = c->cumcnt;
  a.ap = c->aperm;
  a.uf = c->uf;
  a.uj = c->uj;
  a.code = c->code;
  a.err = c->err;
  a.ntx = (c->g.nx + m3::TX - 1) / m3::TX;
  a.nty = (c->g.ny + m3::TY - 1) / m3::TY;
  a.ntz = (c->g.nz + m3::TZ - 1) / m3::TZ;
  const int nblk = xcd_grid(a.ntx * a.nty * a.ntz);
  hipLaunchKernelGGL(k_push_deposit_mixed3d, dim3(nblk), dim3(m3::NT), 0, c->st, a);
  return hipGetLastError();
}

}  // namespace wpic
