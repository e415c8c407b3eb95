// k_mixed2d.hip -- the mixed-precision form of the fused push + deposit +
// wrap (the same physics as 2d/common/particle.f90:48-179 and
// 2d/common/field.f90:189-316 followed by the particle boundaries).
//
// A particle is an int32 x cell plus FP32 offsets (x - ix, y - row) in [0, 1)
// and FP32 momenta: positions keep ~1e-7 of a cell everywhere in the box, the
// shape functions see offsets directly, and a particle record is 32 B instead
// of 48 B.  Push and deposit run in FP32 (FMA contraction on), each cell's
// stayers summed in FP32 and the tile's current in FP64 in LDS; the tile is
// added to the FP64 uj with FP64 atomics, and the field solve
// is the FP64 one.
#include "wpic_internal.h"

namespace wpic {

namespace mx {
constexpr int TX = 32, TY = 4, NT = 256;
constexpr int SFW = TX + 2, SFH = TY + 2;
constexpr int ACW = TX + 4, ACH = TY + 4;
constexpr int QW = 128;  // queued cell-changing particles per wave: 63 left over and 64 of a pass at most
}  // namespace mx

struct MixArgs {
  Grid2D g;
  PartsM A, B;
  const int* rowbase;
  const int* cumcnt;
  const int* ap;  // A's slot -> record (null: identity)
  const double* uf;
  double* uj;
  int* code;
  int* err;
  int ntx, nty;
  int tw;     // columns of cells a workgroup takes (the push)
  int* rcnt;  // particles per (species, row, x cell) after the step, or null
};

// cell-centred field component c at (i, j) (particle.f90:74-80), FP64
__device__ inline double cell_field_m(const Grid2D& g, const double* uf, int c, int i, int j) {
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

__device__ inline void shape3f(float dh, float& s0, float& s1, float& s2) {
  s0 = 0.5f * (0.5f - dh) * (0.5f - dh);
  s1 = 0.75f - dh * dh;
  s2 = 0.5f * (0.5f + dh) * (0.5f + dh);
}

// ds = (new shape shifted by inc) - s0, index 0..4 <-> -2..2, with the
// reference's smo_* weights (field.f90:244-266); |inc| <= 1 except for a
// particle that a reflecting wall sends across two cells, where the formula is
// applied as the reference applies it
__device__ inline void ds_of(float s0m, float s00, float s0p, float fnew, int inc, float ds[5]) {
  float s1m, s10, s1p;
  shape3f(fnew - 0.5f, s1m, s10, s1p);
  const float a = (float)abs(inc);
  const float smo1 = inc < 0 ? a : 0.0f, smo2 = 1.0f - a, smo3 = inc > 0 ? a : 0.0f;
  ds[0] = s1m * smo1;
  ds[1] = s1m * smo2 + s10 * smo1 - s0m;
  ds[2] = s10 * smo2 + s1p * smo1 + s1m * smo3 - s00;
  ds[3] = s1p * smo2 + s10 * smo3 - s0p;
  ds[4] = s1p * smo3;
}

// FP32 reciprocal and reciprocal square root of the hardware (about one ulp):
// the mixed form's arithmetic is FP32 throughout, so correctly rounded
// division sequences buy nothing its 1e-7 offsets can hold
__device__ inline float rcpf(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline float rsqf(float x) { return __builtin_amdgcn_rsqf(x); }

// The 4-node window [lo, lo + 3] (of the 5 nodes -2..2) of one axis that holds
// every non-zero s0 and ds: S0 and DS on it, the new shape with the reference's
// weights, |inc| moved by one node and 1 - |inc| unmoved, as in the FP64 kernel
__device__ inline void window_f(float o, float f, int inc, float S0[4], float DS[4], int& lo) {
  float t0, t1, t2, u0, u1, u2;
  shape3f(o - 0.5f, t0, t1, t2);
  shape3f(f - 0.5f, u0, u1, u2);
  const bool left = inc < 0;
  lo = left ? 0 : 1;
  const float far = (float)abs(inc), near = 1.0f - far;
  const float p = left ? far : near, q = left ? near : far;
  S0[0] = left ? 0.0f : t0;
  S0[1] = left ? t0 : t1;
  S0[2] = left ? t1 : t2;
  S0[3] = left ? t2 : 0.0f;
  DS[0] = p * u0 - S0[0];
  DS[1] = p * u1 + q * u0 - S0[1];
  DS[2] = p * u2 + q * u1 - S0[2];
  DS[3] = q * u2 - S0[3];
}

// The fields of a cell side by side, so that the gather's 54 values come in 18
// LDS reads at immediate offsets from one address
struct alignas(16) Fields4 {
  float bx, by, bz, ex;
};
struct alignas(8) Fields2 {
  float ey, ez;
};

// Push, deposit, wrap and exchange code in one pass, as the FP64 fast kernel
// does it (k_push2d.hip): wave w walks row w of the tile, 64 / G cells a round
// (one per G-lane group, all species as one list behind a two-deep load
// pipeline).  A particle that stays in its cell adds to 21 FP32 sums in its
// lane's registers, reduced over the group once per cell; one that changes
// cell joins the wave's LDS queue, and whenever 64 have gathered the whole
// wave deposits them.  The tile's current is FP64 in LDS (FP32 LDS atomics
// serialize badly when lanes meet on a node) and goes to uj with one FP64
// atomic per node.
//
// At 128 particles a cell the kernel is bound by memory: 1024x1024, 64 ppc
// moves 11.6 GB (9.7 algorithmic: the record each way, its permutation entry
// and its exchange code) in 2.9 ms, 4.0 TB/s where a plain copy reaches 4.8.
// With one array per field and 65 FP32 sums per lane over 32-lane groups it
// took 3.4 ms.
template <int G, int BC>
__global__ __launch_bounds__(mx::NT, 3) void k_push_deposit_mixed(MixArgs a) {
#pragma clang fp contract(fast)
  using namespace mx;
  __shared__ Fields4 sf4[SFW * SFH];
  __shared__ Fields2 sf2[SFW * SFH];
  __shared__ double acc[3][ACW * ACH];
  __shared__ float spc[WPIC_MAXSP][5];  // fac1, txxx, fac2, qk, q
  __shared__ float xqd[NT / 64][5][QW];  // ox, oy, new offsets, q vz
  __shared__ int xqc[NT / 64][QW];       // cell in the tile | species << 8 | x step + 8 << 10 | y step + 1 << 14
  // particles per (species, row, cell) after the step for the tile's cells
  // and their one-cell halo (rcnt)
  __shared__ int hcn[WPIC_MAXSP][TY + 2][TX + 2];
  const bool counting = a.rcnt != nullptr;

  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * a.tw;
  const int j0 = g.nys + (tile / a.ntx) * TY;
  const int tid = threadIdx.x;

  {
    const int w = a.tw + 2, n = w * SFH;
    for (int k = tid; k < 6 * n; k += NT) {
      const int c = k / n, rem = k - c * n;
      const int r = rem / w, q = rem - r * w;
      const int i = i0 - 1 + q, j = j0 - 1 + r;
      if (i <= g.nxge + 1 && j <= g.nye + 1) {
        const float v = (float)cell_field_m(g, a.uf, c, i, j);
        float* const p = c < 4 ? &sf4[r * SFW + q].bx + c : &sf2[r * SFW + q].ey + (c - 4);
        *p = v;
      }
    }
  }
  for (int k = tid; k < 3 * ACW * ACH; k += NT) (&acc[0][0])[k] = 0.0;
  if (counting)
    for (int k = tid; k < WPIC_MAXSP * (TY + 2) * (TX + 2); k += NT) (&hcn[0][0][0])[k] = 0;
  // per-species constants (particle.f90:92-94, field.f90:274), formed in FP64
  // and rounded once
  if (tid < g.nsp && tid < WPIC_MAXSP) {
    const double q = g.q[tid], rm = g.r[tid];
    const float fac1 = (float)(q / rm * 0.5 * g.delt);
    spc[tid][0] = fac1;
    spc[tid][1] = fac1 * fac1;
    spc[tid][2] = (float)(q * g.delt / rm);
    spc[tid][3] = (float)(q * g.delx * g.d_delt);
    spc[tid][4] = (float)q;
  }
  __syncthreads();

  static_assert(NT / 64 == TY && 8 % (64 / G) == 0, "one wave per tile row, whole rounds of any tile width");
  constexpr int RX = 64 / G;  // cells per wave round
  const int w = tid >> 6, lane = tid & 63, lg = lane % G;
  const int lj = w, j = j0 + lj;
  const float delt = (float)g.delt;
  const float ic2 = (float)(1.0 / (g.c * g.c));
  const float cc2 = (float)(g.c * g.c);
  int nq = 0;  // queued particles, the same in all lanes
  float(*const qd)[QW] = xqd[w];
  int* const qc = xqc[w];

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
      const int e = qc[q];
      const int qli = (e & 255) % TX, qlj = (e & 255) / TX;
      const int incx = ((e >> 10) & 15) - 8, incy = ((e >> 14) & 3) - 1;
      const float qk = spc[(e >> 8) & 3][3];
      const float ox = qd[0][q], oy = qd[1][q], fx = qd[2][q], fy = qd[3][q], qvz = qd[4][q];
      if (BC == WPIC_BC_PERIODIC) {
        float S0x[4], DSx[4], S0y[4], DSy[4];
        int lox, loy;
        window_f(ox, fx, incx, S0x, DSx, lox);
        window_f(oy, fy, incy, S0y, DSy, loy);
        const bool mx = incx != 0, my = incy != 0;
        double* const o = &acc[0][(qlj + loy) * ACW + (qli + lox)];  // window node (0, 0)
        // the fourth node of an axis along which the particle keeps its cell
        // carries nothing, and that axis' third face only rounding
        const float cx0 = -DSx[0], cx1 = cx0 - DSx[1], cx2 = cx1 - DSx[2];
#pragma unroll
        for (int n = 0; n < 4; n++) {
          if (n == 3 && !my) break;
          const float ay = S0y[n] + 0.5f * DSy[n];
          const float wy = qk * ay, A = qvz * ay, B = qvz * (0.5f * S0y[n] + (1.0f / 3.0f) * DSy[n]);
          double* const r = o + n * ACW;
          double* const z = r + 2 * ACW * ACH;
          atomicAdd(r + 1, (double)(cx0 * wy));
          atomicAdd(r + 2, (double)(cx1 * wy));
          atomicAdd(z, (double)(S0x[0] * A + DSx[0] * B));
          atomicAdd(z + 1, (double)(S0x[1] * A + DSx[1] * B));
          atomicAdd(z + 2, (double)(S0x[2] * A + DSx[2] * B));
          if (mx) {
            atomicAdd(r + 3, (double)(cx2 * wy));
            atomicAdd(z + 3, (double)(S0x[3] * A + DSx[3] * B));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        float wx[4], cy = 0.0f;
#pragma unroll
        for (int n = 0; n < 4; n++) wx[n] = qk * (S0x[n] + 0.5f * DSx[n]);
#pragma unroll
        for (int m = 0; m < 3; m++) {
          if (m == 2 && !my) break;
          cy -= DSy[m];
          double* const r = o + ACW * ACH + (m + 1) * ACW;
          atomicAdd(r, (double)(cy * wx[0]));
          atomicAdd(r + 1, (double)(cy * wx[1]));
          atomicAdd(r + 2, (double)(cy * wx[2]));
          if (mx) atomicAdd(r + 3, (double)(cy * wx[3]));
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        // a wall may reflect by more than one cell: the full 5x5 block
        float sx0, sx1, sx2, sy0, sy1, sy2, dsx[5], dsy[5];
        shape3f(ox - 0.5f, sx0, sx1, sx2);
        shape3f(oy - 0.5f, sy0, sy1, sy2);
        ds_of(sx0, sx1, sx2, fx, incx, dsx);
        ds_of(sy0, sy1, sy2, fy, incy, dsy);
        const float s0x[5] = {0.0f, sx0, sx1, sx2, 0.0f}, s0y[5] = {0.0f, sy0, sy1, sy2, 0.0f};
        double* const o = &acc[0][qlj * ACW + qli];  // node (-2, -2)
        float cx = 0.0f, cy = 0.0f;
#pragma unroll
        for (int m = 0; m < 4; m++) {
          cx -= dsx[m];
          cy -= dsy[m];
#pragma unroll
          for (int n = 0; n < 5; n++) {
            const float vx = cx * (qk * (s0y[n] + 0.5f * dsy[n])), vy = cy * (qk * (s0x[n] + 0.5f * dsx[n]));
            if (vx != 0.0f) atomicAdd(o + n * ACW + m + 1, (double)vx);
            if (vy != 0.0f) atomicAdd(o + ACW * ACH + (m + 1) * ACW + n, (double)vy);
          }
        }
#pragma unroll
        for (int jp = 0; jp < 5; jp++) {
          const float A = qvz * (s0y[jp] + 0.5f * dsy[jp]), B = qvz * (0.5f * s0y[jp] + (1.0f / 3.0f) * dsy[jp]);
#pragma unroll
          for (int ip = 0; ip < 5; ip++) {
            const float v = s0x[ip] * A + dsx[ip] * B;
            if (v != 0.0f) atomicAdd(o + 2 * ACW * ACH + jp * ACW + ip, (double)v);
          }
        }
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
    // stayers: [0,6) Jx (face m, y node u - 1) at 3 m + u, [6,12) Jy (face m,
    // x node u - 1), [12,21) Jz (y node v - 1, x node u - 1) at 12 + 3 v + u
    float v[21];
#pragma unroll
    for (int k = 0; k < 21; k++) v[k] = 0.0f;

    // the cell's particles over all species as one list, walked with a
    // two-deep software pipeline: the record of element t + G and the
    // permutation entry of element t + 2G are in flight while element t is
    // pushed
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
    RecM pr = {i, 0.5f, 0.5f, 0.0f, 0.0f, 0.0f, 0};
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
    // every lane of the wave runs the passes of the wave's fullest cell in one
    // straight line, as in the FP64 kernel: a lane past its cell's last
    // particle repeats that one with zero charge and stores nothing
    for (int t = lg; __any(t < tot); t += G) {
      const bool act = t < tot;
      float ox, oy, fx, fy, qvz;
      int s, incx, incy;
      bool mover;
      {
        int pi;
        cl.slot(g.nsp, t, s, pi);
        ox = pr.ox, oy = pr.oy;
        const float u1 = pr.ux, u2 = pr.uy, u3 = pr.uz;
        const uint64_t id = pr.id;
        if (t + G < tot) pr = load_rec(a.A, ia_nn);
        if (t + 2 * G < tot) {
          int s_, p_;
          cl.slot(g.nsp, t + 2 * G, s_, p_);
          ia_nn = a.ap ? a.ap[p_] : p_;
        }
        const float* kc = spc[s];
        const float fac1 = kc[0], txxx = kc[1], fac2 = kc[2];
        // the reads of the gather's next row are in flight while one is combined
        int so = lj * SFW + li;
        asm volatile("" : "+v"(so));
        Fields4 f4[2][3];
        Fields2 f2[2][3];
        auto load = [&](int r) {
#pragma unroll
          for (int k = 0; k < 3; k++) {
            f4[r & 1][k] = sf4[so + r * SFW + k];
            f2[r & 1][k] = sf2[so + r * SFW + k];
          }
        };
        load(0);
        __builtin_amdgcn_sched_barrier(0);
        float sx[3], sy[3];
        shape3f(ox - 0.5f, sx[0], sx[1], sx[2]);
        shape3f(oy - 0.5f, sy[0], sy[1], sy[2]);
        float bpx = 0.0f, bpy = 0.0f, bpz = 0.0f, epx = 0.0f, epy = 0.0f, epz = 0.0f;
#pragma unroll
        for (int r = 0; r < 3; r++) {
          if (r < 2) load(r + 1);
          __builtin_amdgcn_sched_barrier(0);
          const Fields4* p = f4[r & 1];
          const Fields2* q = f2[r & 1];
          bpx += (p[0].bx * sx[0] + p[1].bx * sx[1] + p[2].bx * sx[2]) * sy[r];
          bpy += (p[0].by * sx[0] + p[1].by * sx[1] + p[2].by * sx[2]) * sy[r];
          bpz += (p[0].bz * sx[0] + p[1].bz * sx[1] + p[2].bz * sx[2]) * sy[r];
          epx += (p[0].ex * sx[0] + p[1].ex * sx[1] + p[2].ex * sx[2]) * sy[r];
          epy += (q[0].ey * sx[0] + q[1].ey * sx[1] + q[2].ey * sx[2]) * sy[r];
          epz += (q[0].ez * sx[0] + q[1].ez * sx[1] + q[2].ez * sx[2]) * sy[r];
          __builtin_amdgcn_sched_barrier(0);
        }
        float uvm1 = u1 + fac1 * epx;
        float uvm2 = u2 + fac1 * epy;
        float uvm3 = u3 + fac1 * epz;
        const float gam2 = cc2 + uvm1 * uvm1 + uvm2 * uvm2 + uvm3 * uvm3;
        const float igam = rsqf(gam2);
        const float gam = gam2 * igam;
        const float fac1r = fac1 * igam;
        const float fac2r = fac2 * rcpf(gam + txxx * (bpx * bpx + bpy * bpy + bpz * bpz) * igam);
        const float uvm4 = uvm1 + fac1r * (uvm2 * bpz - uvm3 * bpy);
        const float uvm5 = uvm2 + fac1r * (uvm3 * bpx - uvm1 * bpz);
        const float uvm6 = uvm3 + fac1r * (uvm1 * bpy - uvm2 * bpx);
        uvm1 = uvm1 + fac2r * (uvm5 * bpz - uvm6 * bpy);
        uvm2 = uvm2 + fac2r * (uvm6 * bpx - uvm4 * bpz);
        uvm3 = uvm3 + fac2r * (uvm4 * bpy - uvm5 * bpx);
        float g3 = uvm1 + fac1 * epx, g4 = uvm2 + fac1 * epy, g5 = uvm3 + fac1 * epz;
        const float gmv = rsqf(1.0f + (g3 * g3 + g4 * g4 + g5 * g5) * ic2);
        // new position as cell + offset
        const float nx_ = ox + g3 * delt * gmv, ny_ = oy + g4 * delt * gmv;
        float fxi = floorf(nx_), fyi = floorf(ny_);
        incx = (int)fxi, incy = (int)fyi;
        fx = nx_ - fxi, fy = ny_ - fyi;
        if (fx >= 1.0f) { fx -= 1.0f; incx += 1; }
        if (fy >= 1.0f) { fy -= 1.0f; incy += 1; }
        int cx = i + incx;
        // reflecting walls act before the deposit (reconnection order,
        // boundary_reconnection.f90:79-91): x' = 2(nxs+1) - x or 2(nxe-1) - x
        if (BC == WPIC_BC_WALLX && (cx < g.nxgs + 1 || cx >= g.nxge - 1)) {
          const int W = cx < g.nxgs + 1 ? 2 * (g.nxgs + 1) : 2 * (g.nxge - 1);
          cx = W - cx - 1;
          fx = 1.0f - fx;
          if (fx >= 1.0f) { fx -= 1.0f; cx += 1; }
          g3 = -g3; g4 = -g4; g5 = -g5;
          incx = cx - i;
        }
        if (act && (incy < -1 || incy > 1)) {
          atomicOr(a.err, ERR_DOMAIN);
          incy = incy < -1 ? -1 : 1;
        }

        // Esirkepov weights from offsets, factored as the FP64 fast kernel
        qvz = kc[4] * (g5 * gmv);
        const bool stays = (incx | incy) == 0;
        mover = act && !stays;
        {
          const float qk = act && stays ? kc[3] : 0.0f, qz = act && stays ? qvz : 0.0f;
          float dsx[3], dsy[3];
          shape3f(fx - 0.5f, dsx[0], dsx[1], dsx[2]);
          shape3f(fy - 0.5f, dsy[0], dsy[1], dsy[2]);
#pragma unroll
          for (int k = 0; k < 3; k++) {
            dsx[k] -= sx[k];
            dsy[k] -= sy[k];
          }
          const float cx1 = -dsx[0], cx2 = cx1 - dsx[1], cy1 = -dsy[0], cy2 = cy1 - dsy[1];
#pragma unroll
          for (int u = 0; u < 3; u++) {
            const float ty = sy[u] + 0.5f * dsy[u];
            const float wy = qk * ty, wx = qk * (sx[u] + 0.5f * dsx[u]);
            v[u] += cx1 * wy;
            v[3 + u] += cx2 * wy;
            v[6 + u] += cy1 * wx;
            v[9 + u] += cy2 * wx;
            const float A = qz * ty, B = qz * (0.5f * sy[u] + (1.0f / 3.0f) * dsy[u]);
#pragma unroll
            for (int k = 0; k < 3; k++) v[12 + 3 * u + k] += sx[k] * A + dsx[k] * B;
          }
        }

        if (act) {
          // periodic x wrap of the cell; the row step goes to the exchange
          if (BC == WPIC_BC_PERIODIC) {
            if (cx < g.nxgs) cx += g.nx;
            else if (cx > g.nxge) cx -= g.nx;
          }
          if (cx < g.nxgs || cx > g.nxge) {
            atomicOr(a.err, ERR_DOMAIN);
            cx = cx < g.nxgs ? g.nxgs : g.nxge;
          }
          store_rec(a.B, pi, RecM{cx, fx, fy, g3, g4, g5, id});
          const int code = ((cx - g.nxgs) << 2) | (incy + 1);
          a.code[pi] = code;
          if (counting && code != (((i - g.nxgs) << 2) | 1)) count_leaver<TX, TY>(g, hcn, a.rcnt, i0, j0, li, lj, s, code);
        }
      }
      const uint64_t mm = __ballot(mover);
      if (mm) {
        if (mover) {
          const int slot = nq + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mm >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mm, 0));
          qd[0][slot] = ox;
          qd[1][slot] = oy;
          qd[2][slot] = fx;
          qd[3][slot] = fy;
          qd[4][slot] = qvz;
          qc[slot] = (lj * TX + li) | (s << 8) | ((incx + 8) << 10) | ((incy + 1) << 14);
        }
        nq += __popcll(mm);
        if (nq >= 64) drain();
      }
    }
    // the stayers' 21 sums over the group, spread over its lanes (a cell without
    // particles adds nothing: its fields may be any, and 0 * NaN is not 0)
    group_reduce<21, G>(v, lane);
#pragma unroll
    for (int f = 0; f < NRES; f++)
      if (tot > 0 && node[f] >= 0 && v[f] != 0.0f) atomicAdd(&acc[0][0] + (node[f] + li), (double)v[f]);
  }
  if (nq) drain();

  __syncthreads();
  if (counting) flush_counts<TX, TY>(g, hcn, a.rcnt, a.cumcnt, i0, j0, a.tw);
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

// The moments of the output sequence in the mixed form: mom_calc__accl's
// half-step kick (2d/common/mom_calc.f90:84-155, delt/2, no move) and
// mom_calc__nvt's CIC deposit of the seven moments (:167-249) fused, FP32 per
// particle from the int32 cell + FP32 offset record, accumulated per species
// in an FP64 LDS node tile (one-node halo; the lanes of a group share their
// cell's nodes, and FP32 LDS atomics that meet on an address serialize far
// worse than FP64 ones) and added to the FP64 mom array with one FP64 atomic
// per node and moment.  The lower CIC node of a particle
// at cell i + offset o is i when o >= 1/2 (weight o - 1/2 on i + 1), else
// i - 1 (weight o + 1/2 on i): int(x/dx - 1/2) and x/dx - 1/2 - ih of the
// reference, with delx = 1.
__global__ __launch_bounds__(mx::NT) void k_mom_mixed(MixArgs a, double* mom) {
#pragma clang fp contract(fast)
  using namespace mx;
  constexpr int GM = 8, NGRP = NT / GM;
  constexpr int MTW = TX + 2, MTH = TY + 2;
  __shared__ float sf[6][SFW * SFH];
  __shared__ double mt[7][MTW * MTH];
  const Grid2D& g = a.g;
  const int ntiles = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  if (tile >= ntiles) return;
  const int i0 = g.nxgs + (tile % a.ntx) * TX;
  const int j0 = g.nys + (tile / a.ntx) * TY;
  const int ncx = min(TX, g.nxge + 1 - i0), ncy = min(TY, g.nye + 1 - j0);
  const int tid = threadIdx.x;
  for (int k = tid; k < 6 * SFW * SFH; k += NT) {
    const int c = k / (SFW * SFH), rem = k - c * (SFW * SFH);
    const int i = i0 - 1 + rem % SFW, j = j0 - 1 + rem / SFW;
    if (i <= g.nxge + 1 && j <= g.nye + 1) sf[c][rem] = (float)cell_field_m(g, a.uf, c, i, j);
  }
  const int grp = tid / GM, lg = tid % GM;
  const float ic2 = (float)(1.0 / (g.c * g.c));
  const float cc2 = (float)(g.c * g.c);
  const int rot = tid % 7;  // lanes meeting on a node add to different planes first

  for (int s = 0; s < g.nsp; s++) {
    for (int k = tid; k < 7 * MTW * MTH; k += NT) (&mt[0][0])[k] = 0.0;
    __syncthreads();
    const double hdelt = g.delt * 0.5;
    const float fac1 = (float)(g.q[s] / g.r[s] * 0.5 * hdelt);
    const float txxx = fac1 * fac1;
    const float fac2 = (float)(g.q[s] * hdelt / g.r[s]);
    for (int cc = grp; cc < TX * TY; cc += NGRP) {
      const int li = cc % TX, lj = cc / TX;
      if (li >= ncx || lj >= ncy) continue;  // uniform within a group
      const int i = i0 + li, j = j0 + lj;
      const int rw = s * g.ny + (j - g.nys);
      const int* cr = a.cumcnt + (size_t)rw * (g.nx + 1);
      const int base = a.rowbase[rw];
      const int pe = base + cr[i - g.nxgs + 1];
      for (int pi = base + cr[i - g.nxgs] + lg; pi < pe; pi += GM) {
        const int ia = a.ap ? a.ap[pi] : pi;
        const float ox = a.A.ox[ia], oy = a.A.oy[ia];
        float sx0, sx1, sx2, sy0, sy1, sy2;
        shape3f(ox - 0.5f, sx0, sx1, sx2);
        shape3f(oy - 0.5f, sy0, sy1, sy2);
        const int so = (lj + 1) * SFW + (li + 1);
        float fl[6];
#pragma unroll
        for (int cm = 0; cm < 6; cm++) {
          const float* f = &sf[cm][so];
          fl[cm] = (f[-SFW - 1] * sx0 + f[-SFW] * sx1 + f[-SFW + 1] * sx2) * sy0 +
                   (f[-1] * sx0 + f[0] * sx1 + f[1] * sx2) * sy1 +
                   (f[SFW - 1] * sx0 + f[SFW] * sx1 + f[SFW + 1] * sx2) * sy2;
        }
        const float bpx = fl[0], bpy = fl[1], bpz = fl[2], epx = fl[3], epy = fl[4], epz = fl[5];
        float uvm1 = a.A.ux[ia] + fac1 * epx;
        float uvm2 = a.A.uy[ia] + fac1 * epy;
        float uvm3 = a.A.uz[ia] + fac1 * epz;
        const float gam = sqrtf(cc2 + uvm1 * uvm1 + uvm2 * uvm2 + uvm3 * uvm3);
        const float igam = 1.0f / gam;
        const float fac1r = fac1 * igam;
        const float fac2r = fac2 / (gam + txxx * (bpx * bpx + bpy * bpy + bpz * bpz) * igam);
        const float uvm4 = uvm1 + fac1r * (uvm2 * bpz - uvm3 * bpy);
        const float uvm5 = uvm2 + fac1r * (uvm3 * bpx - uvm1 * bpz);
        const float uvm6 = uvm3 + fac1r * (uvm1 * bpy - uvm2 * bpx);
        uvm1 = uvm1 + fac2r * (uvm5 * bpz - uvm6 * bpy);
        uvm2 = uvm2 + fac2r * (uvm6 * bpx - uvm4 * bpz);
        uvm3 = uvm3 + fac2r * (uvm4 * bpy - uvm5 * bpx);
        const float ux = uvm1 + fac1 * epx, uy = uvm2 + fac1 * epy, uz = uvm3 + fac1 * epz;
        const float gi = 1.0f / sqrtf(1.0f + (ux * ux + uy * uy + uz * uz) * ic2);
        const bool hx = ox >= 0.5f, hy = oy >= 0.5f;
        const float dx = hx ? ox - 0.5f : ox + 0.5f, dxm = 1.0f - dx;
        const float dy = hy ? oy - 0.5f : oy + 0.5f, dym = 1.0f - dy;
        const int lx = li + (hx ? 1 : 0), ly = lj + (hy ? 1 : 0);  // lower node in the tile (halo at 0)
        float mv[7] = {1.0f, ux * gi, uy * gi, uz * gi, ux * ux * gi, uy * uy * gi, uz * uz * gi};
        const float w00 = dxm * dym, w10 = dx * dym, w01 = dxm * dy, w11 = dx * dy;
        double* node = &mt[0][ly * MTW + lx];
#pragma unroll
        for (int q = 0; q < 7; q++) {
          const int plane = q + rot < 7 ? q + rot : q + rot - 7;
          const float v = mv[plane];
          double* p = node + plane * (MTW * MTH);
          atomicAdd(p, (double)(v * w00));
          atomicAdd(p + 1, (double)(v * w10));
          atomicAdd(p + MTW, (double)(v * w01));
          atomicAdd(p + MTW + 1, (double)(v * w11));
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
      unsafeAtomicAdd(mom + midx(g, I, J, s) + comp, v);
    }
    __syncthreads();
  }
}

hipError_t launch_mom_mixed(wpic_ctx* c) {
  MixArgs a;
  a.g = c->g;
  a.A = c->MA;
  a.B = c->MB;
  a.rowbase = c->rowbaseA;
  a.cumcnt = c->cumcnt;
  a.ap = c->aperm;
  a.uf = c->uf;
  a.uj = c->uj;
  a.code = c->code;
  a.err = c->err;
  a.ntx = (c->g.nx + mx::TX - 1) / mx::TX;
  a.nty = (c->g.ny + mx::TY - 1) / mx::TY;
  hipError_t e = launch_zero(c, c->mom, (size_t)7 * (c->g.nx + 2) * (c->g.ny + 2) * c->g.nsp);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mom_mixed, dim3(xcd_grid(a.ntx * a.nty)), dim3(mx::NT), 0, c->st, a, c->mom);
  return hipGetLastError();
}

hipError_t launch_push_deposit_mixed(wpic_ctx* c) {
  MixArgs a;
  a.g = c->g;
  a.A = c->MA;
  a.B = c->MB;
  a.rowbase = c->rowbaseA;
  a.cumcnt = c->cumcnt;
  a.ap = c->aperm;
  a.uf = c->uf;
  a.uj = c->uj;
  a.code = c->code;
  a.err = c->err;
  a.tw = tile_width(c->g);
  a.ntx = (c->g.nx + a.tw - 1) / a.tw;
  a.nty = (c->g.ny + mx::TY - 1) / mx::TY;
  a.rcnt = c->rcnt_fill ? c->rcnt : nullptr;
  const int nblk = xcd_grid(a.ntx * a.nty);
  // lane groups as in the FP64 push (launch_push_deposit)
  const bool wide = c->npart >= 96ll * c->g.nx * c->g.ny;
#define L(G, BC) hipLaunchKernelGGL((k_push_deposit_mixed<G, BC>), dim3(nblk), dim3(mx::NT), 0, c->st, a)
  if (c->g.bc == WPIC_BC_WALLX) {
    if (wide)
      L(16, WPIC_BC_WALLX);
    else
      L(8, WPIC_BC_WALLX);
  } else {
    if (wide)
      L(16, WPIC_BC_PERIODIC);
    else
      L(8, WPIC_BC_PERIODIC);
  }
#undef L
  return hipGetLastError();
}

}  // namespace wpic
