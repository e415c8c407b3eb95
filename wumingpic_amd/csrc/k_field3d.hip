// k_field3d.hip -- the 3D implicit FDTD update of 3d/common/field.f90:70-208:
// current ghost folds (boundary_periodic__curre, 3d/common/boundary_periodic.f90:
// 676-978), the right-hand side gkl (:128-158), the three CG solves of cgm
// (:409-560) in lock step with per-component stopping, the E update (:164-187),
// the field ghost fills (boundary_periodic__dfield, :458-673) and uf += df.
//
// CG vectors hold the interior only; the 7-point stencil maps an out-of-range
// face neighbour to its periodic image, the value boundary_periodic__phi
// (:981-1099) copies into that ghost.  Dot products: fast mode sums fixed
// per-block partials in a fixed tree (deterministic), parity mode sums
// serially in the reference's (k, j, i) order.
#include "wpic_internal3d.h"

namespace wpic {

namespace {

constexpr double kPi = 3.141592653589793;  // 4d0*atan(1d0)

__device__ inline double bsum256(double v, double* sh) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return t;
}

__device__ inline size_t tid1() { return blockIdx.x * (size_t)blockDim.x + threadIdx.x; }

}  // namespace

// ---------------------------------------------------------------------------
// current ghosts, in the order of boundary_periodic__curre
// ---------------------------------------------------------------------------
// y: fold the two ghost rows of every (i, k), ghosts included
__global__ void k_curre3_yfold(Grid3D g, double* uj) {
  const size_t t = tid1();
  const size_t per = (size_t)g.fw * g.fd;
  if (t >= 3 * per) return;
  const int comp = (int)(t / per);
  const int I = g.nxgs - 2 + (int)(t % g.fw), K = g.nzs - 2 + (int)((t % per) / g.fw);
  double* u = uj + plane3(g) * comp;
  const int nys = g.nys, nye = g.nye;
  const double a = u[fidx3(g, I, nys - 2, K)], b = u[fidx3(g, I, nys - 1, K)];
  u[fidx3(g, I, nye - 1, K)] = u[fidx3(g, I, nye - 1, K)] + a;
  u[fidx3(g, I, nye, K)] = u[fidx3(g, I, nye, K)] + b;
  const double c = u[fidx3(g, I, nye + 1, K)], d = u[fidx3(g, I, nye + 2, K)];
  u[fidx3(g, I, nys, K)] = u[fidx3(g, I, nys, K)] + c;
  u[fidx3(g, I, nys + 1, K)] = u[fidx3(g, I, nys + 1, K)] + d;
}

// z: fold the two ghost planes for interior j, all i
__global__ void k_curre3_zfold(Grid3D g, double* uj) {
  const size_t t = tid1();
  const size_t per = (size_t)g.fw * g.ny;
  if (t >= 3 * per) return;
  const int comp = (int)(t / per);
  const int I = g.nxgs - 2 + (int)(t % g.fw), J = g.nys + (int)((t % per) / g.fw);
  double* u = uj + plane3(g) * comp;
  const int nzs = g.nzs, nze = g.nze;
  const double a = u[fidx3(g, I, J, nzs - 2)], b = u[fidx3(g, I, J, nzs - 1)];
  u[fidx3(g, I, J, nze - 1)] = u[fidx3(g, I, J, nze - 1)] + a;
  u[fidx3(g, I, J, nze)] = u[fidx3(g, I, J, nze)] + b;
  const double c = u[fidx3(g, I, J, nze + 1)], d = u[fidx3(g, I, J, nze + 2)];
  u[fidx3(g, I, J, nzs)] = u[fidx3(g, I, J, nzs)] + c;
  u[fidx3(g, I, J, nzs + 1)] = u[fidx3(g, I, J, nzs + 1)] + d;
}

// one ghost row copied back in y, for interior k
__global__ void k_curre3_ycopy(Grid3D g, double* uj) {
  const size_t t = tid1();
  const size_t per = (size_t)g.fw * g.nz;
  if (t >= 3 * per) return;
  const int comp = (int)(t / per);
  const int I = g.nxgs - 2 + (int)(t % g.fw), K = g.nzs + (int)((t % per) / g.fw);
  double* u = uj + plane3(g) * comp;
  u[fidx3(g, I, g.nye + 1, K)] = u[fidx3(g, I, g.nys, K)];
  u[fidx3(g, I, g.nys - 1, K)] = u[fidx3(g, I, g.nye, K)];
}

// one ghost plane copied back in z, for j in nys-1..nye+1
__global__ void k_curre3_zcopy(Grid3D g, double* uj) {
  const size_t t = tid1();
  const size_t per = (size_t)g.fw * (g.ny + 2);
  if (t >= 3 * per) return;
  const int comp = (int)(t / per);
  const int I = g.nxgs - 2 + (int)(t % g.fw), J = g.nys - 1 + (int)((t % per) / g.fw);
  double* u = uj + plane3(g) * comp;
  u[fidx3(g, I, J, g.nze + 1)] = u[fidx3(g, I, J, g.nzs)];
  u[fidx3(g, I, J, g.nzs - 1)] = u[fidx3(g, I, J, g.nze)];
}

// x: fold then copy two layers, every (j, k)
__global__ void k_curre3_x(Grid3D g, double* uj) {
  const size_t t = tid1();
  const size_t per = (size_t)g.fh * g.fd;
  if (t >= 3 * per) return;
  const int comp = (int)(t / per);
  const int J = g.nys - 2 + (int)(t % g.fh), K = g.nzs - 2 + (int)((t % per) / g.fh);
  double* u = uj + plane3(g) * comp;
  const int nxs = g.nxgs, nxe = g.nxge;
#define U(i) u[fidx3(g, i, J, K)]
  U(nxe - 1) = U(nxe - 1) + U(nxs - 2);
  U(nxe) = U(nxe) + U(nxs - 1);
  U(nxs) = U(nxs) + U(nxe + 1);
  U(nxs + 1) = U(nxs + 1) + U(nxe + 2);
  U(nxs - 2) = U(nxe - 1);
  U(nxs - 1) = U(nxe);
  U(nxe + 1) = U(nxs);
  U(nxe + 2) = U(nxs + 1);
#undef U
}

// ---------------------------------------------------------------------------
// CG
// ---------------------------------------------------------------------------
struct Cg3Args {
  Grid3D g;
  const double *uf, *uj;
  double* df;
  double *phi, *pold, *pnew, *r, *b, *ap;  // [3][nx*ny*nz]
  double* part;                            // [3][3][NPB3]: per component, see k_cg3_a
  CgScal *sc, *sp;                         // this iteration's scalars and the previous one's
  int* err;
  CgPoll* poll;  // where to tell the host how the solve stands (null: not now)
  int nb0, nb;   // blocks (and partial sums) of k_cg3_init, and of an iteration's kernels per component
  int first;     // the solve's first iteration
};

// in 32-bit arithmetic: a context holds fewer than 2^31 cells
__device__ inline void decode3(const Grid3D& g, size_t q, int& i, int& j, int& k) {
  const unsigned qq = (unsigned)q, nx = (unsigned)g.nx, ny = (unsigned)g.ny;
  const unsigned row = qq / nx;
  i = g.nxgs + (int)(qq - row * nx);
  j = g.nys + (int)(row % ny);
  k = g.nzs + (int)(row / ny);
}

// One block's sum of its threads' values, kept as partial sum `slot` of
// component l.
enum { S_RR = 0, S_PAP = 1, S_BB = 2 };  // r.r, p.ap, b.b
__device__ inline void put_part3(const Cg3Args& a, int l, int slot, double v, double* sh) {
  const double t = bsum256(v, sh);
  if (threadIdx.x == 0) a.part[(l * 3 + slot) * NPB3 + blockIdx.x] = t;
}
// the sum of a component's n partial sums, the same bits in every block
__device__ inline double part_sum3(const Cg3Args& a, int l, int slot, int n, double* sh) {
  const double* p = a.part + (l * 3 + slot) * NPB3;
  double t[NPB3 / 256], v = 0.0;
#pragma unroll
  for (int q = 0; q < NPB3 / 256; q++) {  // (no branch: all loads on their way at once)
    const int b = threadIdx.x + 256 * q;
    t[q] = p[b < n ? b : 0];
  }
#pragma unroll
  for (int q = 0; q < NPB3 / 256; q++) v += threadIdx.x + 256 * q < n ? t[q] : 0.0;
  return bsum256(v, sh);
}

// gkl (field.f90:128-158), b = f5 gkl, the warm start phi = df(l),
// r = b + phi(k-1) + phi(j-1) + phi(i-1) - f4 phi + phi(i+1) + phi(j+1) +
// phi(k+1), sums b^2 and r^2; in parity mode b and p = r are stored as well
template <bool PARITY>
__global__ __launch_bounds__(256) void k_cg3_init(Cg3Args a) {
  __shared__ double sh[4];
  const Grid3D& g = a.g;
  const size_t n = (size_t)g.nx * g.ny * g.nz, pl = plane3(g);
  const double *U1 = a.uf, *U2 = a.uf + pl, *U3 = a.uf + 2 * pl, *U4 = a.uf + 3 * pl, *U5 = a.uf + 4 * pl,
               *U6 = a.uf + 5 * pl;
  const double *J1 = a.uj, *J2 = a.uj + pl, *J3 = a.uj + 2 * pl;
  const double f1 = g.f1, f2 = g.f2, f3 = g.f3, f4 = g.f4, f5 = g.f5;
  double sb[3] = {0.0, 0.0, 0.0}, sr[3] = {0.0, 0.0, 0.0};
  for (size_t q = blockIdx.x * 256 + threadIdx.x; q < n; q += (size_t)a.nb0 * 256) {
    int i, j, k;
    decode3(g, q, i, j, k);
#define F(P, ii, jj, kk) P[fidx3(g, ii, jj, kk)]
    const double gk1 = +f2 * (+F(U1, i, j, k - 1) + F(U1, i, j - 1, k) + F(U1, i - 1, j, k) - 6e0 * F(U1, i, j, k) +
                              F(U1, i + 1, j, k) + F(U1, i, j + 1, k) + F(U1, i, j, k + 1) +
                              f3 * (-F(J3, i, j - 1, k) + F(J3, i, j, k) + F(J2, i, j, k - 1) - F(J2, i, j, k))) -
                       f1 * (-F(U6, i, j - 1, k) + F(U6, i, j, k) + F(U5, i, j, k - 1) - F(U5, i, j, k));
    const double gk2 = +f2 * (+F(U2, i, j, k - 1) + F(U2, i, j - 1, k) + F(U2, i - 1, j, k) - 6e0 * F(U2, i, j, k) +
                              F(U2, i + 1, j, k) + F(U2, i, j + 1, k) + F(U2, i, j, k + 1) +
                              f3 * (-F(J1, i, j, k - 1) + F(J1, i, j, k) + F(J3, i - 1, j, k) - F(J3, i, j, k))) -
                       f1 * (-F(U4, i, j, k - 1) + F(U4, i, j, k) + F(U6, i - 1, j, k) - F(U6, i, j, k));
    const double gk3 = +f2 * (+F(U3, i, j, k - 1) + F(U3, i, j - 1, k) + F(U3, i - 1, j, k) - 6e0 * F(U3, i, j, k) +
                              F(U3, i + 1, j, k) + F(U3, i, j + 1, k) + F(U3, i, j, k + 1) +
                              f3 * (-F(J2, i - 1, j, k) + F(J2, i, j, k) + F(J1, i, j - 1, k) - F(J1, i, j, k))) -
                       f1 * (-F(U5, i - 1, j, k) + F(U5, i, j, k) + F(U4, i, j - 1, k) - F(U4, i, j, k));
#undef F
    const double gk[3] = {gk1, gk2, gk3};
    // the cell and its neighbours' periodic images in the field planes
    const size_t f = fidx3(g, i, j, k), sy = (size_t)g.fw, sz = (size_t)g.fw * g.fh;
    const size_t fw = i == g.nxgs ? f + (g.nx - 1) : f - 1, fe = i == g.nxge ? f - (g.nx - 1) : f + 1;
    const size_t fs = j == g.nys ? f + sy * (g.ny - 1) : f - sy, fn = j == g.nye ? f - sy * (g.ny - 1) : f + sy;
    const size_t fb = k == g.nzs ? f + sz * (g.nz - 1) : f - sz, ft = k == g.nze ? f - sz * (g.nz - 1) : f + sz;
#pragma unroll
    for (int l = 0; l < 3; l++) {
      const double* ph = a.df + pl * l;
      const double bv = f5 * gk[l], pc = ph[f];
      const double rv = bv + ph[fb] + ph[fs] + ph[fw] - f4 * pc + ph[fe] + ph[fn] + ph[ft];
      a.phi[(size_t)l * n + q] = pc;
      a.r[(size_t)l * n + q] = rv;
      if (PARITY) {
        a.b[(size_t)l * n + q] = bv;
        a.pold[(size_t)l * n + q] = rv;
      }
      sb[l] = sb[l] + bv * bv;
      sr[l] = sr[l] + rv * rv;
    }
  }
  if (!PARITY) {
    for (int l = 0; l < 3; l++) {
      put_part3(a, l, S_BB, sb[l], sh);
      put_part3(a, l, S_RR, sr[l], sh);
    }
  }
}

// Parity mode's scalars, from serial sums, one wave a component: sum_g = |b|^2, eps =
// sqrt(sum_g)*err (field.f90:454-456), sumr_g, the loop's first test
__global__ __launch_bounds__(64) void k_cg3_parity0(Cg3Args a) {
  const int l = blockIdx.x;
  const size_t n = (size_t)a.g.nx * a.g.ny * a.g.nz;
  const double *b = a.b + (size_t)l * n, *r = a.r + (size_t)l * n;
  const double bb = serial_dot(b, b, n), rr = serial_dot(r, r, n);
  if (threadIdx.x) return;
  CgScal& c = a.sc[l];
  c.sum_g = bb;
  c.eps = sqrt(c.sum_g) * a.g.cg_err;
  c.sumr_g = rr;
  c.ite = 0;
  c.bv = 0.0;
  c.active = (sqrt(c.sumr_g) > c.eps) && (c.sum_g > c.eps);
}

__global__ __launch_bounds__(64) void k_cg3_parity_a(Cg3Args a) {
  const int l = blockIdx.x;
  CgScal& c = a.sc[l];
  if (!c.active) return;
  const size_t n = (size_t)a.g.nx * a.g.ny * a.g.nz;
  const double *r = a.r + (size_t)l * n, *p = a.pnew + (size_t)l * n, *ap = a.ap + (size_t)l * n;
  const double rr = serial_dot(r, r, n), pap = serial_dot(p, ap, n);
  if (threadIdx.x) return;
  c.sumr_g = rr;
  c.sum2_g = pap;
  c.av = c.sumr_g / c.sum2_g;
  c.ite = c.ite + 1;
  c.sum_g = sqrt(c.sumr_g);
}

__global__ __launch_bounds__(64) void k_cg3_parity_b(Cg3Args a) {
  const int l = blockIdx.x;
  CgScal& c = a.sc[l];
  if (!c.active) return;
  if (c.ite >= 100) {
    if (threadIdx.x == 0) {
      atomicOr(a.err, ERR_CG);
      c.active = 0;
    }
    return;
  }
  const size_t n = (size_t)a.g.nx * a.g.ny * a.g.nz;
  const double* r = a.r + (size_t)l * n;
  const double rr = serial_dot(r, r, n);
  if (threadIdx.x) return;
  c.bv = rr / c.sumr_g;
  c.active = c.sum_g > c.eps;
}

// The nodes of one component in the blocks' own order: a block marches a tile
// of 32 x 8 columns through a slab of z levels; the values at levels k-1, k,
// k+1 of a column stay in registers, level k of the tile (with its one-column
// halo) goes through LDS, so that each is read from HBM once per node.  What
// the next level needs is loaded before the current one is combined, and two
// LDS buffers leave one barrier a level.  The work units (tile, slab) are
// dealt to the nb blocks.  `load(m)` gives node m's raw words and `val` its
// value p from them; `pre(q)` loads what `node(q, p, ap, words)` needs of its
// own, ap being f4 p - the sum of the six neighbours, the per-node expression
// of the reference's order (:483-505).  `scal()` runs after the first loads are
// on their way, by all of the block, and says whether to go on (every block has
// a unit).
constexpr int TXC3 = 32, TYC3 = 8;
struct Slabs3 {
  int ntx, ntile, len, units;
};
__host__ __device__ inline Slabs3 slabs3(const Grid3D& g) {
  Slabs3 s;
  s.ntx = (g.nx + TXC3 - 1) / TXC3;
  s.ntile = s.ntx * ((g.ny + TYC3 - 1) / TYC3);
  int nsl = NPB3 / s.ntile;
  if (nsl < 1) nsl = 1;
  if (nsl > g.nz) nsl = g.nz;
  s.len = (g.nz + nsl - 1) / nsl;
  s.units = s.ntile * ((g.nz + s.len - 1) / s.len);
  return s;
}
constexpr int SM3 = (TYC3 + 2) * (TXC3 + 2);
template <class Load, class Val, class Pre, class Node, class Scal>
__device__ inline void march3(const Grid3D& g, int nb, double (*sm)[SM3], Load load, Val val, Pre pre, Node node,
                              Scal scal) {
  constexpr int TXC = TXC3, TYC = TYC3, SW3 = TXC + 2;
  const double f4 = g.f4;
  const Slabs3 S = slabs3(g);
  const int tx = threadIdx.x % TXC, ty = threadIdx.x / TXC;
  const int so = (ty + 1) * SW3 + tx + 1;
  const size_t np = (size_t)g.nx * g.ny;
  int par = 0;  // alternates over levels and units
  for (int u = blockIdx.x; u < S.units; u += nb) {
    const int sl = u / S.ntile, t = u - sl * S.ntile;
    const int k0 = sl * S.len, k1 = k0 + S.len - 1 < g.nz ? k0 + S.len - 1 : g.nz - 1;
    const int i = (t % S.ntx) * TXC + tx, j = (t / S.ntx) * TYC + ty;
    const bool act = i < g.nx && j < g.ny;
    const bool bw = act && tx == 0, be = act && (tx == TXC - 1 || i == g.nx - 1);
    const bool bs = act && ty == 0, bn = act && (ty == TYC - 1 || j == g.ny - 1);
    // the column, and the ones whose values this thread adds to the halo
    const int c = act ? i + g.nx * j : 0;
    const int cw = i == 0 ? c + g.nx - 1 : c - 1, ce = i == g.nx - 1 ? c - (g.nx - 1) : c + 1;
    const int cs = j == 0 ? c + g.nx * (g.ny - 1) : c - g.nx, cn = j == g.ny - 1 ? c - g.nx * (g.ny - 1) : c + g.nx;
    auto lev = [&](int k) { return np * (size_t)(k < 0 ? g.nz - 1 : (k >= g.nz ? k - g.nz : k)); };
    decltype(load(0)) rB{}, rC{}, rT{}, hw{}, he{}, hs{}, hn{};
    decltype(pre(0)) own{};
    {
      const size_t z = lev(k0);
      if (act) {
        rB = load(c + lev(k0 - 1));
        rC = load(c + z);
        rT = load(c + lev(k0 + 1));
        own = pre(c + z);
      }
      if (bw) hw = load(cw + z);
      if (be) he = load(ce + z);
      if (bs) hs = load(cs + z);
      if (bn) hn = load(cn + z);
    }
    if (u == (int)blockIdx.x && !scal()) return;
    double pB = val(rB), pC = val(rC);
    for (int k = k0; k <= k1; k++, par ^= 1) {
      double* const s = sm[par] + so;
      if (act) s[0] = pC;
      if (bw) s[-1] = val(hw);
      if (be) s[1] = val(he);
      if (bs) s[-SW3] = val(hs);
      if (bn) s[SW3] = val(hn);
      const double pT = val(rT);
      const auto mine = own;
      if (k < k1) {
        const size_t z = lev(k + 1);
        if (act) {
          rT = load(c + lev(k + 2));
          own = pre(c + z);
        }
        if (bw) hw = load(cw + z);
        if (be) he = load(ce + z);
        if (bs) hs = load(cs + z);
        if (bn) hn = load(cn + z);
      }
      __syncthreads();
      if (act)
        node(c + np * (size_t)k, pC, -pB - s[-SW3] - s[-1] + f4 * pC - s[1] - s[SW3] - pT, mine);
      pB = pC;
      pC = pT;
    }
  }
}

// p = r + bv p (the previous iteration's update, fused), ap, sum p.ap
// (:483-505).  Fast mode has two launches an iteration and no stored ap, as in
// 2D: every block of k_cg3_a adds the partial sums of r.r, every block of
// k_cg3_b those of p.ap, in the same order; k_cg3_b forms ap again from p.
//
// What bounds it at 256^3: traffic, 4.6 GB an iteration in 0.86 ms (5.3 TB/s, a
// part of it from the cache behind L2) where the arrays themselves are 3.2 GB:
// a 32-column tile reads whole lines for its one-column halos.  On small grids
// the launches, as in 2D.  A whole solve of 8 iterations with its right-hand side, next to the sort
// on the other stream: 67x45x38 365 -> 212 us, 64^3 430 -> 286, 160x144x128
// 2.19 -> 1.69 ms, 256^3 11.8 -> 8.5.  Without the loads ahead of the level in
// work and with two barriers a level the new form was no faster than the old.
template <bool PARITY>
__global__ __launch_bounds__(256) void k_cg3_a(Cg3Args a) {
  __shared__ double sh[4];
  __shared__ double sm[2][SM3];
  const int l = blockIdx.y;
  const Grid3D& g = a.g;
  const size_t n = (size_t)g.nx * g.ny * g.nz;
  const bool first = !PARITY && a.first;
  const double *r = a.r + (size_t)l * n, *po = a.pold + (size_t)l * n;
  double *pn = a.pnew + (size_t)l * n, *ap = a.ap + (size_t)l * n;
  double bv = 0.0, s = 0.0;
  bool go = false;
  auto scal = [&]() -> bool {
    if (PARITY) {
      bv = a.sc[l].bv;
      return a.sc[l].active;
    }
    const CgScal c = a.sp[l];
    const double rr = part_sum3(a, l, S_RR, first ? a.nb0 : a.nb, sh);
    double sum_g = c.sum_g, eps = c.eps;
    int active, ite = c.ite;
    if (first) {
      sum_g = part_sum3(a, l, S_BB, a.nb0, sh);
      eps = sqrt(sum_g) * g.cg_err;
      active = sqrt(rr) > eps && sum_g > eps;
      ite = 0;
    } else {
      active = c.active && sqrt(c.sumr_g) > eps;
      bv = rr / c.sumr_g;
    }
    const double sumr = active ? rr : c.sumr_g;
    if (active) ite++;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      CgScal& o = a.sc[l];
      o.sum_g = sum_g;
      o.eps = eps;
      o.sumr_g = sumr;
      o.ite = ite;
      o.active = active;
      if (a.poll) {
        // (the host's own memory: past the caches, no fence needed)
        const int more = active && sqrt(sumr) > eps;
        __hip_atomic_store(&a.poll->more[l], more, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&a.poll->ite[l], ite, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (l == 0) __hip_atomic_store(&a.poll->err, *a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
    go = active;
    return go;
  };
  struct None {};
  auto pre = [](size_t) { return None{}; };
  auto node = [&](size_t q, double pC, double av, None) {
    pn[q] = pC;
    if (PARITY) ap[q] = av;
    s = s + pC * av;
  };
  if (first)
    march3(g, a.nb, sm, [&](size_t m) { return r[m]; }, [](double v) { return v; }, pre, node, scal);
  else
    march3(g, a.nb, sm, [&](size_t m) { return make_double2(r[m], po[m]); },
           [&](double2 v) { return v.x + bv * v.y; }, pre, node, scal);
  if (go) put_part3(a, l, S_PAP, s, sh);
}

// phi += av p; r -= av ap; sum r^2 (:507-530)
template <bool PARITY>
__global__ __launch_bounds__(256) void k_cg3_b(Cg3Args a) {
  __shared__ double sh[4];
  __shared__ double sm[2][PARITY ? 1 : SM3];
  const int l = blockIdx.y;
  if (!a.sc[l].active) return;
  const Grid3D& g = a.g;
  const size_t n = (size_t)g.nx * g.ny * g.nz;
  double *ph = a.phi + (size_t)l * n, *r = a.r + (size_t)l * n;
  const double *p = a.pnew + (size_t)l * n, *ap = a.ap + (size_t)l * n;
  if constexpr (PARITY) {
    const double av = a.sc[l].av;
    for (size_t q = blockIdx.x * 256 + threadIdx.x; q < n; q += (size_t)a.nb * 256) {
      ph[q] = ph[q] + av * p[q];
      r[q] = r[q] - av * ap[q];
    }
  } else {
    double av = 0.0, s = 0.0;
    march3(g, a.nb, sm, [&](size_t m) { return p[m]; }, [](double v) { return v; },
           [&](size_t q) { return make_double2(ph[q], r[q]); },
           [&](size_t q, double pC, double apq, double2 v) {
             ph[q] = v.x + av * pC;
             const double rv = v.y - av * apq;
             r[q] = rv;
             s = s + rv * rv;
           },
           [&]() {
             av = a.sc[l].sumr_g / part_sum3(a, l, S_PAP, a.nb, sh);
             return true;
           });
    put_part3(a, l, S_RR, s, sh);
  }
}

// The CG's result, the E update (field.f90:164-187) and the increments' ghosts
// (boundary_periodic__dfield, 3d/common/boundary_periodic.f90:458-673) in two
// passes: df on the interior, from phi (whose periodic image is the ghost the
// boundary routine would have filled); then every ghost of df from its image
// and uf += df.
__global__ void k_e3_update(Cg3Args a) {
  const Grid3D& g = a.g;
  const size_t n = (size_t)g.nx * g.ny * g.nz;
  const size_t q = tid1();
  if (q >= n) return;
  int i, j, k;
  decode3(g, q, i, j, k);
  const size_t pl = plane3(g), f = fidx3(g, i, j, k);
  const size_t e = i == g.nxge ? q - (g.nx - 1) : q + 1;
  const size_t no = j == g.nye ? q - (size_t)g.nx * (g.ny - 1) : q + g.nx;
  const size_t up = k == g.nze ? q - (size_t)g.nx * g.ny * (g.nz - 1) : q + (size_t)g.nx * g.ny;
  const size_t fe = f + 1, fn = f + g.fw, ft = f + (size_t)g.fw * g.fh;
  const double f1 = g.f1, gfac = g.gfac, pdt = g.pi4dt;
  const double *P1 = a.phi, *P2 = a.phi + n, *P3 = a.phi + 2 * n;
  const double *U1 = a.uf, *U2 = a.uf + pl, *U3 = a.uf + 2 * pl;
  const double b1 = P1[q], b2 = P2[q], b3 = P3[q], u1 = U1[f], u2 = U2[f], u3 = U3[f];
  double* d = a.df + f;
  d[0] = b1;
  d[pl] = b2;
  d[2 * pl] = b3;
  d[3 * pl] = +f1 * (+gfac * (-b3 + P3[no] + b2 - P2[up]) + (-u3 + U3[fn] + u2 - U2[ft])) - pdt * a.uj[f];
  d[4 * pl] = +f1 * (+gfac * (-b1 + P1[up] + b3 - P3[e]) + (-u1 + U1[ft] + u3 - U3[fe])) - pdt * a.uj[pl + f];
  d[5 * pl] = +f1 * (+gfac * (-b2 + P2[e] + b1 - P1[no]) + (-u2 + U2[fe] + u1 - U1[fn])) - pdt * a.uj[2 * pl + f];
}

__global__ void k_add3(Grid3D g, double* __restrict__ uf, double* __restrict__ df) {
  const size_t pl = plane3(g);
  const size_t q = tid1();
  if (q >= pl) return;
  const unsigned qq = (unsigned)q, row = qq / (unsigned)g.fw;
  int i = g.nxgs - 2 + (int)(qq - row * g.fw), j = g.nys - 2 + (int)(row % (unsigned)g.fh),
      k = g.nzs - 2 + (int)(row / (unsigned)g.fh);
  i = i < g.nxgs ? i + g.nx : (i > g.nxge ? i - g.nx : i);
  j = j < g.nys ? j + g.ny : (j > g.nye ? j - g.ny : j);
  k = k < g.nzs ? k + g.nz : (k > g.nze ? k - g.nz : k);
  const size_t src = fidx3(g, i, j, k);
#pragma unroll
  for (int c = 0; c < 6; c++) {
    const double v = df[pl * c + src];
    if (src != q) df[pl * c + q] = v;
    uf[pl * c + q] = uf[pl * c + q] + v;
  }
}

__global__ void k_fill3(double* p, size_t n, double v) {
  for (size_t q = tid1(); q < n; q += (size_t)gridDim.x * blockDim.x) p[q] = v;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static Cg3Args cg3_args(wpic_ctx3d* c) {
  Cg3Args a;
  a.g = c->g;
  a.uf = c->uf;
  a.uj = c->uj;
  a.df = c->df;
  a.phi = c->phi;
  a.pold = c->pa;
  a.pnew = c->pb;
  a.r = c->rr;
  a.b = c->bb;
  a.ap = c->ap;
  a.part = c->part;
  a.sc = a.sp = c->scal;
  a.err = c->err;
  a.poll = nullptr;
  const size_t n = (size_t)c->g.nx * c->g.ny * c->g.nz;
  a.nb0 = (int)((n + 255) / 256 < NPB3 ? (n + 255) / 256 : NPB3);
  const int units = slabs3(c->g).units;
  a.nb = units < NPB3 ? units : NPB3;
  a.first = 0;
  return a;
}

static unsigned grid_n(size_t n) {
  size_t b = (n + 255) / 256;
  if (b > 8192) b = 8192;
  return (unsigned)(b ? b : 1);
}

static unsigned grid_all(size_t n) { return (unsigned)((n + 255) / 256 ? (n + 255) / 256 : 1); }

hipError_t launch_fill3d(wpic_ctx3d* c, double* p, size_t n, double v) {
  hipLaunchKernelGGL(k_fill3, dim3(grid_n(n)), dim3(256), 0, c->st, p, n, v);
  return hipGetLastError();
}

hipError_t launch_curre_bc3d(wpic_ctx3d* c) {
  const Grid3D& g = c->g;
  hipLaunchKernelGGL(k_curre3_yfold, dim3(grid_all(3 * (size_t)g.fw * g.fd)), dim3(256), 0, c->st, g, c->uj);
  hipLaunchKernelGGL(k_curre3_zfold, dim3(grid_all(3 * (size_t)g.fw * g.ny)), dim3(256), 0, c->st, g, c->uj);
  hipLaunchKernelGGL(k_curre3_ycopy, dim3(grid_all(3 * (size_t)g.fw * g.nz)), dim3(256), 0, c->st, g, c->uj);
  hipLaunchKernelGGL(k_curre3_zcopy, dim3(grid_all(3 * (size_t)g.fw * (g.ny + 2))), dim3(256), 0, c->st, g, c->uj);
  hipLaunchKernelGGL(k_curre3_x, dim3(grid_all(3 * (size_t)g.fh * g.fd)), dim3(256), 0, c->st, g, c->uj);
  return hipGetLastError();
}

hipError_t launch_cg_init3d(wpic_ctx3d* c) {
  Cg3Args a = cg3_args(c);
  if (c->mode == WPIC_MODE_PARITY) {
    hipLaunchKernelGGL(k_cg3_init<true>, dim3(a.nb0), dim3(256), 0, c->st, a);
    hipLaunchKernelGGL(k_cg3_parity0, dim3(3), dim3(64), 0, c->st, a);
  } else {
    hipLaunchKernelGGL(k_cg3_init<false>, dim3(a.nb0), dim3(256), 0, c->st, a);
  }
  return hipGetLastError();
}

hipError_t launch_cg_iter3d(wpic_ctx3d* c, int it, bool poll) {
  Cg3Args a = cg3_args(c);
  if (it & 1) {
    a.pold = c->pb;
    a.pnew = c->pa;
  }
  const dim3 grid(a.nb, 3);
  if (c->mode == WPIC_MODE_PARITY) {
    hipLaunchKernelGGL(k_cg3_a<true>, grid, dim3(256), 0, c->st, a);
    hipLaunchKernelGGL(k_cg3_parity_a, dim3(3), dim3(64), 0, c->st, a);
    hipLaunchKernelGGL(k_cg3_b<true>, grid, dim3(256), 0, c->st, a);
    hipLaunchKernelGGL(k_cg3_parity_b, dim3(3), dim3(64), 0, c->st, a);
    return hipGetLastError();
  }
  a.sc = c->scal + 3 * (it & 1);
  a.sp = c->scal + 3 * (~it & 1);
  a.first = it == 0;
  a.poll = poll ? c->poll : nullptr;
  hipLaunchKernelGGL(k_cg3_a<false>, grid, dim3(256), 0, c->st, a);
  // the host learns how the solve stands while k_cg3_b still runs
  if (poll) {
    const hipError_t e = hipEventRecord(c->ev_poll, c->st);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_cg3_b<false>, grid, dim3(256), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_field_end3d(wpic_ctx3d* c) {
  const Cg3Args a = cg3_args(c);
  hipLaunchKernelGGL(k_e3_update, dim3(grid_all((size_t)c->g.nx * c->g.ny * c->g.nz)), dim3(256), 0, c->st, a);
  hipLaunchKernelGGL(k_add3, dim3(grid_all(plane3(c->g))), dim3(256), 0, c->st, c->g, c->uf, c->df);
  return hipGetLastError();
}

}  // namespace wpic
