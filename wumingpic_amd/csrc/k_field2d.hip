// k_field2d.hip -- implicit FDTD update (Hoshino 2013) of 2d/common/field.f90:
// current ghost folds, the right-hand side gkl (:125-146), the three CG solves
// of cgm (:319-461) run in lock step with per-component stopping, the E update
// (:154-171), the field ghost fills and uf += df (:176-184).
//
// All kernels are coalesced sweeps over x-fastest planes.  Ghost values of the
// CG vectors are not stored: the 5-point stencil maps an out-of-range
// neighbour to the interior value the boundary routine would have copied
// there (boundary_periodic.f90:511-568, boundary_reconnection.f90:505-579),
// with the same sign, so the stencil sees the same bits.
//
// Dot products: fast mode sums fixed per-block partials in a fixed tree
// (deterministic); parity mode sums serially in the reference's (j, i) order.
#include "wpic_internal.h"

namespace wpic {

constexpr double kPi = 3.141592653589793;  // 4.0D0*atan(1.0D0)

// ---------------------------------------------------------------------------
// deterministic block reduction (256 threads), every thread receiving the sum
// ---------------------------------------------------------------------------
__device__ inline double block_sum256(double v, double* sh) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return t;
}

// ---------------------------------------------------------------------------
// current ghost folds at one rank: boundary_periodic.f90:369-506
// ---------------------------------------------------------------------------
__global__ void k_curre_y(Grid2D g, double* uj) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 3 * g.fw) return;
  const int comp = t / g.fw, I = g.nxgs - 2 + t % g.fw;
  double* u = uj + (size_t)g.fw * g.fh * comp;
  const int nys = g.nys, nye = g.nye;
  const double a = u[fidx(g, I, nys - 2)], b = u[fidx(g, I, nys - 1)];
  u[fidx(g, I, nye - 1)] = u[fidx(g, I, nye - 1)] + a;
  u[fidx(g, I, nye)] = u[fidx(g, I, nye)] + b;
  const double c = u[fidx(g, I, nye + 1)], d = u[fidx(g, I, nye + 2)];
  u[fidx(g, I, nys)] = u[fidx(g, I, nys)] + c;
  u[fidx(g, I, nys + 1)] = u[fidx(g, I, nys + 1)] + d;
  u[fidx(g, I, nye + 1)] = u[fidx(g, I, nys)];
  u[fidx(g, I, nye + 2)] = u[fidx(g, I, nys + 1)];
  u[fidx(g, I, nys - 2)] = u[fidx(g, I, nye - 1)];
  u[fidx(g, I, nys - 1)] = u[fidx(g, I, nye)];
}

__global__ void k_curre_x(Grid2D g, double* uj) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 3 * g.fh) return;
  const int comp = t / g.fh, J = g.nys - 2 + t % g.fh;
  double* u = uj + (size_t)g.fw * g.fh * comp;
  const int nxs = g.nxgs, nxe = g.nxge;
  u[fidx(g, nxe - 1, J)] = u[fidx(g, nxe - 1, J)] + u[fidx(g, nxs - 2, J)];
  u[fidx(g, nxe, J)] = u[fidx(g, nxe, J)] + u[fidx(g, nxs - 1, J)];
  u[fidx(g, nxs, J)] = u[fidx(g, nxs, J)] + u[fidx(g, nxe + 1, J)];
  u[fidx(g, nxs + 1, J)] = u[fidx(g, nxs + 1, J)] + u[fidx(g, nxe + 2, J)];
  u[fidx(g, nxs - 2, J)] = u[fidx(g, nxe - 1, J)];
  u[fidx(g, nxs - 1, J)] = u[fidx(g, nxe, J)];
  u[fidx(g, nxe + 1, J)] = u[fidx(g, nxs, J)];
  u[fidx(g, nxe + 2, J)] = u[fidx(g, nxs + 1, J)];
}

// ---------------------------------------------------------------------------
// field ghost fills: boundary_periodic.f90:263-352; walls :350-359 of
// boundary_reconnection.f90
// ---------------------------------------------------------------------------
__global__ void k_dfield_y(Grid2D g, double* df) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 6 * g.nx) return;
  const int comp = t / g.nx, I = g.nxgs + t % g.nx;
  double* d = df + (size_t)g.fw * g.fh * comp;
  const int nys = g.nys, nye = g.nye;
  const double a = d[fidx(g, I, nys)], b = d[fidx(g, I, nys + 1)];
  d[fidx(g, I, nye + 1)] = a;
  d[fidx(g, I, nye + 2)] = b;
  const double c = d[fidx(g, I, nye - 1)], e = d[fidx(g, I, nye)];
  d[fidx(g, I, nys - 2)] = c;
  d[fidx(g, I, nys - 1)] = e;
}

__global__ void k_dfield_x(Grid2D g, double* df) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.fh) return;
  const int J = g.nys - 2 + t;
  const size_t pl = (size_t)g.fw * g.fh;
  const int nxs = g.nxgs, nxe = g.nxge;
  if (g.bc == WPIC_BC_SHOCK) {
    // boundary_shock.f90:395-405: the left wall as the reconnection's, zeros
    // beyond the injection edge
    df[fidx(g, nxs - 1, J)] = -df[fidx(g, nxs, J)];
    for (int c = 1; c <= 3; c++) df[pl * c + fidx(g, nxs - 1, J)] = df[pl * c + fidx(g, nxs + 1, J)];
    for (int c = 4; c <= 5; c++) df[pl * c + fidx(g, nxs - 1, J)] = -df[pl * c + fidx(g, nxs, J)];
    for (int c = 0; c < 6; c++) df[pl * c + fidx(g, nxe + 1, J)] = 0.0;
    return;
  }
  if (g.bc == WPIC_BC_WALLX) {
    double* d1 = df;
    d1[fidx(g, nxs - 1, J)] = -d1[fidx(g, nxs, J)];
    for (int c = 1; c <= 3; c++) df[pl * c + fidx(g, nxs - 1, J)] = df[pl * c + fidx(g, nxs + 1, J)];
    for (int c = 4; c <= 5; c++) df[pl * c + fidx(g, nxs - 1, J)] = -df[pl * c + fidx(g, nxs, J)];
    d1[fidx(g, nxe, J)] = -d1[fidx(g, nxe - 1, J)];
    for (int c = 1; c <= 3; c++) df[pl * c + fidx(g, nxe + 1, J)] = df[pl * c + fidx(g, nxe - 1, J)];
    for (int c = 4; c <= 5; c++) df[pl * c + fidx(g, nxe, J)] = -df[pl * c + fidx(g, nxe - 1, J)];
    return;
  }
  for (int c = 0; c < 6; c++) {
    double* d = df + pl * c;
    d[fidx(g, nxs - 2, J)] = d[fidx(g, nxe - 1, J)];
    d[fidx(g, nxs - 1, J)] = d[fidx(g, nxe, J)];
    d[fidx(g, nxe + 1, J)] = d[fidx(g, nxs, J)];
    d[fidx(g, nxe + 2, J)] = d[fidx(g, nxs + 1, J)];
  }
}

// ---------------------------------------------------------------------------
// CG helpers
// ---------------------------------------------------------------------------
struct CgArgs {
  Grid2D g;
  const double *uf, *uj;
  double* df;
  double *phi, *pold, *pnew, *r, *b, *ap;  // each [3][nx*ny]
  double* part;                            // [3][3][NPB]: per component, see k_cg_a
  CgScal *sc, *sp;                         // this iteration's scalars and the previous one's
  int* err;
  CgPoll* poll;  // where to tell the host how the solve stands (null: not now)
  int nb0, nb;   // blocks (and partial sums) per component of k_cg_init and of an iteration's kernels
  int first;     // the solve's first iteration
};

// where the boundary routine takes the value it puts at (i, j) for component l
// (0..2), and its sign; (i, j) is at most one cell outside the interior, in x
// or in y (sgn = 0: the boundary routine puts a zero there)
__device__ inline void map_ij(const Grid2D& g, int& i, int& j, int l, double& sgn) {
  sgn = 1.0;
  if (j < g.nys) j = g.nye;
  else if (j > g.nye) j = g.nys;
  if (g.bc == WPIC_BC_SHOCK) {
    // boundary_shock.f90:603-621
    if (i < g.nxgs) {
      if (l == 0) { sgn = -1.0; i = g.nxgs; } else i = g.nxgs + 1;
    } else if (i > g.nxge) {
      sgn = 0.0;
      i = g.nxge;
    }
  } else if (g.bc == WPIC_BC_WALLX) {
    if (i < g.nxgs) {
      if (l == 0) { sgn = -1.0; i = g.nxgs; } else i = g.nxgs + 1;
    } else if (i > g.nxge) {
      if (l == 0) { sgn = -1.0; i = g.nxge - 2; } else i = g.nxge - 1;
    }
  } else {
    if (i < g.nxgs) i = g.nxge;
    else if (i > g.nxge) i = g.nxgs;
  }
}

// the ghost value for the sign map_ij returned: v, -v or a +0 zero
__device__ inline double signed_val(double sgn, double v) { return sgn > 0.0 ? v : (sgn < 0.0 ? -v : 0.0); }

// One block's sum of its threads' values, kept as partial sum `slot` of
// component l.
enum { S_RR = 0, S_PAP = 1, S_BB = 2 };  // r.r, p.ap, b.b
__device__ inline void put_part(const CgArgs& a, int l, int slot, double v, double* sh) {
  const double t = block_sum256(v, sh);
  if (threadIdx.x == 0) a.part[(l * 3 + slot) * NPB + blockIdx.x] = t;
}
// the sum of a component's partial sums, the same bits in every block
__device__ inline double part_sum(const CgArgs& a, int l, int slot, int n, double* sh) {
  const double* p = a.part + (l * 3 + slot) * NPB;
  double t[NPB / 256], v = 0.0;
#pragma unroll
  for (int q = 0; q < NPB / 256; q++) {  // (no branch: all loads on their way at once)
    const int b = threadIdx.x + 256 * q;
    t[q] = p[b < n ? b : 0];
  }
#pragma unroll
  for (int q = 0; q < NPB / 256; q++) v += threadIdx.x + 256 * q < n ? t[q] : 0.0;
  return block_sum256(v, sh);
}

// Node (i, j) of component l: b = f5 gkl (field.f90:125-146), the warm start
// phi = df(l) and r = b + (neighbours of phi) - f4 phi (:366-381)
__device__ inline void residual0(const CgArgs& a, int l, int i, int j, double& bv, double& pc, double& rv) {
  const Grid2D& g = a.g;
  const size_t pl = (size_t)g.fw * g.fh;
  const double *U1 = a.uf, *U2 = a.uf + pl, *U3 = a.uf + 2 * pl, *U4 = a.uf + 3 * pl, *U5 = a.uf + 4 * pl,
               *U6 = a.uf + 5 * pl;
  const double *J1 = a.uj, *J2 = a.uj + pl, *J3 = a.uj + 2 * pl;
  const double* df = a.df + pl * l;
  const double f1 = g.f1, f2 = g.f2, f3 = g.f3, f4 = g.f4, f5 = g.f5;
#define F(P, ii, jj) P[fidx(g, ii, jj)]
  double gk;
  if (l == 0)
    gk = +f2 * (+F(U1, i, j - 1) + F(U1, i - 1, j) - 4. * F(U1, i, j) + F(U1, i + 1, j) + F(U1, i, j + 1) +
                f3 * (-F(J3, i, j - 1) + F(J3, i, j))) -
         f1 * (-F(U6, i, j - 1) + F(U6, i, j));
  else if (l == 1)
    gk = +f2 * (+F(U2, i, j - 1) + F(U2, i - 1, j) - 4. * F(U2, i, j) + F(U2, i + 1, j) + F(U2, i, j + 1) -
                f3 * (-F(J3, i - 1, j) + F(J3, i, j))) +
         f1 * (-F(U6, i - 1, j) + F(U6, i, j));
  else
    gk = +f2 * (+F(U3, i, j - 1) + F(U3, i - 1, j) - 4. * F(U3, i, j) + F(U3, i + 1, j) + F(U3, i, j + 1) +
                f3 * (-F(J2, i - 1, j) + F(J2, i, j) + F(J1, i, j - 1) - F(J1, i, j))) -
         f1 * (-F(U5, i - 1, j) + F(U5, i, j) + F(U4, i, j - 1) - F(U4, i, j));
#undef F
  auto ph = [&](int ii, int jj) {
    double sg;
    map_ij(g, ii, jj, l, sg);
    return signed_val(sg, df[fidx(g, ii, jj)]);
  };
  bv = f5 * gk;
  pc = df[fidx(g, i, j)];
  rv = bv + ph(i, j - 1) + ph(i - 1, j) - f4 * pc + ph(i + 1, j) + ph(i, j + 1);
}

// phi, r and the sums b^2 and r^2; in parity mode b and p = r are stored as
// well.  Component l = blockIdx.y.
template <bool PARITY>
__global__ __launch_bounds__(256) void k_cg_init(CgArgs a) {
  __shared__ double sh[4];
  const Grid2D& g = a.g;
  const int n = g.nx * g.ny, l = blockIdx.y;
  double sb = 0.0, sr = 0.0;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += a.nb0 * 256) {
    double bv, pc, rv;
    residual0(a, l, g.nxgs + k % g.nx, g.nys + k / g.nx, bv, pc, rv);
    const size_t q = (size_t)l * n + k;
    a.phi[q] = pc;
    a.r[q] = rv;
    if (PARITY) {
      a.b[q] = bv;
      a.pold[q] = rv;
    }
    sb = sb + bv * bv;
    sr = sr + rv * rv;
  }
  if (!PARITY) {
    put_part(a, l, S_BB, sb, sh);
    put_part(a, l, S_RR, sr, sh);
  }
}

// how component l stands, into the host's own memory: past the caches, no fence needed
__device__ inline void tell_host(const CgArgs& a, int l, int more, int ite) {
  __hip_atomic_store(&a.poll->more[l], more, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&a.poll->ite[l], ite, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (l == 0) __hip_atomic_store(&a.poll->err, *a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Parity mode's scalars, from serial sums over the interior in (j, i) order,
// one wave a component.

// sum_g = |b|^2, eps = sqrt(sum_g)*err (field.f90:351-364), sumr_g; enter the
// loop iff sqrt(sumr_g) > eps and sum_g > eps (:383-387)
__global__ __launch_bounds__(64) void k_cg_parity0(CgArgs a) {
  const int l = blockIdx.x, n = a.g.nx * a.g.ny;
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

// av = sumr_g / sum2_g (:409-415); sum_g = sqrt(sumr_g) (:426)
__global__ __launch_bounds__(64) void k_cg_parity_a(CgArgs a) {
  const int l = blockIdx.x, n = a.g.nx * a.g.ny;
  CgScal& c = a.sc[l];
  if (!c.active) return;
  const double *r = a.r + (size_t)l * n, *p = a.pnew + (size_t)l * n, *ap = a.ap + (size_t)l * n;
  const double rr = serial_dot(r, r, n), pap = serial_dot(p, ap, n);
  if (threadIdx.x) return;
  c.sumr_g = rr;
  c.sum2_g = pap;
  c.av = c.sumr_g / c.sum2_g;
  c.ite = c.ite + 1;
  c.sum_g = sqrt(c.sumr_g);
}

// ite >= ite_max stops (:427-430); bv = sum1/sumr_g (:441-442); loop test
__global__ __launch_bounds__(64) void k_cg_parity_b(CgArgs a) {
  const int l = blockIdx.x, n = a.g.nx * a.g.ny;
  CgScal& c = a.sc[l];
  if (!c.active) return;
  if (c.ite >= 100) {
    if (threadIdx.x == 0) {
      atomicOr(a.err, ERR_CG);
      c.active = 0;
    }
    return;
  }
  const double* r = a.r + (size_t)l * n;
  const double rr = serial_dot(r, r, n);
  if (threadIdx.x) return;
  c.bv = rr / c.sumr_g;
  c.active = c.sum_g > c.eps;
}

// The nodes of one component: each wave marches 64 columns through a few rows.
// The values of a column at rows j-1, j, j+1 stay in registers and those of the
// neighbouring columns come from the neighbouring lanes (beyond the strip or
// the box from memory), so that a row is read once per strip; the next row's
// words are in flight while one is combined, and no barrier ties the waves
// together.  `load(m)` gives node m's raw words and `val` its value p; `pre(q)`
// loads what `node(q, p, ap, words)` needs of its own, ap being f4 p - the sum
// of the four neighbours.  `scal()` runs after the first loads are on their
// way, by all of the block, and says whether to go on.
template <class Load, class Val, class Pre, class Node, class Scal>
__device__ inline void march2(const Grid2D& g, int nb, int l, Load load, Val val, Pre pre, Node node, Scal scal) {
  constexpr int WAVE_SHL1 = 0x130, WAVE_SHR1 = 0x138;  // from the lane above, below
  const double f4 = g.f4;
  const Strips2 S = strips2(g);
  const int lane = threadIdx.x & 63;
  const int w0 = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  bool go = true, first = true;
  for (int u = w0; first || u < S.units; u += nb * 4) {
    const bool some = u < S.units;
    const int i = g.nxgs + (some ? u % S.ntx : 0) * 64 + lane;
    const int j0 = g.nys + (some ? u / S.ntx : 0) * S.len;
    const int j1 = !some ? j0 - 1 : (j0 + S.len - 1 < g.nye ? j0 + S.len - 1 : g.nye);
    const bool act = some && i <= g.nxge;
    const bool bw = act && (lane == 0 || i == g.nxgs), be = act && (lane == 63 || i == g.nxge);
    // the columns west and east, where the boundary takes them from, and their sign
    double sw = 1.0, se = 1.0;
    int iw = i - 1, ie = i + 1, jj = j0;
    map_ij(g, iw, jj, l, sw);
    map_ij(g, ie, jj, l, se);
    auto at = [&](int ii, int j) { return cidx(g, ii, j < g.nys ? g.nye : (j > g.nye ? g.nys : j)); };
    decltype(load(0)) rB{}, rC{}, rT{}, hw{}, he{};
    decltype(pre(0)) own{};
    if (act) {
      rB = load(at(i, j0 - 1));
      rC = load(at(i, j0));
      rT = load(at(i, j0 + 1));
      own = pre(at(i, j0));
    }
    if (bw) hw = load(at(iw, j0));
    if (be) he = load(at(ie, j0));
    if (first) go = scal();
    first = false;
    if (!go) return;
    double pB = val(rB), pC = val(rC);
    for (int j = j0; j <= j1; j++) {
      const double pT = val(rT);
      const double hwv = val(hw), hev = val(he);
      const auto mine = own;
      if (j < j1) {
        if (act) {
          rT = load(at(i, j + 2));
          own = pre(at(i, j + 1));
        }
        if (bw) hw = load(at(iw, j + 1));
        if (be) he = load(at(ie, j + 1));
      }
      double pW = dpp_f64<WAVE_SHR1>(pC), pE = dpp_f64<WAVE_SHL1>(pC);
      if (bw) pW = signed_val(sw, hwv);
      if (be) pE = signed_val(se, hev);
      if (act) node(cidx(g, i, j), pC, -pB - pW + f4 * pC - pE - pT, mine);
      pB = pC;
      pC = pT;
    }
  }
}

// p = r + bv p (previous iteration's :444-450, fused here), then
// ap = f4 p - sum of neighbours; sum p.ap (:391-407).
//
// Fast mode has two launches an iteration, not four: every block of k_cg_a
// adds the partial sums of r.r that k_cg_init or k_cg_b left, every block of
// k_cg_b those of p.ap, in the same order, so that all see the same scalars
// (k_cg_a keeps them in sc, reading the previous iteration's from sp: the two
// alternate).  ap is not stored: k_cg_b forms it again from p, one array less
// each way.
//
// What bounds it: on a small grid the launches and the chain of dependent
// memory round trips in each (so the first loads go out before the partial
// sums are awaited, and those are all read at once); on a large one the memory
// behind L2.  A whole solve of 7 to 9 iterations, with its right-hand side:
// 64x64 164 -> 79 us, 250x187 183 -> 102, 1024x1024 1.31 -> 1.13 ms,
// 1024x2048 with walls 1.24 -> 0.83 ms.  (One launch for a whole solve in one
// workgroup per component, p in LDS, took 72 us at 64x64 and left the step's
// time as it was.)
template <bool PARITY>
__global__ __launch_bounds__(256) void k_cg_a(CgArgs a) {
  __shared__ double sh[4];
  const int l = blockIdx.y;
  const Grid2D& g = a.g;
  const int n = g.nx * g.ny;
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
    const double rr = part_sum(a, l, S_RR, first ? a.nb0 : a.nb, sh);
    double sum_g = c.sum_g, eps = c.eps;
    int active, ite = c.ite;
    if (first) {
      sum_g = part_sum(a, l, S_BB, a.nb0, sh);
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
      if (a.poll) tell_host(a, l, active && sqrt(sumr) > eps, ite);
    }
    go = active;
    return go;
  };
  struct None {};
  auto pre = [](int) { return None{}; };
  auto node = [&](int q, double pC, double av, None) {
    pn[q] = pC;
    if (PARITY) ap[q] = av;
    s = s + pC * av;
  };
  if (first)
    march2(g, a.nb, l, [&](int m) { return r[m]; }, [](double v) { return v; }, pre, node, scal);
  else
    march2(g, a.nb, l, [&](int m) { return make_double2(r[m], po[m]); },
           [&](double2 v) { return v.x + bv * v.y; }, pre, node, scal);
  if (go) put_part(a, l, S_PAP, s, sh);
}

// phi += av p; r -= av ap (:417-424); sum r^2 (:432-439)
template <bool PARITY>
__global__ __launch_bounds__(256) void k_cg_b(CgArgs a) {
  __shared__ double sh[4];
  const int l = blockIdx.y;
  if (!a.sc[l].active) return;
  const Grid2D& g = a.g;
  const int n = g.nx * g.ny;
  double *ph = a.phi + (size_t)l * n, *r = a.r + (size_t)l * n;
  const double *pn = a.pnew + (size_t)l * n, *ap = a.ap + (size_t)l * n;
  if constexpr (PARITY) {
    const double av = a.sc[l].av;
    for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += a.nb * 256) {
      ph[k] = ph[k] + av * pn[k];
      r[k] = r[k] - av * ap[k];
    }
  } else {
    double av = 0.0, s = 0.0;
    march2(g, a.nb, l, [&](int m) { return pn[m]; }, [](double v) { return v; },
           [&](int q) { return make_double2(ph[q], r[q]); },
           [&](int q, double pC, double apq, double2 v) {
             ph[q] = v.x + av * pC;
             const double rv = v.y - av * apq;
             r[q] = rv;
             s = s + rv * rv;
           },
           [&]() {
             av = a.sc[l].sumr_g / part_sum(a, l, S_PAP, a.nb, sh);
             return true;
           });
    put_part(a, l, S_RR, s, sh);
  }
}

// Periodic box: the CG's result, the E update and the increments' ghosts in
// two passes instead of seven launches.  First df on the interior, from phi
// (whose periodic image is the ghost that boundary_periodic__dfield would have
// filled); then every ghost of df from its image and uf += df.
__device__ inline int wrap1(int i, int lo, int hi, int n) { return i < lo ? i + n : (i > hi ? i - n : i); }

__global__ void k_field_e_periodic(CgArgs a) {
  const Grid2D& g = a.g;
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const int e = cidx(g, i == g.nxge ? g.nxgs : i + 1, j), no = cidx(g, i, j == g.nye ? g.nys : j + 1);
  const size_t pl = (size_t)g.fw * g.fh;
  const int f = fidx(g, i, j), fe = f + 1, fn = f + g.fw;
  const double f1 = g.f1, gfac = g.gfac, pdt = g.pi4dt;
  const double *P1 = a.phi, *P2 = a.phi + n, *P3 = a.phi + 2 * (size_t)n;
  const double *U1 = a.uf, *U2 = a.uf + pl, *U3 = a.uf + 2 * pl;
  double* d = a.df + f;
  const double b1 = P1[k], b2 = P2[k], b3 = P3[k];
  d[0] = b1;
  d[pl] = b2;
  d[2 * pl] = b3;
  d[3 * pl] = +f1 * (+gfac * (-b3 + P3[no]) + (-U3[f] + U3[fn])) - pdt * a.uj[f];
  d[4 * pl] = -f1 * (+gfac * (-b3 + P3[e]) + (-U3[f] + U3[fe])) - pdt * a.uj[pl + f];
  d[5 * pl] = +f1 * (+gfac * (-b2 + P2[e] + b1 - P1[no]) + (-U2[f] + U2[fe] + U1[f] - U1[fn])) - pdt * a.uj[2 * pl + f];
}

__global__ void k_field_add_periodic(Grid2D g, double* __restrict__ uf, double* __restrict__ df) {
  const int pl = g.fw * g.fh;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= pl) return;
  const int I = g.nxgs - 2 + k % g.fw, J = g.nys - 2 + k / g.fw;
  const int src = fidx(g, wrap1(I, g.nxgs, g.nxge, g.nx), wrap1(J, g.nys, g.nye, g.ny));
#pragma unroll
  for (int c = 0; c < 6; c++) {
    const size_t o = (size_t)pl * c;
    const double v = df[o + src];
    if (src != k) df[o + k] = v;
    uf[o + k] = uf[o + k] + v;
  }
}

// db(l, interior) = phi (:455-457)
__global__ void k_cg_store(CgArgs a) {
  const Grid2D& g = a.g;
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const size_t pl = (size_t)g.fw * g.fh;
  for (int l = 0; l < 3; l++) a.df[pl * l + fidx(g, i, j)] = a.phi[(size_t)l * n + k];
}

// E update (field.f90:154-171)
__global__ void k_e_update(Grid2D g, const double* __restrict__ uf, const double* __restrict__ uj,
                           double* __restrict__ df) {
  const int n = g.nx * g.ny;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = g.nxgs + k % g.nx, j = g.nys + k / g.nx;
  const size_t pl = (size_t)g.fw * g.fh;
  const double f1 = g.f1, gfac = g.gfac, pdt = g.pi4dt;
#define D(c, ii, jj) df[pl * ((c)-1) + fidx(g, ii, jj)]
#define U(c, ii, jj) uf[pl * ((c)-1) + fidx(g, ii, jj)]
#define J(c, ii, jj) uj[pl * ((c)-1) + fidx(g, ii, jj)]
  const double e4 = +f1 * (+gfac * (-D(3, i, j) + D(3, i, j + 1)) + (-U(3, i, j) + U(3, i, j + 1))) - pdt * J(1, i, j);
  const double e5 = -f1 * (+gfac * (-D(3, i, j) + D(3, i + 1, j)) + (-U(3, i, j) + U(3, i + 1, j))) - pdt * J(2, i, j);
  const double e6 = +f1 * (+gfac * (-D(2, i, j) + D(2, i + 1, j) + D(1, i, j) - D(1, i, j + 1)) +
                           (-U(2, i, j) + U(2, i + 1, j) + U(1, i, j) - U(1, i, j + 1))) -
                    pdt * J(3, i, j);
  D(4, i, j) = e4;
  D(5, i, j) = e5;
  D(6, i, j) = e6;
#undef D
#undef U
#undef J
}

__global__ void k_uf_add(size_t n, double* __restrict__ uf, const double* __restrict__ df) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x)
    uf[k] = uf[k] + df[k];
}

// uf += df over columns nxgs-2..nxge+2 of a cut grid (field.f90:176-184 with
// nxe below the planes' edge); the columns beyond keep their values
__global__ void k_uf_add_cols(Grid2D g, double* __restrict__ uf, const double* __restrict__ df) {
  const int w = g.nx + 4;
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t >= (size_t)6 * w * g.fh) return;
  const int i = (int)(t % w);
  const size_t rest = t / w;
  const int J = (int)(rest % g.fh), comp = (int)(rest / g.fh);
  const size_t k = (size_t)g.fw * g.fh * comp + (size_t)g.fw * J + i;
  uf[k] = uf[k] + df[k];
}

__global__ void k_fill(double* p, size_t n, double v) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x) p[k] = v;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// The field solve's grid.  While the shock's box expands the solve spans
// nodes nxgs..nxa (field.f90 runs every loop over nxs..nxe, the CG's vectors
// and sums included, and its boundary routines act at nxe+1): the same grid
// with nx and nxge cut there, over the full-size planes (fidx keeps the
// storage width fw).
static Grid2D field_grid(const wpic_ctx* c) {
  Grid2D g = c->g;
  if (g.nxa != g.nxge) {
    g.nx = g.nxa - g.nxgs + 1;
    g.nxge = g.nxa;
  }
  return g;
}

static CgArgs cg_args(wpic_ctx* c) {
  CgArgs a;
  a.g = field_grid(c);
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
  a.nb0 = cg_blocks(a.g);
  const int nb = (strips2(a.g).units + 3) / 4;
  a.nb = nb < NPB ? nb : NPB;
  a.first = 0;
  return a;
}

static int grid_for(size_t n, int bs = 256) {
  size_t g = (n + bs - 1) / bs;
  if (g > 65535u * 16u) g = 65535u * 16u;
  return (int)(g ? g : 1);
}

hipError_t launch_fill(wpic_ctx* c, double* p, size_t n, double v) {
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n) < 8192 ? grid_for(n) : 8192), dim3(256), 0, c->st, p, n, v);
  return hipGetLastError();
}

hipError_t launch_zero(wpic_ctx* c, double* p, size_t n) { return launch_fill(c, p, n, 0.0); }

// (the y fold runs over every column of the plane: beyond nxa+2 the current
// is zero while the shock's box expands)
hipError_t launch_curre_bc(wpic_ctx* c) {
  hipLaunchKernelGGL(k_curre_y, dim3(grid_for(3 * c->g.fw)), dim3(256), 0, c->st, c->g, c->uj);
  if (c->g.bc == WPIC_BC_PERIODIC)
    hipLaunchKernelGGL(k_curre_x, dim3(grid_for(3 * c->g.fh)), dim3(256), 0, c->st, c->g, c->uj);
  return hipGetLastError();
}

hipError_t launch_dfield_bc(wpic_ctx* c) {
  const Grid2D g = field_grid(c);
  hipLaunchKernelGGL(k_dfield_y, dim3(grid_for(6 * g.nx)), dim3(256), 0, c->st, g, c->df);
  hipLaunchKernelGGL(k_dfield_x, dim3(grid_for(g.fh)), dim3(256), 0, c->st, g, c->df);
  return hipGetLastError();
}

hipError_t launch_cg_init(wpic_ctx* c) {
  CgArgs a = cg_args(c);
  if (c->mode == WPIC_MODE_PARITY) {
    hipLaunchKernelGGL(k_cg_init<true>, dim3(a.nb0, 3), dim3(256), 0, c->st, a);
    hipLaunchKernelGGL(k_cg_parity0, dim3(3), dim3(64), 0, c->st, a);
  } else {
    hipLaunchKernelGGL(k_cg_init<false>, dim3(a.nb0, 3), dim3(256), 0, c->st, a);
  }
  return hipGetLastError();
}

// the solve's scalars after r, its partial sums and b were set elsewhere (the
// adjoint's transposed solves)
hipError_t launch_cg_start(wpic_ctx* c) {
  CgArgs a = cg_args(c);
  if (c->mode == WPIC_MODE_PARITY) hipLaunchKernelGGL(k_cg_parity0, dim3(3), dim3(64), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_cg_iter(wpic_ctx* c, int it, bool poll) {
  CgArgs a = cg_args(c);
  // p alternates between the two buffers: iteration it reads (it even ? pa : pb)
  if (it & 1) {
    a.pold = c->pb;
    a.pnew = c->pa;
  }
  const dim3 grid(a.nb, 3);
  if (c->mode == WPIC_MODE_PARITY) {
    hipLaunchKernelGGL(k_cg_a<true>, grid, dim3(256), 0, c->st, a);
    hipLaunchKernelGGL(k_cg_parity_a, dim3(3), dim3(64), 0, c->st, a);
    hipLaunchKernelGGL(k_cg_b<true>, grid, dim3(256), 0, c->st, a);
    hipLaunchKernelGGL(k_cg_parity_b, dim3(3), dim3(64), 0, c->st, a);
    return hipGetLastError();
  }
  a.sc = c->scal + 3 * (it & 1);
  a.sp = c->scal + 3 * (~it & 1);
  a.first = it == 0;
  a.poll = poll ? c->poll : nullptr;
  hipLaunchKernelGGL(k_cg_a<false>, grid, dim3(256), 0, c->st, a);
  // the host learns how the solve stands while k_cg_b still runs
  if (poll) {
    const hipError_t e = hipEventRecord(c->ev_poll, c->st);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_cg_b<false>, grid, dim3(256), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_field_end_periodic(wpic_ctx* c) {
  CgArgs a = cg_args(c);
  hipLaunchKernelGGL(k_field_e_periodic, dim3(grid_for((size_t)a.g.nx * a.g.ny)), dim3(256), 0, c->st, a);
  hipLaunchKernelGGL(k_field_add_periodic, dim3(grid_for((size_t)a.g.fw * a.g.fh)), dim3(256), 0, c->st, a.g, c->uf,
                     c->df);
  return hipGetLastError();
}

hipError_t launch_cg_store(wpic_ctx* c) {
  CgArgs a = cg_args(c);
  hipLaunchKernelGGL(k_cg_store, dim3(grid_for((size_t)a.g.nx * a.g.ny)), dim3(256), 0, c->st, a);
  return hipGetLastError();
}

hipError_t launch_e_update(wpic_ctx* c) {
  const Grid2D g = field_grid(c);
  hipLaunchKernelGGL(k_e_update, dim3(grid_for((size_t)g.nx * g.ny)), dim3(256), 0, c->st, g, c->uf, c->uj, c->df);
  return hipGetLastError();
}

hipError_t launch_uf_add(wpic_ctx* c) {
  if (c->g.nxa != c->g.nxge) {
    const Grid2D g = field_grid(c);
    const size_t n = (size_t)6 * (g.nx + 4) * g.fh;
    hipLaunchKernelGGL(k_uf_add_cols, dim3(grid_for(n)), dim3(256), 0, c->st, g, c->uf, c->df);
    return hipGetLastError();
  }
  const size_t n = (size_t)6 * c->g.fw * c->g.fh;
  hipLaunchKernelGGL(k_uf_add, dim3(grid_for(n) < 8192 ? grid_for(n) : 8192), dim3(256), 0, c->st, n, c->uf, c->df);
  return hipGetLastError();
}

}  // namespace wpic
