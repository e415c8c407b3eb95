// wpic_internal.h -- device helpers, the context and the kernel launchers of
// the 2D MI355X step loop.  Only the library's own translation units include
// this; the public boundary is include/wpic.h.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/wpic.h"

namespace wpic {

// ---------------------------------------------------------------------------
// Grid and physics constants, passed by value to every kernel.
// Field planes carry the reference's two ghost layers:
// i in nxgs-2..nxge+2, j in nys-2..nye+2, x fastest (coalesced along x).
// ---------------------------------------------------------------------------
struct Grid2D {
  int nx, ny, nxgs, nxge, nygs, nyge, nys, nye;
  int nxa;     // the active right edge node nxe (= nxge; below it while the shock's box expands)
  int fw, fh;  // plane width nx+4 and height ny+4
  int bc, nsp;
  double delx, delt, c, gfac, d_delx, d_delt;
  double f1, f2, f3, f4, f5, pi4dt;  // field.f90:53-57; 4*pi*delt
  double spanx, spany;               // nx*delx, ny*delx rounded down
  double wall_lo, wall_hi;           // 2*(nxs+1)*delx, 2*(nxa-1)*delx
  double u0, xend;                   // WPIC_BC_SHOCK: injection 4-velocity, moving mirror position
  double q[WPIC_MAXSP], r[WPIC_MAXSP];
  long long ncap;                    // particle capacity per species
  double cg_err;                     // CG relative tolerance (field.f90:339: 1e-6)
};

// reflecting x walls: the reconnection's pair, or the shock's left wall and
// injection edge (their current, moment and y boundaries are the same)
__host__ __device__ inline bool walls(const Grid2D& g) { return g.bc != WPIC_BC_PERIODIC; }

__host__ __device__ inline int fidx(const Grid2D& g, int i, int j) {
  return (i - (g.nxgs - 2)) + g.fw * (j - (g.nys - 2));
}
// interior cell index (CG vectors, parity deposit blocks)
__host__ __device__ inline int cidx(const Grid2D& g, int i, int j) {
  return (i - g.nxgs) + g.nx * (j - g.nys);
}

// moments mom(7, nxgs-1:nxge+1, nys-1:nye+1, nsp): the seven moments of a
// node contiguous, as the reference's array
__host__ __device__ inline size_t midx(const Grid2D& g, int i, int j, int s) {
  return (size_t)7 * ((size_t)(i - (g.nxgs - 1)) + (size_t)(g.nx + 2) * ((size_t)(j - (g.nys - 1)) + (size_t)(g.ny + 2) * s));
}

// One field of an array of particle records: record i's value lies i strides
// (in units of T) from the first one's.
template <class T, int STRIDE>
struct Col {
  T* p;
  __host__ __device__ T& operator[](size_t i) const { return p[i * STRIDE]; }
};

// A particle buffer: 48-byte records (x, y, ux, uy, uz, id) one after another,
// the reference's own up(:, ii) layout; the id is raw 64 bits.  A record that
// is read out of slot order (a particle that changed cell or row) then costs
// the one or two cache lines it lies in instead of one line per field, and
// the run of records a lane group reads or writes shares a line with its
// neighbours only at its two ends.  The push reads and writes a record as
// three 16-byte words.
struct Parts {
  Col<double, 6> x, y, ux, uy, uz;
  Col<uint64_t, 6> id;
};
constexpr int PART_DOUBLES = 6;
inline Parts parts_at(double* r) {
  return Parts{{r}, {r + 1}, {r + 2}, {r + 3}, {r + 4}, {reinterpret_cast<uint64_t*>(r + 5)}};
}

struct Rec {
  double x, y, ux, uy, uz;
  uint64_t id;
};
__device__ inline Rec load_rec(const Parts& P, size_t i) {
  const double2* r = reinterpret_cast<const double2*>(P.x.p + PART_DOUBLES * i);
  const double2 a = r[0], b = r[1], c = r[2];
  return Rec{a.x, a.y, b.x, b.y, c.x, (uint64_t)__double_as_longlong(c.y)};
}
__device__ inline void store_rec(const Parts& P, size_t i, const Rec& q) {
  double2* r = reinterpret_cast<double2*>(P.x.p + PART_DOUBLES * i);
  r[0] = make_double2(q.x, q.y);
  r[1] = make_double2(q.ux, q.uy);
  r[2] = make_double2(q.uz, __longlong_as_double((long long)q.id));
}

// mixed-precision particles: 32-byte records of x cell index, FP32 in-cell
// offsets (x - ix and y - row, both in [0, 1)), FP32 momenta and the id, two
// 16-byte words
struct PartsM {
  Col<int, 8> ix;
  Col<float, 8> ox, oy, ux, uy, uz;
  Col<uint64_t, 4> id;
};
constexpr int PARTM_FLOATS = 8;
inline PartsM partsm_at(float* r) {
  return PartsM{{reinterpret_cast<int*>(r)}, {r + 1}, {r + 2}, {r + 3}, {r + 4}, {r + 5},
                {reinterpret_cast<uint64_t*>(r + 6)}};
}

struct RecM {
  int ix;
  float ox, oy, ux, uy, uz;
  uint64_t id;
};
__device__ inline RecM load_rec(const PartsM& P, size_t i) {
  const int4* r = reinterpret_cast<const int4*>(P.ix.p + PARTM_FLOATS * i);
  const int4 a = r[0], b = r[1];
  return RecM{a.x, __int_as_float(a.y), __int_as_float(a.z), __int_as_float(a.w), __int_as_float(b.x),
              __int_as_float(b.y), (uint64_t)(uint32_t)b.z | ((uint64_t)(uint32_t)b.w << 32)};
}
__device__ inline void store_rec(const PartsM& P, size_t i, const RecM& q) {
  int4* r = reinterpret_cast<int4*>(P.ix.p + PARTM_FLOATS * i);
  r[0] = make_int4(q.ix, __float_as_int(q.ox), __float_as_int(q.oy), __float_as_int(q.ux));
  r[1] = make_int4(__float_as_int(q.uy), __float_as_int(q.uz), (int)(uint32_t)q.id, (int)(uint32_t)(q.id >> 32));
}

// an in-cell offset in [0, 1) as FP32: rounding up to 1 is pulled back below
__host__ __device__ inline float to_offset(double f) {
  float o = (float)f;
  if (o >= 1.0f) o = 0x1.fffffep-1f;
  if (o < 0.0f) o = 0.0f;
  return o;
}

// device error bits, OR-ed by kernels and checked by the host at sync points
enum : int { ERR_DOMAIN = 1, ERR_CG = 2, ERR_ROW = 4 };

// ---------------------------------------------------------------------------
// Round-toward-minus-infinity double arithmetic (the periodic particle wraps
// run under ieee_down: boundary_periodic.f90:74,124).  Correctly rounded-down
// results from round-to-nearest operations plus an exact error term.
// ---------------------------------------------------------------------------
__host__ __device__ inline double next_down(double s) {
  long long b;
  __builtin_memcpy(&b, &s, 8);
  if (s > 0.0)
    b -= 1;
  else
    b += 1;
  double r;
  __builtin_memcpy(&r, &b, 8);
  return r;
}

__host__ __device__ inline double rd_add(double a, double b) {
  double s = a + b;
  if (s == 0.0) {
    if (a == 0.0 && b == 0.0 && !__builtin_signbit(a) && !__builtin_signbit(b)) return 0.0;
    return -0.0;
  }
  double bb = s - a;
  double err = (a - (s - bb)) + (b - bb);
  if (err < 0.0) s = next_down(s);
  return s;
}

__host__ __device__ inline double rd_mul(double a, double b) {
  double p = a * b;
  double err = __builtin_fma(a, b, -p);
  if (err < 0.0) p = next_down(p);
  return p;
}

// int(x / delx) of the particle boundaries, under round-down
// (boundary_periodic.f90:74) or round-to-nearest: with delx = 1, the only
// cell width a context accepts (sort__bucket bins by int(x)), the quotient is
// x itself in every rounding mode
__host__ __device__ inline int cell_of(double x) { return (int)x; }

// The x boundary that acts on a pushed particle before the deposit:
// reconnection walls (boundary_reconnection.f90:79-91, WPIC_BC_WALLX) or the
// shock's left wall and the mirror moving with the inflow at xend, which sends
// ux to 2 u0 - ux (boundary_shock__injection, boundary_shock.f90:270-293,
// WPIC_BC_SHOCK).  INJ false gives boundary_shock__particle_x's wall pair.
template <int BC, bool INJ = true>
__host__ __device__ inline void reflect_x(const Grid2D& g, double& x, double& ux, double& uy, double& uz) {
  if (BC == WPIC_BC_PERIODIC) return;
  const int ipos = cell_of(x);
  if (ipos < g.nxgs + 1) {
    x = g.wall_lo - x;
    ux = -ux; uy = -uy; uz = -uz;
  } else if (BC == WPIC_BC_SHOCK && INJ) {
    if (x > g.xend) {
      x = +2. * g.xend - x;
      ux = +2. * g.u0 - ux;
      uy = -uy; uz = -uz;
    }
  } else if (ipos >= g.nxa - 1) {
    x = g.wall_hi - x;
    ux = -ux; uy = -uy; uz = -uz;
  }
}


// quadratic spline with nodes at cell centres (particle.f90:99-107)
__host__ __device__ inline void shape3(double dh, double& s0, double& s1, double& s2) {
  s0 = 0.5 * (0.5 - dh) * (0.5 - dh);
  s1 = 0.75 - dh * dh;
  s2 = 0.5 * (0.5 + dh) * (0.5 + dh);
}

// Two staged cell-centred field components side by side: one 16-byte LDS read
struct alignas(16) FieldPair {
  double a, b;
};

// The correctly rounded square root of x and the correctly rounded reciprocal
// of that root, as sqrt(x) and 1. / sqrt(x) give them.  The compiler's own
// sequences scale against overflow and handle zeros and infinities, twice
// over; for x within 2^-200 .. 2^200 none of that is needed and the
// reciprocal starts from the root's own iterate instead of a new seed.
//   y ~ 1/sqrt(x) from the hardware; g ~ sqrt(x) and h ~ 1/(2 sqrt(x)) refined
//   together by Goldschmidt's iteration, then g corrected twice with the exact
//   residual x - g g (a fused multiply-add), which rounds it correctly; the
//   reciprocal of g from 2 h by one Newton step and one correction with the
//   exact residual 1 - g r (P. Markstein, IBM J. Res. Dev. 34, 111 (1990)).
// That last correction rounds wrongly for one significand of the root, all ones
// (its reciprocal lies just above the middle of two doubles): such roots, told
// by their lower word, take the compiler's sequences as well.
__device__ inline void sqrt_and_inverse(double x, double& root, double& inv) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  e = fma(-g, g, x);
  g = fma(e, h, g);
  e = fma(-g, g, x);
  g = fma(e, h, g);
  double r = h + h;
  e = fma(-g, r, 1.0);
  r = fma(e, r, r);
  e = fma(-g, r, 1.0);
  r = fma(e, r, r);
  root = g;
  inv = r;
  // exponent outside [-200, 200), sign or NaN, or the root's all ones (one branch
  // for the wave: lanes that part here cost the caller's live registers a copy
  // each)
  const bool out = ((unsigned)__double2hiint(x) - 0x33700000u >= 0x19000000u) | (__double2loint(g) == -1);
  if (__builtin_expect(__any(out), 0)) {
    const double q = sqrt(x);
    root = out ? q : g;
    inv = out ? 1. / q : r;
  }
}

// The particles of one cell over all species, as one list: element t is slot
// beg[s] + t - cum[s] of species s, the last s with cum[s] <= t (species
// beyond nsp carry cum = INT_MAX).  Kept as named scalars and resolved with
// masks: a chain of selects over an array is turned by the compiler into an
// indexed table in scratch memory.  Most runs have two species, so the masks
// of the third and fourth sit behind one scalar branch.
struct CellList {
  int o0, d1, d2, d3, c1, c2, c3;  // slot offset of species 0, its steps to 1..3, their first elements
  int ob;                          // the offset of the species set last (building d1..d3)
  __device__ void set(int s, int beg, int cum) {
    const int o = beg - cum;
    if (s == 0) { o0 = o; }
    if (s == 1) { d1 = o - ob; c1 = cum; }
    if (s == 2) { d2 = o - ob; c2 = cum; }
    if (s == 3) { d3 = o - ob; c3 = cum; }
    ob = o;
  }
  __device__ void slot(int nsp, int t, int& s, int& p) const {
    static_assert(WPIC_MAXSP == 4, "CellList holds four species");
    const int m1 = -(int)(t >= c1);
    s = -m1;
    p = t + o0 + (m1 & d1);
    if (nsp > 2) {
      const int m2 = -(int)(t >= c2), m3 = -(int)(t >= c3);
      s -= m2 + m3;
      p += (m2 & d2) + (m3 & d3);
    }
  }
};

// Sum over the 16 lanes of a DPP row (lanes 16r .. 16r+15), every lane of the
// row receiving it: quad permutes for the partners 1 and 2 apart, then row
// rotations by 4 and 8.  Cross-lane moves on the VALU (DPP) instead of
// ds_bpermute through the LDS crossbar.  Each row must be wholly active or
// wholly inactive (rows never exchange data).
template <int CTRL>
__device__ inline float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double dpp_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
constexpr int DPP_QUAD_XOR1 = 0xB1;  // quad_perm [1, 0, 3, 2]
constexpr int DPP_QUAD_XOR2 = 0x4E;  // quad_perm [2, 3, 0, 1]
constexpr int DPP_ROW_ROR4 = 0x124;
constexpr int DPP_ROW_ROR8 = 0x128;
template <class T>
__device__ inline T row16_sum(T v) {
  if constexpr (sizeof(T) == 8) {
    v += dpp_f64<DPP_QUAD_XOR1>(v);
    v += dpp_f64<DPP_QUAD_XOR2>(v);
    v += dpp_f64<DPP_ROW_ROR4>(v);
    v += dpp_f64<DPP_ROW_ROR8>(v);
  } else {
    v += dpp_f32<DPP_QUAD_XOR1>(v);
    v += dpp_f32<DPP_QUAD_XOR2>(v);
    v += dpp_f32<DPP_ROW_ROR4>(v);
    v += dpp_f32<DPP_ROW_ROR8>(v);
  }
  return v;
}

// Sum over the 64 lanes of a wholly active wave, the same bits in every lane.
__device__ inline double wave_sum(double v) {
  v = row16_sum(v);
  double r[4];
#pragma unroll
  for (int q = 0; q < 4; q++)
    r[q] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 16 * q),
                            __builtin_amdgcn_readlane(__double2loint(v), 16 * q));
  return (r[0] + r[1]) + (r[2] + r[3]);
}

// x . y added up from +0 in index order (the parity modes' sums), by a wholly
// active wave, the same bits in every lane: the lanes read and multiply 64
// elements at a time, the next 256 on their way, and the products are added one
// after another.  (Past the end they are +0, which changes no sum that began as
// +0.)  Read by the adding lane itself, an element costs its share of a memory
// wait: 65 ns where this takes 10 (a parity step at 256x256, 16 ppc: 89 -> 15
// ms).
__device__ inline double serial_dot(const double* x, const double* y, size_t n) {
  constexpr int U = 4;
  const size_t lane = threadIdx.x & 63;
  double a[U], b[U], s = 0.0;
  auto load = [&](size_t k0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t k = k0 + 64 * u + lane;
      a[u] = k < n ? x[k] : 0.0;
      b[u] = k < n ? y[k] : 0.0;
    }
  };
  load(0);
  for (size_t k0 = 0; k0 < n; k0 += 64 * U) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = a[u] * b[u];
    load(k0 + 64 * U);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int l = 0; l < 64; l++)
        s = s + __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v[u]), l),
                                 __builtin_amdgcn_readlane(__double2loint(v[u]), l));
  }
  return s;
}

constexpr int DPP_ROW_HALF_MIRROR = 0x141;  // lane l and 7 - l of each half row

// Sums over the G lanes of a group (4, half a DPP row or a whole one) of N
// values at once, each sum left in one lane.  Every step halves both the
// lanes that still differ and the values each holds: of a pair of values a
// lane keeps one and hands the other to its partner (lane l and l ^ 8, then
// 7 - l, l ^ 2 and l ^ 1 within the half row and the quad), so N values cost
// about N exchanges in all instead of N per step.  group_index gives the value
// that a lane's f-th result is the sum of, or -1 for a copy of another
// lane's.
template <int CTRL, class T>
__device__ inline T dpp_get(T v) {
  if constexpr (sizeof(T) == 8)
    return dpp_f64<CTRL>(v);
  else
    return dpp_f32<CTRL>(v);
}
template <int N, int CTRL, class T>
__device__ inline void halve(T* v, bool hi) {
#pragma unroll
  for (int k = 0; k < N / 2; k++) {
    const T keep = hi ? v[2 * k + 1] : v[2 * k], give = hi ? v[2 * k] : v[2 * k + 1];
    v[k] = keep + dpp_get<CTRL>(give);
  }
  if constexpr (N & 1) v[N / 2] = v[N - 1] + dpp_get<CTRL>(v[N - 1]);
}
constexpr int group_left(int n, int g) { return g == 1 ? n : group_left((n + 1) / 2, g / 2); }
// leaves group_left(N, G) results in v
template <int N, int G, class T>
__device__ inline void group_reduce(T* v, int lane) {
  static_assert(G == 4 || G == 8 || G == 16, "groups within a DPP row");
  if constexpr (G == 16) {
    halve<N, DPP_ROW_ROR8>(v, lane & 8);
    group_reduce<(N + 1) / 2, 8>(v, lane);
  } else if constexpr (G == 8) {
    halve<N, DPP_ROW_HALF_MIRROR>(v, lane & 4);
    group_reduce<(N + 1) / 2, 4>(v, lane);
  } else {
    halve<N, DPP_QUAD_XOR2>(v, lane & 2);
    halve<(N + 1) / 2, DPP_QUAD_XOR1>(v, lane & 1);
  }
}
template <int N, int G>
__device__ inline int group_index(int f, int lane) {
  constexpr int n1 = (N + 1) / 2;
  if constexpr (G == 1) {
    return f;
  } else {
    // the half row's mirror flips the lower bits of its upper quad: the
    // partner of l < 4 is 7 - l
    const int k = group_index<n1, G / 2>(f, lane);
    if (k < 0) return -1;
    const int i = 2 * k + ((lane & (G / 2)) ? 1 : 0);
    return i < N ? i : -1;
  }
}

// The sort's per-cell counts kept by a fused push: every cell of the tile
// keeps its particles (cumcnt, added when the tile's counts are flushed)
// except those that leave it, each of which moves one count from its own cell
// to the cell and row of its exchange code ((new x cell - nxgs) << 2 | row
// step + 1): in the tile's LDS counts (one-cell halo), or straight to rcnt
// when the destination lies beyond (a wrap across the box).  rcnt is
// [nsp*ny][nx].
template <int TXC, int TYC>
__device__ inline void count_leaver(const Grid2D& g, int (*hcn)[TYC + 2][TXC + 2], int* rcnt, int i0, int j0, int li,
                                    int lj, int s, int code) {
  atomicAdd(&hcn[s][lj + 1][li + 1], -1);
  const int cn = (code >> 2) + g.nxgs, dy = (code & 3) - 1;
  const int hx = cn - i0 + 1;
  if (hx >= 0 && hx <= TXC + 1) {
    atomicAdd(&hcn[s][lj + 1 + dy][hx], 1);
  } else {
    int jn = j0 + lj + dy;
    if (jn < g.nys) jn += g.ny;
    else if (jn > g.nye) jn -= g.ny;
    atomicAdd(&rcnt[((size_t)s * g.ny + (jn - g.nys)) * g.nx + (cn - g.nxgs)], 1);
  }
}
// the counts of a tile tw columns wide, with its cells' own particles, added
// to rcnt (rows wrap periodically in y)
template <int TXC, int TYC>
__device__ inline void flush_counts(const Grid2D& g, int (*hcn)[TYC + 2][TXC + 2], int* rcnt, const int* cumcnt,
                                    int i0, int j0, int tw) {
  const int w = TXC + 2, n = (TYC + 2) * w;
  for (int k = threadIdx.x; k < g.nsp * n; k += blockDim.x) {
    const int s = k / n, rem = k - s * n;
    const int hr = rem / w, hx = rem % w;
    int v = hcn[s][hr][hx];
    const int cx = i0 - 1 + hx;
    int jn = j0 - 1 + hr;
    if (hr >= 1 && hr <= TYC && hx >= 1 && hx <= tw && cx <= g.nxge && jn <= g.nye) {
      const int* cr = cumcnt + ((size_t)s * g.ny + (jn - g.nys)) * (g.nx + 1) + (cx - g.nxgs);
      v += cr[1] - cr[0];
    }
    if (v == 0) continue;
    if (jn < g.nys) jn += g.ny;
    else if (jn > g.nye) jn -= g.ny;
    atomicAdd(&rcnt[((size_t)s * g.ny + (jn - g.nys)) * g.nx + (cx - g.nxgs)], v);
  }
}

// Slots in an LDS queue for the active lanes of a wave with one atomic on the
// counter *n: the active lanes get consecutive slots in lane order.
__device__ inline int wave_enqueue(int* n) {
  const uint64_t m = __ballot(1);
  const int lane = __lane_id();
  const int leader = __ffsll((unsigned long long)m) - 1;
  int base = 0;
  if (lane == leader) base = atomicAdd(n, __popcll(m));
  base = __shfl(base, leader);
  return base + __popcll(m & ((1ull << lane) - 1));
}

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous band of logical tiles so neighbouring tiles (which share halo
// atomics) meet in the same L2.  Launch 8*ceil(n/8) groups; extra ones exit.
__device__ inline int xcd_tile(int bid, int ntiles) {
  const int per = (ntiles + 7) >> 3;
  return (bid & 7) * per + (bid >> 3);
}
inline int xcd_grid(int ntiles) { return ((ntiles + 7) >> 3) << 3; }

// Columns of cells a push workgroup takes (of four rows): 32, or 16 or 8 where
// the grid would not give each of the 256 CUs two workgroups otherwise (a
// narrow tile stages and flushes more halo per cell).
inline int tile_width(const Grid2D& g) {
  const int nty = (g.ny + 3) / 4;
  int w = 32;
  while (w > 8 && ((g.nx + w - 1) / w) * nty < 512) w >>= 1;
  return w;
}

// ---------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------
struct CgScal {
  double sum_g, eps, sumr_g, sum2_g, av, bv;
  int ite, active;
};

// how a fast solve stands after an iteration, written by the device into the
// host's pinned memory: components that go on, iterations done, error bits
struct CgPoll {
  int more[3], ite[3], err;
};

// A context's pinned slots for large copies to the host (wpic_copy.hip), made
// by the first such copy and given back with the context.
struct HostRing {
  static constexpr int NSLOT = 12;
  char* buf = nullptr;
  hipEvent_t ev[NSLOT] = {};
};
// `bytes` from device memory to the caller's array, in stream order; done on
// return
hipError_t copy_to_host(HostRing& ring, int device, hipStream_t st, void* dst, const void* src, size_t bytes);
void ring_free(HostRing& ring);

struct TimerRec {
  std::string name;
  hipEvent_t a, b;
};

}  // namespace wpic

struct wpic_ctx {
  wpic_params2d P;
  wpic::Grid2D g;
  int mode;
  hipStream_t st;
  // the step's exchange and sort run on st2 while the field solve runs on st
  // (they share no buffer); ev_push / ev_sort order them around the push
  hipStream_t st2;
  hipEvent_t ev_push, ev_sort;
  int device;

  // particles: species s occupies [s*ncap, (s+1)*ncap); rows compact within
  // A holds the sorted particles (the reference's up) as aperm[k] -> slot of
  // A's buffer (null: identity); B holds gp, slot-aligned with A after the
  // push, which moves each record and its id.  The sort writes only the
  // permutation, then A and B swap buffers (ids included): the records are
  // read through aperm by the next push.
  wpic::Parts A, B;
  bool mixed;            // WPIC_MODE_MIXED context: MA/MB hold the particles
  wpic::PartsM MA, MB;
  int* aperm;            // A's slot -> record in A's buffer, or null
  int* permbuf;          // [N] the sort's permutation
  int *code, *R, *holes, *ulist, *dlist;
  int* rows[3];                   // row structures: rowbase [nsp*ny] then np2 [nsp*ny]
  int ra, rb, rn;                 // which row structure belongs to A, B, the exchange
  int *rowbaseA, *np2A, *cumcnt;  // [nsp*ny], [nsp*ny], [nsp*ny*(nx+1)]
  int *rowbaseB, *np2B;           // rows of B (gp)
  int *rowbaseN, *np2N;           // rows after the y exchange
  int* rowcnt;                    // [nsp*ny][4] leavers, up, down, incoming
  // [nsp*ny][nx] particles per (species, row, x cell) after the step's push:
  // the mixed push counts them (rcnt_fill) and the fast sort takes the rows'
  // cell counts from them instead of counting the codes again
  int* rcnt;
  bool rcnt_fill;
  bool b_valid;       // B holds a gp array
  bool b_aligned;     // B's slots are A's slots (after particle__solv)
  int pusher;         // WPIC_PUSHER_BORIS or WPIC_PUSHER_VAY
  long long npart;    // particles at the last load or injection (all species): picks the push's lane groups
  bool b_accl;        // B is mom_calc__accl's gp: A's positions, A's cell order
  bool exch_pending;  // R / N rows describe B after bc__particle_y
  std::vector<int> h_rows[3];  // host mirrors of the row structures
  bool h_rows_ok[3];

  // fields: planes of (nx+4)*(ny+4)
  double *uf, *df, *uj;
  double* pjbuf;  // parity-mode per-cell current blocks [nx*ny][65]

  // CG: interior vectors per component
  double *phi, *pa, *pb, *rr;            // [3][nx*ny]
  double *bb, *ap;                       // [3][nx*ny] b (parity mode, adjoint) and A p (parity mode, lazy)
  double* part;                          // block partial sums [3][3][NPB]
  wpic::CgScal* scal;                    // [2][3]
  int* err;                              // device error bits
  wpic::CgPoll* poll;                    // pinned host memory
  hipEvent_t ev_poll;                    // recorded after the iteration that writes it
  int cg_iters[3];
  int cg_hint;  // the largest iteration count of the last solve (the first batch's size)

  wpic::HostRing ring;
  double* staging;  // transfer staging (lazy)
  size_t staging_n;
  long long* aosbase;  // [nsp*ny] row starts in a compact AoS transfer buffer
  double* gbuf;        // Gauss residual / rho scratch (lazy)
  double* mom;         // moments mom(7, nxgs-1:nxge+1, nys-1:nye+1, nsp) (lazy)
  double* red;      // diagnostics reduction scratch
  size_t red_n;

  bool timing;
  std::vector<wpic::TimerRec> timers;
  std::vector<std::pair<std::string, std::pair<double, long long>>> tsum;

  int* perm_out;          // when set, the sort records the gp slot of every sorted slot
  struct AdjState* adj;   // recorded run and adjoint arrays (wpic_adj.h), lazy
};

namespace wpic {

// partial-sum blocks of a CG component: one per 256 cells, at most NPB (the
// number, and so the order of the sums, depends on the grid alone)
constexpr int NPB = 1024;
inline int cg_blocks(const Grid2D& g) {
  const int n = (g.nx * g.ny + 255) / 256;
  return n < NPB ? n : NPB;
}
// Work units of an iteration's kernels: 64 columns of `len` rows for each wave,
// len so that a grid gives some 2,048 units (a wave that marches more rows
// reads fewer of its neighbours')
struct Strips2 {
  int ntx, len, units;
};
__host__ __device__ inline Strips2 strips2(const Grid2D& g) {
  Strips2 s;
  s.ntx = (g.nx + 63) / 64;
  int len = (int)((long long)s.ntx * g.ny / 2048);
  s.len = len < 1 ? 1 : (len > 16 ? 16 : len);
  s.units = s.ntx * ((g.ny + s.len - 1) / s.len);
  return s;
}

int set_error(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

// launchers (each enqueues on ctx->st) -------------------------------------
// push / deposit
hipError_t launch_push_deposit(wpic_ctx* c, bool push, bool deposit);
hipError_t launch_gather_pj(wpic_ctx* c);
// fields
hipError_t launch_zero(wpic_ctx* c, double* p, size_t n);
hipError_t launch_curre_bc(wpic_ctx* c);
hipError_t launch_dfield_bc(wpic_ctx* c);
hipError_t launch_cg_init(wpic_ctx* c);
hipError_t launch_cg_iter(wpic_ctx* c, int it, bool poll);
hipError_t launch_field_end_periodic(wpic_ctx* c);
hipError_t launch_cg_store(wpic_ctx* c);
hipError_t launch_e_update(wpic_ctx* c);
hipError_t launch_uf_add(wpic_ctx* c);
hipError_t launch_energy(wpic_ctx* c, double* dout);
hipError_t launch_gauss(wpic_ctx* c, double* G, double* rho);
hipError_t launch_codes_identity(wpic_ctx* c);
// particles: boundaries, exchange, sort
hipError_t launch_wrapx(wpic_ctx* c, bool injection);
hipError_t launch_ic_shock(wpic_ctx* c, unsigned long long seed, int np2, double v0, const double* sd, double l_damp,
                           const double* b);
hipError_t launch_inject(wpic_ctx* c, unsigned long long seed, int it, const int* base_new, const int* nl,
                         const long long* idoff, double v0, const double* sd, double l_damp, double by, double bz,
                         bool reloc);
hipError_t launch_rowscan(wpic_ctx* c, bool ywrap);
hipError_t launch_rowcount(wpic_ctx* c);
hipError_t launch_rowbuild(wpic_ctx* c);
hipError_t launch_rowsort(wpic_ctx* c);
hipError_t launch_rowsort_fast(wpic_ctx* c);
// transfers and initial state
hipError_t launch_records_in(wpic_ctx* c, const double* aos, long long n, int which);
hipError_t launch_records_out(wpic_ctx* c, double* aos, int which);
hipError_t launch_planes_from_aos(wpic_ctx* c, const double* aos, double* planes, int ncomp);
hipError_t launch_planes_to_aos(wpic_ctx* c, const double* planes, double* aos, int ncomp);
hipError_t launch_ic_beams(wpic_ctx* c, unsigned long long seed, int n_ppc, double udrift, double uth_e,
                           double uth_i);
hipError_t launch_fill(wpic_ctx* c, double* p, size_t n, double v);
hipError_t launch_ic_weibel(wpic_ctx* c, unsigned long long seed, int n0, const double* sd, double t_ani);
// hp: x0, y0, lcs, b0, e1, ncs, nbg, f1, f2, sd1, sd2
hipError_t launch_ic_harris(wpic_ctx* c, unsigned long long seed, int np2, int ibg, const double* hp);
hipError_t launch_gather_rows(wpic_ctx* c, const Parts& src, const int* ap, const Parts& dst, const int* rows);
// moments (mom_calc.f90, boundary_*__mom): deposit kinds
enum { MOM_TILE_KICK = 0, MOM_TILE_GP = 1, MOM_ANY = 2, MOM_PARITY_ALIGNED = 3, MOM_PARITY_ANY = 4 };
hipError_t launch_mom_accl(wpic_ctx* c);
hipError_t launch_mom_deposit(wpic_ctx* c, int kind);
hipError_t launch_mom_bc(wpic_ctx* c);
// mixed-precision form
hipError_t launch_push_deposit_mixed(wpic_ctx* c);
hipError_t launch_up_to_mixed(wpic_ctx* c, const double* aos);
hipError_t launch_mixed_to_aos(wpic_ctx* c, double* aos);
hipError_t launch_ic_beams_mixed(wpic_ctx* c, unsigned long long seed, int n_ppc, double udrift, double uth_e,
                                 double uth_i);
hipError_t launch_energy_mixed(wpic_ctx* c, double* dout);
hipError_t launch_mom_mixed(wpic_ctx* c);

// one fused step (wpic_step2d's body) and the CG iteration loop of field__fdtd_i
int step_once(wpic_ctx* c);
int cg_loop(wpic_ctx* c);
int check_err_ctx(wpic_ctx* c);
hipError_t launch_cg_start(wpic_ctx* c);
// adjoint
hipError_t launch_adj_unsort(wpic_ctx* c, const int* rows, const int* perm, const double* lamA, double* lamB,
                             size_t N);
hipError_t launch_adj_field1(wpic_ctx* c, const double* lamF, double* lamF2, double* lamJ);
hipError_t launch_adj_field2(wpic_ctx* c, double* lamF2, double* lamJ);
hipError_t launch_adj_particles(wpic_ctx* c, const Parts& P, const int* rows, const int* cumcnt, const double* uf,
                                const double* lamB, const double* lamJ, double* lamA, double* lamT, size_t N);
hipError_t launch_adj_t2f(wpic_ctx* c, const double* lamT, double* lamF);
hipError_t launch_adj_seed(wpic_ctx* c, double* lamF, double seed);
hipError_t launch_adj_params(wpic_ctx* c, const Parts& P, const int* rows, const double* lamA, size_t N,
                             const double* lamF, double udrift, double uth_e, int mode, int n_ppc,
                             double* out);
hipError_t launch_perturb_bz(wpic_ctx* c, double amp, int mode);
hipError_t launch_adj_lamF_to_planes(wpic_ctx* c, const double* lamF, double* planes);
void adj_free(wpic_ctx* c);

void timer_begin(wpic_ctx* c, const char* name, hipEvent_t* a);
void timer_end(wpic_ctx* c, hipEvent_t a);

}  // namespace wpic
