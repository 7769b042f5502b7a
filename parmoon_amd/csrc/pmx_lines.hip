// pmx_lines.hip -- matrix rows on the line layout: products, defects, Jacobi,
// the line-group sweeps of the multicolour smoother and the small levels that
// run in one workgroup; stream-ordered launchers.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "pmx_kernels.hpp"
#include "pmx_lines.hpp"
#include "pmx_ops.hpp"

namespace pmx {

// ============================================================ rows of a line
// A unit of max(64, P) lanes holds the row pairs of 64 / P lines (one line for
// P >= 64), and kSplits units of a workgroup share the same rows: unit w adds
// the groups k = w mod kSplits, so that every row has several short chains of
// loads in flight; unit 0 combines the partial sums in the order of w.  The
// sums over the groups before the line and after it are kept apart, and every
// kernel adds them in this one order, so a row's result does not depend on
// which kernel or workgroup shape computed it.
//
// Bound by HBM: a product reads every value once and the x run of a group once
// per row pair.  64^3 Q2, FP32 / FP64: 100 / 206 us per product (5.3 / 5.2
// TB/s of values; a copy reaches 4.9 TB/s read plus written).  Rows of a
// residue class on a lane, with a run of x per row instead of per pair, took
// 139 / 296 us.  Splits 1, 2, 4, 8 measured 106, 103, 100, 98 us (FP32
// product) and 17, 16.2, 15.9, 17 us per group launch of a sweep.
template <typename T> struct PairSums {
  T lo_o, lo_e, hi_o, hi_e;  // groups before / after the line, odd and even row
};
// this unit's partial sums: lo / hi select the parts
template <typename T, typename V, int O, int U>
__device__ __forceinline__ PairSums<T> pair_sums(const V *v, const T *x, const int *off, int nlo, int ng, bool lo,
                                                 bool hi, int w, int P, int M, int d3) {
  PairSums<T> s{0, 0, 0, 0};
  if (lo) add_groups<T, V, O, U>(v, x, off, w, nlo, kSplits, P, M, d3, s.lo_o, s.lo_e);
  if (hi) add_groups<T, V, O, U>(v, x, off, nlo + 1 + w, ng, kSplits, P, M, d3, s.hi_o, s.hi_e);
  return s;
}
template <typename T> __device__ __forceinline__ void add_partial(PairSums<T> &s, const PairSums<T> &p) {
  s.lo_o += p.lo_o;
  s.lo_e += p.lo_e;
  s.hi_o += p.hi_o;
  s.hi_e += p.hi_e;
}
// the line's own group without the diagonal, added to the sum of the others;
// c: the group's values, x: the run from lattice coordinate 2m
template <typename T, typename V, int O>
__device__ __forceinline__ T own_odd(const V *c, const T *x, T s) {
  s = fma((T)c[0], x[0], s);
  return fma((T)c[2], x[2], s);
}
template <typename T, typename V, int O>
__device__ __forceinline__ T own_even(const V *c, const T *x, T s) {
#pragma unroll
  for (int e = 0; e < 2 * O + 1; e++)
    if (e != O) s = fma((T)c[3 + e], x[e + 2 - O], s);
  return s;
}
// distance of the second part of the last pair's run (clamped to the lattice)
template <int O> __device__ __forceinline__ int run_split(int m, int P) { return m == P - 1 ? (O == 2 ? 1 : 2) : 3; }

// MODE 0: y = A x (MatVect, Blas2.C:86-118)
// MODE 1: y = f - A x (ScalarDefect, Blas2.C:37-83)
// MODE 2: y = (1-w) x + w (f - A_off x)/d (TMGLevel3D::Jacobi, MGLevel3D.C:469-563)
// HALF (modes 0, 1): the sums over the groups after the lines are those that
// the last backward sweep left in psum (x has not changed since), so only the
// first half of the values is read.  64^3 Q2 FP32: 100 -> 53 us.
template <typename T, int O, int MODE, bool HALF>
__global__ __launch_bounds__(512) void k_line_rows(LineSet set, int lg, const T *__restrict__ val,
                                                   const T *__restrict__ x, const T *__restrict__ f,
                                                   T *__restrict__ y, double omega, const T *__restrict__ psum) {
  using L = Lines<O>;
  __shared__ PairSums<T> red[kSplits - 1][128];
  const int P = 1 << lg, M = 2 * P + 1, ul = lg < 6 ? 6 : lg;
  const int t = threadIdx.x & ((1 << ul) - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> ul);
  const UnitLines u = unit_lines<O>(set, M, lg, xcd_remap(blockIdx.x, gridDim.x));
  const int m = t & (P - 1), yy = u.y0 + L::S * (t >> lg);
  const bool ok = yy <= M - 2;
  const int ly = ok ? yy : u.y0, c = line_class<O>(u.y0, u.z);
  const GroupTable<O> &g = group_table<O>();
  const int nlo = g.nlo[c], ng = g.ng[c], d3 = run_split<O>(m, P);
  const T *v = val + line_values<T, O>(P, L::group_base(P, ly, u.z), m);
  const int p0 = M * (ly + M * u.z) + 2 * m;
  T own[L::VL], xr[5], fo = 0, fe = 0, ho = 0, he = 0;
  if (w == 0) {
    if (HALF) {
      ho = psum[p0 + 1];
      he = psum[p0 + 2];
    }
    load_group<T, O>(v + (int64_t)nlo * (L::VL * P), P, own);
    load_run<T, 3>(x + p0, xr);
    load_run<T, O == 2 ? 2 : 1>(x + p0 + d3, xr + 3);
    if (MODE >= 1) {
      fo = f[p0 + 1];
      fe = f[p0 + 2];
    }
  }
  PairSums<T> s = pair_sums<T, T, O, 2>(v, x + p0, g.off[c], nlo, ng, true, !HALF, w, P, M, d3);
  if (w) red[w - 1][t] = s;
  __syncthreads();
  if (w || !ok) return;
#pragma unroll
  for (int q = 0; q < kSplits - 1; q++) add_partial(s, red[q][t]);
  if (HALF) {
    s.hi_o = ho;
    s.hi_e = he;
  }
  T ro = own_odd<T, T, O>(own, xr, s.lo_o + s.hi_o), re = own_even<T, T, O>(own, xr, s.lo_e + s.hi_e);
  const T xo = xr[1], xe = xr[2];
  if (MODE == 2) {
    const T a = (T)omega;
    ro = (1 - a) * xo + a * (fo - ro) / own[1];
    re = (1 - a) * xe + a * (fe - re) / own[3 + O];
  } else {
    ro = fma(own[1], xo, ro);
    re = fma(own[3 + O], xe, re);
    if (MODE == 1) {
      ro = fo - ro;
      re = fe - re;
    }
  }
  y[p0 + 1] = ro;
  if (m < P - 1) y[p0 + 2] = re;
}

// ============================================================ line sweeps
// x = w ((f - A_off x)/d - x) + x (TMGLevel3D::SOR, MGLevel3D.C:280-361) for
// the rows of a line, colour by colour.  l: the line's x in LDS (coordinate
// 0 .. 2P).  The lanes of a line belong to one wavefront (P <= 64: LDS
// operations of a wavefront complete in order) or to one workgroup (P = 128).
enum { kForward = 0, kBackward = 1, kForwardBackward = 2, kBackwardForward = 3 };
template <typename T> struct PairRow {
  T fo, fe, so, se, dio, die;  // right-hand side, sums of the other lines, diagonals
};
template <typename T, typename V, int O>
__device__ __forceinline__ void line_steps(T *l, const V *own, const PairRow<T> &r, int m, int P, int seq, double omega,
                                           bool active, bool wide) {
  constexpr int C = Lines<O>::C;
  const int co = (2 * m + 1) % C, ce = (2 * m + 2) % C;
  // at a turn the repeated colour reproduces its rows bit for bit when omega
  // is 1 (the neighbours it reads are unchanged) and is skipped
  const int skip = omega == 1.0 ? 1 : 0, n = seq < 2 ? C : 2 * C - skip;
  for (int i = 0; i < n; i++) {
    int c = i < C ? i : 2 * C - 1 - skip - i;
    if (seq == kBackward || seq == kBackwardForward) c = C - 1 - c;
    if (wide) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (!active) continue;
    const bool odd = c == co;
    if (odd || (c == ce && m < P - 1)) {
      T *q = l + 2 * m;
      T x[5];
#pragma unroll
      for (int e = 0; e < 3; e++) x[e] = q[e];
      if (odd) {
        const T gs = (r.fo - own_odd<T, V, O>(own, x, r.so)) / r.dio;
        q[1] = skip ? gs : (T)omega * (gs - x[1]) + x[1];
      } else {
        x[3] = q[3];
        if (O == 2) x[4] = q[4];
        const T gs = (r.fe - own_even<T, V, O>(own, x, r.se)) / r.die;
        q[2] = skip ? gs : (T)omega * (gs - x[2]) + x[2];
      }
    }
  }
}

// One line group of a sweep; V = _Float16: row-scaled values a_ij / a_ii with
// dinv = 1 / a_ii (x = w (f dinv - W_off x - x) + x).
//
// Half sums.  In a forward sweep the lines before a row's line already hold
// their new x; the backward sweep reaches the row before it changes them, so
// the row's sum over them is the same (and likewise the sums over the lines
// after it from a backward to the next forward sweep).  The sums are kept in
// psum: a backward launch reads only the values after its lines, a following
// forward launch only those before them, and n symmetric sweeps read the
// matrix n + 1/2 times (n when x starts at zero) instead of 2n.
// Bound by the launch (about 4 us whatever its size) plus the values from HBM:
// 64^3 Q2 FP32 15.9 us per group of 58 MB with all values, 10 us with half of
// them.  A launch per colour, 3 C^2 of them, took 8.7 us each (26 us for the
// rows of a group).
enum {
  kSumLo = 1, kSumHi = 2,                         // sums to compute
  kSumKept = 4,                                   // the other one is in psum (else it is 0)
  kKeepLo = 16, kKeepHi = 32, kKeepZero = 48,     // what to leave in psum
};
template <typename T, typename V, int O>
__global__ __launch_bounds__(512) void k_line_sweep(LineSet set, int lg, int seq, int sums, const V *__restrict__ val,
                                                    T *x, const T *__restrict__ f, T *__restrict__ psum, double omega,
                                                    const int *__restrict__ bnd_set, const float *__restrict__ dinv) {
  using L = Lines<O>;
  constexpr bool kScaled = sizeof(V) == 2;
  __shared__ PairSums<T> red[kSplits - 1][128];
  __shared__ T lx[264];
  const int P = 1 << lg, M = 2 * P + 1, ul = lg < 6 ? 6 : lg;
  const int t = threadIdx.x & ((1 << ul) - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> ul);
  const UnitLines u = unit_lines<O>(set, M, lg, xcd_remap(blockIdx.x, gridDim.x));
  const int m = t & (P - 1), yy = u.y0 + L::S * (t >> lg);
  const bool ok = yy <= M - 2;
  const int ly = ok ? yy : u.y0, c = line_class<O>(u.y0, u.z);
  const GroupTable<O> &g = group_table<O>();
  const int nlo = g.nlo[c], ng = g.ng[c], d3 = run_split<O>(m, P);
  const V *v = val + line_values<V, O>(P, L::group_base(P, ly, u.z), m);
  const int p0 = M * (ly + M * u.z) + 2 * m;
  V own[L::VL];
  PairRow<T> r{0, 0, 0, 0, 1, 1};
  T *l = lx + (t >> lg) * (2 * P + 2), ko = 0, ke = 0;
  // a start from zero has no sums over the lines after a row, unless the
  // boundary values are not zero
  const bool lo = sums & kSumLo, hi = (sums & kSumHi) || (bnd_set && *bnd_set != 0);
  if (w == 0) {
    if (sums & kSumKept) {
      ko = psum[p0 + 1];
      ke = psum[p0 + 2];
    }
    load_group<V, O>(v + (int64_t)nlo * (L::VL * P), P, own);
    r.fo = f[p0 + 1];
    r.fe = f[p0 + 2];
    if constexpr (kScaled) {
      r.fo *= dinv[p0 + 1];
      r.fe *= dinv[p0 + 2];
    } else {
      r.dio = (T)own[1];
      r.die = (T)own[3 + O];
    }
    l[2 * m + 1] = x[p0 + 1];
    l[2 * m + 2] = x[p0 + 2];
    if (m == 0) l[0] = x[p0];
  }
  PairSums<T> s = pair_sums<T, V, O, 2>(v, x + p0, g.off[c], nlo, ng, lo, hi, w, P, M, d3);
  if (w) red[w - 1][t] = s;
  __syncthreads();
  const bool wide = P > 64;
  if (w && !wide) return;
  if (w == 0) {
#pragma unroll
    for (int q = 0; q < kSplits - 1; q++) add_partial(s, red[q][t]);
    if (sums & kSumKept) {
      if (lo) {
        s.hi_o = ko;
        s.hi_e = ke;
      } else {
        s.lo_o = ko;
        s.lo_e = ke;
      }
    }
    r.so = s.lo_o + s.hi_o;
    r.se = s.lo_e + s.hi_e;
  }
  line_steps<T, V, O>(l, own, r, m, P, seq, omega, w == 0, wide);
  if (w || !ok) return;
  const int keep = sums & kKeepZero;
  x[p0 + 1] = l[2 * m + 1];
  if (keep) psum[p0 + 1] = keep == kKeepLo ? s.lo_o : keep == kKeepHi ? s.hi_o : T(0);
  if (m < P - 1) {
    x[p0 + 2] = l[2 * m + 2];
    if (keep) psum[p0 + 2] = keep == kKeepLo ? s.lo_e : keep == kKeepHi ? s.hi_e : T(0);
  }
}

// ============================================================ one workgroup
// A whole sweep of a small level in one workgroup: the level's x is in LDS,
// the line groups follow each other with workgroup barriers.  A lane's row
// pair may belong to any line of the group (its class and group table are the
// lane's own), 4 x 64 pairs at a time with kSplits wavefronts each.
constexpr int kWgThreads = 1024, kWgSlots = kWgThreads / 64 / kSplits;
template <int O> struct WgTables {
  int off[Lines<O>::S * Lines<O>::S][Lines<O>::kMaxGroups];
};
template <int O> __device__ __forceinline__ void wg_tables(WgTables<O> &s) {
  constexpr int n = Lines<O>::S * Lines<O>::S * Lines<O>::kMaxGroups;
  const int *src = &group_table<O>().off[0][0];
  for (int i = threadIdx.x; i < n; i += kWgThreads) (&s.off[0][0])[i] = src[i];
}
// Runs fn(pair sums, line, lane data) for the pairs of the lines y = y0 + ys j,
// z = z0 + zs k of the level; every thread of the workgroup calls it.
struct WgPair {
  int m, p0, c;       // pair, lattice index of coordinate 2m, class
  int64_t base;       // groups stored before the line
  bool ok;
};
template <typename T, int O, class F>
__device__ __forceinline__ void wg_lines(const WgTables<O> &tb, PairSums<T> (*red)[kSplits - 1][64], int lg, int y0,
                                         int ys, int z0, int zs, const T *__restrict__ val, const T *lx, bool lo,
                                         bool hi, F fn) {
  using L = Lines<O>;
  const int P = 1 << lg, M = 2 * P + 1;
  if (y0 > M - 2 || z0 > M - 2) return;
  const int ny = (M - 2 - y0) / ys + 1, nz = (M - 2 - z0) / zs + 1, np = ny * nz * P;
  const int t = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = wave / kSplits, w = wave % kSplits;
  const GroupTable<O> &g = group_table<O>();
  for (int q0 = 0; q0 < np; q0 += 64 * kWgSlots) {
    const int q = q0 + 64 * slot + t, qc = q < np ? q : np - 1;
    const int ln = qc >> lg, kz = ln / ny;
    const int y = y0 + ys * (ln - kz * ny), z = z0 + zs * kz;
    WgPair pr;
    pr.ok = q < np;
    pr.m = qc & (P - 1);
    pr.c = line_class<O>(y, z);
    pr.base = L::group_base(P, y, z);
    pr.p0 = M * (y + M * z) + 2 * pr.m;
    const T *v = val + line_values<T, O>(P, pr.base, pr.m);
    const int nlo = g.nlo[pr.c], ng = g.ng[pr.c];
    T own[L::VL];
    if (w == 0) load_group<T, O>(v + (int64_t)nlo * (L::VL * P), P, own);
    PairSums<T> s = pair_sums<T, T, O, 2>(v, lx + pr.p0, tb.off[pr.c], nlo, ng, lo, hi, w, P, M, run_split<O>(pr.m, P));
    if (w) red[slot][w - 1][t] = s;
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int k = 0; k < kSplits - 1; k++) add_partial(s, red[slot][k][t]);
      fn(pr, s, own);
    }
    __syncthreads();
  }
}
template <typename T, int O>
__device__ __forceinline__ void wg_sweep(const WgTables<O> &tb, PairSums<T> (*red)[kSplits - 1][64], int lg,
                                         const T *__restrict__ val, T *lx, const T *__restrict__ f, double omega,
                                         bool ssor) {
  using L = Lines<O>;
  constexpr int G = L::C * L::C;
  const int P = 1 << lg;
  for (int i = 0; i < (ssor ? 2 * G - 1 : G); i++) {
    const int gi = i < G ? i : 2 * G - 2 - i;
    const int seq = i >= G ? kBackward : (ssor && i == G - 1) ? kForwardBackward : kForward;
    const int yr = gi % L::C, zr = gi / L::C;
    wg_lines<T, O>(tb, red, lg, yr ? yr : L::C, L::C, zr ? zr : L::C, L::C, val, lx, true, true,
                   [&](const WgPair &pr, const PairSums<T> &s, const T *own) {
                     const PairRow<T> r{f[pr.p0 + 1], f[pr.p0 + 2], s.lo_o + s.hi_o, s.lo_e + s.hi_e, own[1], own[3 + O]};
                     line_steps<T, T, O>(lx + pr.p0 - 2 * pr.m, own, r, pr.m, P, seq, omega, pr.ok, false);
                   });
  }
}
// the level's x, Dirichlet rows x = f
template <typename T>
__device__ __forceinline__ void wg_stage(T *lx, const T *x, const T *__restrict__ f, int N, const int *__restrict__ bnd,
                                         int nb) {
  for (int i = threadIdx.x; i < N; i += kWgThreads) lx[i] = x[i];
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += kWgThreads) lx[bnd[i]] = f[bnd[i]];
  __syncthreads();
}
template <typename T, int O>
__global__ __launch_bounds__(kWgThreads) void k_sweep_wg(int lg, const T *__restrict__ val, T *x,
                                                         const T *__restrict__ f, double omega, int ssor,
                                                         const int *__restrict__ bnd, int nb) {
  extern __shared__ __align__(16) unsigned char sweep_lds[];
  T *lx = reinterpret_cast<T *>(sweep_lds);
  __shared__ WgTables<O> tb;
  __shared__ PairSums<T> red[kWgSlots][kSplits - 1][64];
  const int M = 2 * (1 << lg) + 1, N = M * M * M;
  wg_tables<O>(tb);
  wg_stage(lx, x, f, N, bnd, nb);
  wg_sweep<T, O>(tb, red, lg, val, lx, f, omega, ssor != 0);
  for (int i = threadIdx.x; i < N; i += kWgThreads) x[i] = lx[i];
}

// ||f - A x|| of the LDS iterate over all rows (Dirichlet rows: 0), the same
// value in every thread
template <typename T, int O>
__device__ double wg_defect_norm(const WgTables<O> &tb, PairSums<T> (*red)[kSplits - 1][64], int lg,
                                 const T *__restrict__ val, const T *lx, const T *__restrict__ f, double *lred) {
  const int P = 1 << lg;
  double sum = 0;
  wg_lines<T, O>(tb, red, lg, 1, 1, 1, 1, val, lx, true, true,
                 [&](const WgPair &pr, const PairSums<T> &s, const T *own) {
                   if (!pr.ok) return;
                   const T *x = lx + pr.p0;
                   T ro = own_odd<T, T, O>(own, x, s.lo_o + s.hi_o);
                   const T d = f[pr.p0 + 1] - fma(own[1], x[1], ro);
                   sum += (double)d * (double)d;
                   if (pr.m < P - 1) {
                     T re = own_even<T, T, O>(own, x, s.lo_e + s.hi_e);
                     const T e = f[pr.p0 + 2] - fma(own[3 + O], x[2], re);
                     sum += (double)e * (double)e;
                   }
                 });
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o, 64);
  if (threadIdx.x % 64 == 0) lred[threadIdx.x / 64] = sum;
  __syncthreads();
  double t = 0;
  for (int w = 0; w < kWgThreads / 64; w++) t += lred[w];
  __syncthreads();
  return sqrt(t);
}
// The coarse-level loop of TMultiGrid3D::Smooth(CoarseSmooth)
// (MultiGrid3D.C:225-337) in one workgroup: res = ||f - A x||, then while
// res > red * res_0 and fewer than maxit sweeps: one Jacobi (kind 1, omega
// damped), SOR (2) or SSOR (3) sweep and res again.  The sweeps compute each
// row as the launched sweeps do (bit-identical iterates); xj: global scratch
// of N entries (Jacobi output).
template <typename T, int O>
__global__ __launch_bounds__(kWgThreads) void k_coarse_wg(int lg, const T *__restrict__ val, T *x,
                                                          const T *__restrict__ f, double omega, int kind, int maxit,
                                                          double red_factor, const int *__restrict__ bnd, int nb,
                                                          T *xj) {
  extern __shared__ __align__(16) unsigned char sweep_lds[];
  T *lx = reinterpret_cast<T *>(sweep_lds);
  __shared__ WgTables<O> tb;
  __shared__ PairSums<T> red[kWgSlots][kSplits - 1][64];
  __shared__ double lred[kWgThreads / 64];
  const int P = 1 << lg, M = 2 * P + 1, N = M * M * M;
  wg_tables<O>(tb);
  for (int i = threadIdx.x; i < nb; i += kWgThreads) xj[bnd[i]] = f[bnd[i]];
  wg_stage(lx, x, f, N, bnd, nb);
  double res = wg_defect_norm<T, O>(tb, red, lg, val, lx, f, lred);
  const double reduction = red_factor * res;
  for (int it = 0; res > reduction && it < maxit; it++) {
    if (kind == 1) {
      const T a = (T)omega;
      wg_lines<T, O>(tb, red, lg, 1, 1, 1, 1, val, lx, true, true,
                     [&](const WgPair &pr, const PairSums<T> &s, const T *own) {
                       if (!pr.ok) return;
                       const T *q = lx + pr.p0;
                       const T ro = own_odd<T, T, O>(own, q, s.lo_o + s.hi_o);
                       xj[pr.p0 + 1] = (1 - a) * q[1] + a * (f[pr.p0 + 1] - ro) / own[1];
                       if (pr.m < P - 1) {
                         const T re = own_even<T, T, O>(own, q, s.lo_e + s.hi_e);
                         xj[pr.p0 + 2] = (1 - a) * q[2] + a * (f[pr.p0 + 2] - re) / own[3 + O];
                       }
                     });
      for (int i = threadIdx.x; i < N; i += kWgThreads) lx[i] = xj[i];
      __syncthreads();
    } else {
      wg_sweep<T, O>(tb, red, lg, val, lx, f, omega, kind == 3);
    }
    res = wg_defect_norm<T, O>(tb, red, lg, val, lx, f, lred);
  }
  for (int i = threadIdx.x; i < N; i += kWgThreads) x[i] = lx[i];
}

// Row-scaled FP16 copy of the FP32 values: entry k of an active row holds
// a_k / a_diag rounded to FP16 (saturated at +-65504, the largest finite FP16
// value), and dinv[p] = 1 / a_diag in FP32.  A pair's slots of a group are
// contiguous (16 bytes for Q2).
template <int O>
__global__ __launch_bounds__(64) void k_scaled_values(LineSet set, int lg, const float *__restrict__ val,
                                                      _Float16 *__restrict__ val16, float *__restrict__ dinv) {
  using L = Lines<O>;
  const int P = 1 << lg, M = 2 * P + 1, segs = lg > 6 ? P / 64 : 1;
  const UnitLines u = unit_lines<O>(set, M, lg, blockIdx.x / segs);
  const int t = threadIdx.x + 64 * (blockIdx.x % segs), m = t & (P - 1), y = u.y0 + L::S * (t >> lg);
  if (y > M - 2) return;
  const GroupTable<O> &g = group_table<O>();
  const int c = line_class<O>(u.y0, u.z), nlo = g.nlo[c], ng = g.ng[c];
  const int64_t base = L::group_base(P, y, u.z);
  const float *v = val + line_values<float, O>(P, base, m);
  _Float16 *o = val16 + line_values<_Float16, O>(P, base, m);
  const float *own = v + (int64_t)nlo * (L::VL * P);
  const int p0 = M * (y + M * u.z) + 2 * m;
  const bool even = m < P - 1;
  const float ro = 1.0f / own[1 * P], re = even ? 1.0f / own[(3 + O) * P] : 0.0f;
  dinv[p0 + 1] = ro;
  if (even) dinv[p0 + 2] = re;
  for (int k = 0; k < ng; k++) {
    float a[L::VL];
    _Float16 h[L::VL];
    load_group<float, O>(v + (int64_t)k * (L::VL * P), P, a);
#pragma unroll
    for (int s = 0; s < L::VL; s++)
      h[s] = (_Float16)fminf(fmaxf(a[s] * (s < 3 ? ro : re), -65504.0f), 65504.0f);
    __builtin_memcpy(o + (int64_t)k * (L::VL * P), h, sizeof(h));
  }
}

// ================================================================ launchers
// Per-dispatch timing of the row kernels: while a timer is installed on the
// calling thread, they are launched through hipExtLaunchKernelGGL with a
// start and a stop event of the timer around each dispatch (the events take
// the dispatch's own begin and end, not the gaps between dispatches).
static thread_local DispatchTimer *g_timer = nullptr;
void set_dispatch_timer(DispatchTimer *t) { g_timer = t; }
double DispatchTimer::total_ms() const {
  double s = 0;
  for (int k = 0; k < used; k++) {
    float ms = 0;
    check(hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]), "dispatch timer");
    s += ms;
  }
  return s;
}
DispatchTimer::~DispatchTimer() {
  for (hipEvent_t e : ev) (void)hipEventDestroy(e);
}
static void timer_events(hipEvent_t *e0, hipEvent_t *e1) {
  DispatchTimer &t = *g_timer;
  if (2 * t.used + 1 >= (int)t.ev.size()) {
    for (int k = 0; k < 2; k++) {
      hipEvent_t e;
      check(hipEventCreate(&e), "event");
      t.ev.push_back(e);
    }
  }
  *e0 = t.ev[2 * t.used];
  *e1 = t.ev[2 * t.used + 1];
  t.used++;
}
template <typename... KA, typename... A>
static void launch(void (*k)(KA...), unsigned grid, unsigned block, hipStream_t st, A... a) {
  if (grid == 0) return;
  if (g_timer) {
    hipEvent_t e0, e1;
    timer_events(&e0, &e1);
    hipExtLaunchKernelGGL(k, dim3(grid), dim3(block), 0, st, e0, e1, 0, a...);
  } else {
    hipLaunchKernelGGL(k, dim3(grid), dim3(block), 0, st, a...);
  }
}

// lines of one class period per unit, planes of a set
static LineSet make_set(const DevLayout &D, int y0, int ys, int z0, int zs, int *units) {
  const int S = D.order == 2 ? 6 : 2, lpu = D.lg < 6 ? 64 >> D.lg : 1, last = D.M - 2;
  LineSet s{y0, ys, 0, z0, zs, 0};
  if (D.lg >= 6) s.upz = y0 <= last ? (last - y0) / ys + 1 : 0;
  for (int y = y0; D.lg < 6 && y <= last && y < y0 + S; y += ys) {
    s.nc++;
    s.upz += ((last - y) / S + 1 + lpu - 1) / lpu;
  }
  *units = z0 <= last ? s.upz * ((last - z0) / zs + 1) : 0;
  return s;
}
LineSet all_lines(const DevLayout &D, int *units) { return make_set(D, 1, 1, 1, 1, units); }
LineSet group_lines(const DevLayout &D, int g, int *units) {
  const int C = D.order == 2 ? 3 : 2, yr = g % C, zr = g / C;
  return make_set(D, yr ? yr : C, C, zr ? zr : C, C, units);
}
static unsigned unit_threads(const DevLayout &D) { return (unsigned)kSplits * std::max(64, 1 << D.lg); }

template <typename T>
void rows_apply(const DevLayout &D, int mode, const T *val, const T *x, const T *f, T *y, double omega,
                hipStream_t st, const T *psum) {
  int units;
  const LineSet s = all_lines(D, &units);
#define PMX_ROWS(O, MODE, HALF) \
  launch(k_line_rows<T, O, MODE, HALF>, (unsigned)units, unit_threads(D), st, s, D.lg, val, x, f, y, omega, psum)
#define PMX_ROWS_M(O)                      \
  if (psum) {                              \
    if (mode == 0) PMX_ROWS(O, 0, true);   \
    else PMX_ROWS(O, 1, true);             \
  } else {                                 \
    switch (mode) {                        \
      case 0: PMX_ROWS(O, 0, false); break;  \
      case 1: PMX_ROWS(O, 1, false); break;  \
      default: PMX_ROWS(O, 2, false); break; \
    }                                      \
  }
  if (D.order == 2) {
    PMX_ROWS_M(2)
  } else {
    PMX_ROWS_M(1)
  }
#undef PMX_ROWS_M
#undef PMX_ROWS
}

template <typename T, typename V>
static void sweep_group(const DevLayout &D, int g, int seq, int sums, const V *val, const float *dinv, T *x, const T *f,
                        T *psum, double omega, const int *bnd_set, hipStream_t st) {
  int units;
  const LineSet s = group_lines(D, g, &units);
  if (D.order == 2)
    launch(k_line_sweep<T, V, 2>, (unsigned)units, unit_threads(D), st, s, D.lg, seq, sums, val, x, f, psum, omega,
           bnd_set, dinv);
  else
    launch(k_line_sweep<T, V, 1>, (unsigned)units, unit_threads(D), st, s, D.lg, seq, sums, val, x, f, psum, omega,
           bnd_set, dinv);
}
template <typename T, typename V>
static void sweeps(const DevLayout &D, const V *val, const float *dinv, T *x, const T *f, T *psum, double omega,
                   bool ssor, int n, bool zero, const int *bnd_set, hipStream_t st) {
  const int G = D.order == 2 ? 9 : 4;
  for (int s = 0; s < n; s++) {
    const bool start = s == 0 && zero;
    const int *bs = start ? bnd_set : nullptr;
    // the last group turns a symmetric sweep around, the first one the next
    // sweep: both directions of its lines in one launch (the last group has no
    // lines after it, the first one none before it: their kept sum is zero)
    for (int g = ssor && s > 0 ? 1 : 0; g < G; g++) {
      const bool turn = ssor && g == G - 1;
      int sums = kSumLo;
      if (s > 0 && ssor) sums |= kSumKept;
      else if (!start) sums |= kSumHi;
      if (ssor) sums |= turn ? kKeepZero : kKeepLo;
      sweep_group<T, V>(D, g, turn ? kForwardBackward : kForward, sums, val, dinv, x, f, psum, omega, bs, st);
    }
    if (!ssor) continue;
    for (int g = G - 2; g >= 0; g--) {
      const bool turn = g == 0 && s + 1 < n;
      sweep_group<T, V>(D, g, turn ? kBackwardForward : kBackward, kSumHi | kSumKept | (turn ? kKeepZero : kKeepHi), val,
                        dinv, x, f, psum, omega, nullptr, st);
    }
  }
}
template <typename T>
void sor_sweeps(const DevLayout &D, const T *val, T *x, const T *f, T *psum, double omega, bool ssor, int n, bool zero,
                const int *bnd_set, hipStream_t st) {
  sweeps<T, T>(D, val, nullptr, x, f, psum, omega, ssor, n, zero, bnd_set, st);
}
void sor_sweeps_scaled(const DevLayout &D, const _Float16 *val16, const float *dinv, float *x, const float *f,
                       float *psum, double omega, bool ssor, int n, bool zero, const int *bnd_set, hipStream_t st) {
  sweeps<float, _Float16>(D, val16, dinv, x, f, psum, omega, ssor, n, zero, bnd_set, st);
}
void scaled_values(const DevLayout &D, const float *val, _Float16 *val16, float *dinv, hipStream_t st) {
  int units;
  const LineSet s = all_lines(D, &units);
  const unsigned g = (unsigned)units * (D.lg > 6 ? (1u << D.lg) / 64 : 1);
  if (D.order == 2) hipLaunchKernelGGL(k_scaled_values<2>, dim3(g), dim3(64), 0, st, s, D.lg, val, val16, dinv);
  else hipLaunchKernelGGL(k_scaled_values<1>, dim3(g), dim3(64), 0, st, s, D.lg, val, val16, dinv);
}
template <typename T>
void sweep_wg(const DevLayout &D, const T *val, T *x, const T *f, double omega, int ssor, hipStream_t st) {
  if (!sweep_wg_fits(D, sizeof(T))) throw std::logic_error("sweep_wg: level does not fit in LDS");
  const size_t lds = (size_t)D.N * sizeof(T);
  if (D.order == 2)
    hipLaunchKernelGGL((k_sweep_wg<T, 2>), dim3(1), dim3(kWgThreads), lds, st, D.lg, val, x, f, omega, ssor, D.boundary,
                       D.nboundary);
  else
    hipLaunchKernelGGL((k_sweep_wg<T, 1>), dim3(1), dim3(kWgThreads), lds, st, D.lg, val, x, f, omega, ssor, D.boundary,
                       D.nboundary);
}
template <typename T>
void coarse_wg(const DevLayout &D, const T *val, T *x, const T *f, double omega, int kind, int maxit, double red,
               T *xj, hipStream_t st) {
  if (!sweep_wg_fits(D, sizeof(T))) throw std::logic_error("coarse_wg: level does not fit in LDS");
  if (kind < 1 || kind > 3) throw std::invalid_argument("coarse_wg: smoother must be 1, 2 or 3");
  const size_t lds = (size_t)D.N * sizeof(T);
  if (D.order == 2)
    hipLaunchKernelGGL((k_coarse_wg<T, 2>), dim3(1), dim3(kWgThreads), lds, st, D.lg, val, x, f, omega, kind, maxit, red,
                       D.boundary, D.nboundary, xj);
  else
    hipLaunchKernelGGL((k_coarse_wg<T, 1>), dim3(1), dim3(kWgThreads), lds, st, D.lg, val, x, f, omega, kind, maxit, red,
                       D.boundary, D.nboundary, xj);
}

// Calibration kernels of the dispatch measurements: a dispatch that does
// nothing, and a plain streaming read (16 bytes per load, two loads per lane)
// whose sum reaches memory only in a case that never occurs.
__global__ void k_empty_dispatch() {}
__global__ __launch_bounds__(256) void k_stream_read(const float4 *__restrict__ a, int64_t n4,
                                                     float *__restrict__ sink) {
  const int64_t i = (int64_t)blockIdx.x * 512 + threadIdx.x;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    if (i + 256 * k < n4) {
      const float4 v = a[i + 256 * k];
      s += v.x + v.y + v.z + v.w;
    }
  }
  if (s == -1234567.0f) sink[0] = s;
}
void empty_dispatch(const DevLayout &D, int group, hipStream_t st) {
  int units;
  (void)group_lines(D, group, &units);
  launch(k_empty_dispatch, (unsigned)units, unit_threads(D), st);
}
void stream_read(const void *p, int64_t bytes, float *sink, hipStream_t st) {
  const int64_t n4 = bytes / 16;
  if (n4 < 1) return;
  if ((reinterpret_cast<uintptr_t>(p) & 15) != 0) throw std::invalid_argument("stream_read: 16-byte alignment");
  launch(k_stream_read, (unsigned)((n4 + 511) / 512), 256u, st, static_cast<const float4 *>(p), n4, sink);
}

#define PMX_INST(T)                                                                                              \
  template void rows_apply<T>(const DevLayout &, int, const T *, const T *, const T *, T *, double, hipStream_t,  \
                              const T *);                                                                        \
  template void sor_sweeps<T>(const DevLayout &, const T *, T *, const T *, T *, double, bool, int, bool,        \
                              const int *, hipStream_t);                                                         \
  template void sweep_wg<T>(const DevLayout &, const T *, T *, const T *, double, int, hipStream_t);              \
  template void coarse_wg<T>(const DevLayout &, const T *, T *, const T *, double, int, int, double, T *, hipStream_t);
PMX_INST(double)
PMX_INST(float)

}  // namespace pmx
