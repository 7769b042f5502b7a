// pmx_lines.hpp -- device side of the line layout (see pmx_internal.hpp): the
// order of a line's groups, the lines of a launch, and the accumulation of
// groups that the row kernels share.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pmx_internal.hpp"

namespace pmx {

// The (dy, dz) groups of a line in storage order: the planes dz whose lattice
// planes come before the line's in the sweep order (z mod C), then the line's
// own plane, then the others; in a plane dz != 0 the lines dy = -ey .. ey, in
// its own plane the lines before it (y mod C), itself, the lines after it.  An
// axis gives its offsets in this order as nibbles (offset + 2) of a word,
// computed and not read from memory: a sweep launch of a few microseconds
// would wait for the table.
struct AxisOrder {
  unsigned seq;  // nibble i: i-th offset + 2
  int e, lo;     // half extent, offsets before 0
};
template <int O> __device__ __forceinline__ AxisOrder axis_order(int t) {
  const int e = Lines<O>::ext(t);
  if constexpr (O == 1) {
    // (t mod 2) = 0: 0, -1, 1; 1: -1, 1, 0
    const bool r = t & 1;
    return AxisOrder{r ? 0x231u : 0x312u, 1, r ? 2 : 0};
  } else {
    // residues mod 3; the extent 2 offsets +-2 have the residue of -+1
    const int r = t % 3;
    const bool w = e == 2;
    const unsigned q0 = w ? 0x43102u : 0x312u;  // 0 | -2 -1 1 2
    const unsigned q1 = w ? 0x30241u : 0x321u;  // -1 2 | 0 | -2 1
    const unsigned q2 = w ? 0x24310u : 0x231u;  // -2 -1 1 2 | 0
    return AxisOrder{r == 0 ? q0 : r == 1 ? q1 : q2, e, r == 0 ? 0 : r == 1 ? (w ? 2 : 1) : (w ? 4 : 2)};
  }
}
template <int O> struct GroupOrder {
  AxisOrder y, z;
  __device__ __forceinline__ GroupOrder(int ly, int lz) : y(axis_order<O>(ly)), z(axis_order<O>(lz)) {}
  __device__ __forceinline__ int wy() const { return 2 * y.e + 1; }
  __device__ __forceinline__ int groups() const { return wy() * (2 * z.e + 1); }
  __device__ __forceinline__ int before() const { return z.lo * wy() + y.lo; }
  // offset of group k in the lattice: dy + M dz
  __device__ __forceinline__ int line(int k, int M) const {
    // k / 3 and k / 5 for k < 25
    const int j = O == 1 || y.e == 1 ? (k * 11) >> 5 : (k * 13) >> 6, i = k - j * wy();
    const int dz = (int)((z.seq >> (4 * j)) & 15) - 2;
    const int dy = dz ? i - y.e : (int)((y.seq >> (4 * i)) & 15) - 2;
    return dy + M * dz;
  }
  // storage position of (dy, dz)
  __device__ __forceinline__ int position(int dy, int dz) const {
    int j = 0, i = dy + y.e;
    for (int q = 0; q < 5; q++)
      if (((z.seq >> (4 * q)) & 15) == (unsigned)(dz + 2) && q <= 2 * z.e) j = q;
    if (dz == 0)
      for (int q = 0; q < 5; q++)
        if (((y.seq >> (4 * q)) & 15) == (unsigned)(dy + 2) && q <= 2 * y.e) i = q;
    return j * wy() + i;
  }
};

// value of row (x, y, z) for the column at (dx, dy, dz)
template <typename V, int O>
__device__ __forceinline__ int64_t value_index(int P, int x, int y, int z, int dx, int dy, int dz) {
  using L = Lines<O>;
  const int k = GroupOrder<O>(y, z).position(dy, dz);
  return (L::group_base(P, y, z) + k) * (L::VL * P) + Slots<V, O>::at(P, (x - 1) >> 1, L::slot(x, dx));
}

// MI355X dispatches consecutive workgroups round-robin over its 8 XCDs.  Remap
// so that each XCD works on one contiguous slice of the launch: the
// neighbouring lines whose x values a block gathers then stay in that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int G) {
  const int X = 8;
  const int q = G / X, r = G % X, xcd = bid % X, k = bid / X;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
}

// The lines a unit of lanes works on: `lanes` = max(64, P) lanes hold
// lanes / P lines of one class, S apart in y.  Unit b of a launch over the
// lines z = set.z0 + set.zs kz, y = set.y0 + set.ys j: one line per unit in
// this order, or (P < 64) the classes set.y0 + c set.ys, c < set.nc, in turn.
struct UnitLines {
  int y0, z;  // first line; line li of the unit is (y0 + S li, z)
};
template <int O> __device__ __forceinline__ UnitLines unit_lines(const LineSet &s, int M, int lg, int b) {
  using L = Lines<O>;
  const int kz = b / s.upz;
  int r = b - kz * s.upz, y = s.y0;
  if (lg >= 6) return UnitLines{y + s.ys * r, s.z0 + s.zs * kz};
  const int lpu = 6 - lg;  // log2 of the lines per unit
  for (int c = 1; c < s.nc; c++) {
    const int n = (((M - 2 - y) / L::S + 1) + (1 << lpu) - 1) >> lpu;
    if (r < n) break;
    r -= n;
    y += s.ys;
  }
  return UnitLines{y + L::S * (r << lpu), s.z0 + s.zs * kz};
}

// W consecutive elements at q in as few loads as their alignment allows
template <typename T, int W> __device__ __forceinline__ void load_run(const T *q, T *r) {
  __builtin_memcpy(r, q, W * sizeof(T));
}

// The stored values of a group (at v) for row pair m.
template <typename V, int O> __device__ __forceinline__ void load_group(const V *v, int P, int m, V *out) {
  using S = Slots<V, O>;
#pragma unroll
  for (int c = 0; c < S::VL; c += S::W) __builtin_memcpy(out + c, v + S::at(P, m, c), S::width(c) * sizeof(V));
}
// first value of a line
template <int O> __device__ __forceinline__ int64_t line_values(int P, int y, int z) {
  return Lines<O>::group_base(P, y, z) * (Lines<O>::VL * P);
}

// Adds groups k0, k0 + step, ... < k1 of a line to the sums of a lane's row
// pair, x = 2m + 1 (so) and 2m + 2 (se).  v: the line's values; x:
// lattice vector at (2m, y, z); d3: distance of the run's second part (3, or
// less for the last pair, whose even row is the boundary node and has zero
// values: its columns are clamped to the lattice).  The order of the sums is
// that of k, whatever the unrolling.
template <typename T, typename V, int O, int U>
__device__ __forceinline__ void add_groups(const V *__restrict__ v, const T *x, const GroupOrder<O> &g, int k0, int k1,
                                           int step, int P, int M, int m, int d3, T &so, T &se) {
  constexpr int VL = Lines<O>::VL, NX = O == 2 ? 5 : 4;
  auto fetch = [&](int k, V *w, T *r) {
    const T *q = x + g.line(k, M) * M;
    load_group<V, O>(v + (int64_t)k * (VL * P), P, m, w);
    load_run<T, 3>(q, r);
    load_run<T, NX - 3>(q + d3, r + 3);
  };
  auto add = [&](const V *w, const T *r) {
#pragma unroll
    for (int e = 0; e < 3; e++) so = fma((T)w[e], r[e], so);
#pragma unroll
    for (int e = 0; e < 2 * O + 1; e++) se = fma((T)w[3 + e], r[e + 2 - O], se);
  };
  // all loads of U groups are issued before the first sum (past the last group
  // it is read again and not added)
  for (int k = k0; k < k1; k += U * step) {
    V w[U][VL];
    T r[U][NX];
#pragma unroll
    for (int u = 0; u < U; u++) fetch(k + u * step < k1 ? k + u * step : k, w[u], r[u]);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (u == 0 || k + u * step < k1) add(w[u], r[u]);
  }
}

}  // namespace pmx
