// pmx_lines.hpp -- device side of the line layout (see pmx_internal.hpp): the
// order of a line's groups, the lines of a launch, and the accumulation of
// groups that the row kernels share.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pmx_internal.hpp"

namespace pmx {

// The (dy, dz) groups of a line in storage order, per class of lines (y mod S,
// z mod S): first the groups whose lines come before the line in the sweep
// order ((z mod C, y mod C), y fastest), then the line itself, then the
// others; each part in (dz, dy) order.
template <int O> struct GroupTable {
  using L = Lines<O>;
  int off[L::S * L::S][L::kMaxGroups];  // (dy + 8) + 16 (dz + 8)
  int pos[L::S * L::S][25];             // storage position of (dy, dz) at (dy + 2) + 5 (dz + 2), -1 if absent
  int nlo[L::S * L::S];                 // groups before the line itself
  int ng[L::S * L::S];                  // all groups
};
template <int O> constexpr GroupTable<O> make_group_table() {
  using L = Lines<O>;
  GroupTable<O> t{};
  for (int b = 0; b < L::S; b++)
    for (int a = 0; a < L::S; a++) {
      const int c = a + L::S * b, ey = L::ext(a), ez = L::ext(b), me = (b % L::C) * L::C + a % L::C;
      for (int i = 0; i < 25; i++) t.pos[c][i] = -1;
      int k = 0;
      for (int part = 0; part < 3; part++) {
        if (part == 1) t.nlo[c] = k;
        for (int dz = -ez; dz <= ez; dz++)
          for (int dy = -ey; dy <= ey; dy++) {
            const int g = ((b + dz + L::S) % L::C) * L::C + (a + dy + L::S) % L::C;
            const bool own = dy == 0 && dz == 0;
            if (!((part == 0 && g < me) || (part == 1 && own) || (part == 2 && g > me))) continue;
            t.pos[c][(dy + 2) + 5 * (dz + 2)] = k;
            t.off[c][k++] = (dy + 8) + 16 * (dz + 8);
          }
      }
      t.ng[c] = k;
    }
  return t;
}
static __device__ constexpr GroupTable<1> kGroups1 = make_group_table<1>();
static __device__ constexpr GroupTable<2> kGroups2 = make_group_table<2>();
template <int O> __device__ __forceinline__ const GroupTable<O> &group_table() {
  if constexpr (O == 1) return kGroups1;
  else return kGroups2;
}
template <int O> __device__ __forceinline__ int line_class(int y, int z) {
  return y % Lines<O>::S + Lines<O>::S * (z % Lines<O>::S);
}

// value of row (x, y, z) for the column at (dx, dy, dz)
template <int O>
__device__ __forceinline__ int64_t value_index(int P, int x, int y, int z, int dx, int dy, int dz) {
  using L = Lines<O>;
  const int k = group_table<O>().pos[line_class<O>(y, z)][(dy + 2) + 5 * (dz + 2)];
  return ((L::group_base(P, y, z) + k) * L::VL + L::slot(x, dx)) * P + ((x - 1) >> 1);
}
// the same in the FP16 smoother values (a pair's slots of a group contiguous)
template <int O>
__device__ __forceinline__ int64_t value_index16(int P, int x, int y, int z, int dx, int dy, int dz) {
  using L = Lines<O>;
  const int k = group_table<O>().pos[line_class<O>(y, z)][(dy + 2) + 5 * (dz + 2)];
  return ((L::group_base(P, y, z) + k) * P + ((x - 1) >> 1)) * L::VL + L::slot(x, dx);
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

// The stored values of a group for the row pair of a lane: element s at
// v[s * P] (FP64, FP32), contiguous (FP16).
template <typename V, int O> __device__ __forceinline__ void load_group(const V *v, int P, V *out) {
  constexpr int VL = Lines<O>::VL;
  if constexpr (sizeof(V) == 2) {
    __builtin_memcpy(out, v, VL * sizeof(V));
  } else {
#pragma unroll
    for (int s = 0; s < VL; s++) out[s] = v[s * P];
  }
}
// offset of a lane's values in a line, and of consecutive groups
template <typename V, int O> __device__ __forceinline__ int64_t line_values(int P, int64_t base, int m) {
  constexpr int VL = Lines<O>::VL;
  if constexpr (sizeof(V) == 2) return (base * P + m) * VL;
  else return base * VL * P + m;
}

// Adds groups k0, k0 + step, ... < k1 of a line to the sums of a lane's row
// pair, x = 2m + 1 (so) and 2m + 2 (se).  v: the lane's values of group 0; x:
// lattice vector at (2m, y, z); d3: distance of the run's second part (3, or
// less for the last pair, whose even row is the boundary node and has zero
// values: its columns are clamped to the lattice).  The order of the sums is
// that of k, whatever the unrolling.
template <typename T, typename V, int O, int U>
__device__ __forceinline__ void add_groups(const V *__restrict__ v, const T *x, const int *__restrict__ off, int k0,
                                           int k1, int step, int P, int M, int d3, T &so, T &se) {
  constexpr int VL = Lines<O>::VL, NX = O == 2 ? 5 : 4;
  auto fetch = [&](int k, V *w, T *r) {
    const int o = off[k];
    const T *q = x + ((o & 15) - 8 + M * ((o >> 4) - 8)) * M;
    load_group<V, O>(v + (int64_t)k * (VL * P), P, w);
    load_run<T, 3>(q, r);
    load_run<T, NX - 3>(q + d3, r + 3);
  };
  auto add = [&](const V *w, const T *r) {
#pragma unroll
    for (int e = 0; e < 3; e++) so = fma((T)w[e], r[e], so);
#pragma unroll
    for (int e = 0; e < 2 * O + 1; e++) se = fma((T)w[3 + e], r[e + 2 - O], se);
  };
  int k = k0;
  for (; k + (U - 1) * step < k1; k += U * step) {
    V w[U][VL];
    T r[U][NX];
#pragma unroll
    for (int u = 0; u < U; u++) fetch(k + u * step, w[u], r[u]);
#pragma unroll
    for (int u = 0; u < U; u++) add(w[u], r[u]);
  }
  for (; k < k1; k += step) {
    V w[VL];
    T r[NX];
    fetch(k, w, r);
    add(w, r);
  }
}

}  // namespace pmx
