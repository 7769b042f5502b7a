// pmx_internal.hpp -- internal data model of libpmx (not part of the C-ABI).
//
// Layout in HBM.  Every level of the hierarchy is a uniformly refined unit
// cube with n = 2^nref cells per direction.  Its Q1/Q2 nodes form a lattice of
// M = order*n + 1 points per direction, and every device vector is stored in
// lattice order (x fastest), length M^3.  The reference DOF numbering
// (ConstructSpace) is only used at the boundary: `lat2dof`/`dof2lat` permute
// between the two.
//
// Operators are stored in the "line layout".  Interior rows are paired along x
// (rows 2m + 1 and 2m + 2, m < P = (M - 1) / 2: an odd and an even node; the
// last even one is the boundary node x = M - 1, whose values are zero), and a
// pair's entries are grouped by the lattice line (y + dy, z + dz) of their
// columns.  A line (y, z) stores its groups one after another, a group holds
// VL = 3 + (2 order + 1) slots per pair (the odd row's 3 entries, dx = -1 .. 1,
// then the even row's, dx = -order .. order) in chunks of 16 bytes (2 FP64, 4
// FP32, 8 FP16 slots; the last chunk holds the rest), chunk after chunk:
//   val[(group_base(P, y, z) + k) * VL * P + Slots<V, order>::at(P, m, s)]
// so that the P lanes of a line load contiguous 16-byte chunks and no column
// index is stored.  (One slot per load costs the same on long lines, but on
// the 8 pairs of a 17^3 line each load touches 8 lines for 32 bytes of each.)
// A group's run of x values (5 for Q2, 4 for Q1) serves both rows of the pair.  The groups of a line whose own lines come before it in
// the sweep order are stored first (k < nlo), then the line itself, then the
// others, so a half sweep streams one contiguous part of each line.
//
// Sweep order.  The multicolour smoother takes the colours of (x, y, z) mod C
// (C = 2 for Q1, 3 for Q2) with x fastest.  Lines with equal (y mod C, z mod C)
// do not couple, so all of them are swept in one launch, each by its own
// workgroup, which takes the x colours of its line one after another: C^2
// launches for the C^3 colours, in the same order of updates.
// Dirichlet rows (lattice boundary) are identity and not stored.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

namespace pmx {

constexpr int kBlock = 256;       // threads per workgroup of the operator kernels
constexpr int kRowsPerBlock = 64; // rows per workgroup of the one-thread-per-row kernels
constexpr int64_t kSweepLdsBytes = 48 * 1024;  // largest x staged in LDS by the single-workgroup kernel
constexpr int kSplits = 4;           // partial sums of a row: group k belongs to partial k mod 4
constexpr int kRedBlocks = 1024;  // partial sums of the deterministic reductions

#if defined(__HIPCC__)
#define PMX_HD __host__ __device__
#else
#define PMX_HD
#endif

// arithmetic of the line layout for order O (1: Q1, 2: Q2)
template <int O> struct Lines {
  static constexpr int C = O == 2 ? 3 : 2;       // colours per axis
  static constexpr int S = O == 2 ? 6 : 2;       // period of the line structure (extent and colour)
  static constexpr int VL = 3 + 2 * O + 1;       // slots of a row pair per group
  static constexpr int kMaxGroups = O == 2 ? 25 : 9;
  // half extent of the stencil along an axis at lattice coordinate t
  PMX_HD static constexpr int ext(int t) { return O == 2 && (t & 1) == 0 ? 2 : 1; }
  PMX_HD static constexpr int width(int t) { return 2 * ext(t) + 1; }
  // sum of the widths of coordinates 1 .. t - 1
  PMX_HD static constexpr int width_sum(int t) {
    return O == 2 ? 8 * ((t - 1) >> 1) + (((t - 1) & 1) ? 3 : 0) : 3 * (t - 1);
  }
  PMX_HD static constexpr int width_total(int P) { return width_sum(2 * P); }
  // groups stored before line (y, z)
  PMX_HD static constexpr int64_t group_base(int P, int y, int z) {
    return (int64_t)width_sum(z) * width_total(P) + width(z) * width_sum(y);
  }
  // slot of column offset dx in row x of a pair
  PMX_HD static constexpr int slot(int x, int dx) { return (x & 1) ? dx + 1 : 3 + dx + O; }
  PMX_HD static constexpr int64_t values(int P) {
    return (int64_t)width_total(P) * width_total(P) * VL * P;
  }
};

// position of slot s of pair m in a group of values of type V
template <typename V, int O> struct Slots {
  static constexpr int VL = Lines<O>::VL, W = 16 / (int)sizeof(V);  // slots per chunk
  PMX_HD static constexpr int width(int c) { return VL - c < W ? VL - c : W; }  // of the chunk at slot c
  PMX_HD static constexpr int at(int P, int m, int s) {
    return (s / W) * W * P + m * width(s / W * W) + s % W;
  }
};

// the lines of a launch (see unit_lines in pmx_lines.hpp)
struct LineSet {
  int y0, ys, nc;  // y classes y0 + c ys, c < nc
  int z0, zs;      // planes z0 + zs kz
  int upz;         // units per plane
};

// residue class of interior nodes mod (2 for Q1, 6 for Q2): one smoother
// colour and one stencil shape
struct Segment {
  int rx, ry, rz;     // residues
  int x0, y0, z0;     // first interior lattice coordinate of the class
  int cx, cy, cz;     // node counts per direction
  int ex, ey, ez;     // stencil half extents
  int colour;
  int ns;             // entries per row (2ex+1)(2ey+1)(2ez+1)
  int64_t count;      // cx*cy*cz
};

struct Layout {
  int nref = 0, order = 1, n = 0, M = 0, S = 2;
  int64_t N = 0;            // lattice nodes = DOFs
  int64_t nactive = 0;      // interior nodes
  int ncolours = 8;
  std::vector<Segment> segs;
  // entries of the interior rows with the rows of each class rounded up to a
  // multiple of 16 (reported by pmx_system_dims)
  int64_t nvals = 0;
  int64_t nstored = 0;      // values of the line layout
  int64_t max_colour_rows = 0;
  std::vector<int> boundary;  // lattice indices of Dirichlet nodes
};

// host mesh / numbering products (the TFESpace3D + TSquareStructure3D data)
struct Numbering {
  int64_t ncells = 0;
  int nb = 8;
  int64_t N = 0, active = 0;
  std::vector<int> begin_index, global_numbers;  // reference numbering
  std::vector<int> lat2dof, dof2lat;
  std::vector<int> rowptr, kcol;                 // built on demand
  bool have_csr = false;
  // per lattice cell (cx + n (cy + n cz)): the signs of e1 + e2 + e3 of the
  // cell's frame in the refinement tree (bit d set: +1 along axis d), i.e. the
  // direction from the cell centre to its reference point (a, a, a)
  std::vector<uint8_t> corner;
};

void build_layout(Layout &L, int nref, int order, int block);
void build_numbering(Numbering &Nb, const Layout &L);
void build_csr(Numbering &Nb, const Layout &L);

// legacy-VTK file of nvar scalar functions (reference numbering) on the
// level's hexahedra, in the layout of TOutput3D::WriteVtk
void write_vtk(const Layout &L, const Numbering &Nb, int nvar, const char *const *names,
               const double *const *values, const char *path);

// reference-numbering colour of a DOF (the multicolour smoother class)
int node_colour(const Layout &L, int x, int y, int z);

}  // namespace pmx
