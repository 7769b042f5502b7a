// pmx_ops.hip -- operator, transfer, assembly and Krylov kernels (gfx950) and
// their stream-ordered launchers.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdlib>
#include <cstdio>
#include <stdexcept>
#include <type_traits>
#include <utility>

#include "pmx_functors.hpp"
#include "pmx_kernels.hpp"
#include "pmx_lines.hpp"
#include "pmx_ops.hpp"

namespace pmx {

__global__ __launch_bounds__(kBlock) void k_reduce_final(const double *__restrict__ part, int np,
                                                         double *__restrict__ out, int do_sqrt) {
  double s = 0;
  for (int i = threadIdx.x; i < np; i += kBlock) s += part[i];
  s = block_sum<double>(s);
  if (threadIdx.x == 0) out[0] = do_sqrt ? sqrt(s) : s;
}

// flag = 1 if a and b differ in any bit (all writers store the same value)
__global__ void k_bits_differ(const double *__restrict__ a, const double *__restrict__ b, int64_t n,
                              int *__restrict__ flag) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (__double_as_longlong(a[i]) != __double_as_longlong(b[i])) *flag = 1;
}
// ============================================================ transfers
// 1D taps of the nodal interpolation from the coarse to the fine lattice
// (the prolongation matrices of FEDatabase3D.C:1656 for Q1/Q2 Lagrange,
// averaged over the cells sharing a fine DOF as MGComponents3D.C:208-488
// does, which for a continuous interpolant is the interpolant itself).
// Taps are held in fixed slots (Q1: 2 prolongation / 3 restriction slots per
// axis, Q2: 3 / 5) in increasing lattice order; a slot that a node does not
// use gets weight 0 and a clamped index, and the kernels add its term as an
// exact 0.  Every load of a node is then issued before the first product
// (no data-dependent trip counts), and the sum runs over the same terms in
// the same order as over the used taps alone, so the result is the same bit
// for bit.
template <int ORDER> struct TransferTaps {
  static constexpr int P = ORDER == 1 ? 2 : 3;  // prolongation taps per axis
  static constexpr int R = ORDER == 1 ? 3 : 5;  // restriction taps per axis
};
template <int ORDER>
__device__ __forceinline__ void prolong_taps(int x, int nc, int *ci, double *w) {
  if (ORDER == 1) {
    const int c = x >> 1;
    const bool odd = x & 1;
    ci[0] = c; w[0] = odd ? 0.5 : 1.0;
    ci[1] = odd ? c + 1 : c; w[1] = odd ? 0.5 : 0.0;
    return;
  }
  int e = x >> 2;
  if (e > nc - 1) e = nc - 1;
  const int r = x - 4 * e;
  ci[0] = 2 * e; ci[1] = 2 * e + 1; ci[2] = 2 * e + 2;
  w[0] = r == 0 ? 1.0 : r == 1 ? 0.375 : r == 3 ? -0.125 : 0.0;
  w[1] = r == 2 ? 1.0 : (r == 1 || r == 3) ? 0.75 : 0.0;
  w[2] = r == 4 ? 1.0 : r == 1 ? -0.125 : r == 3 ? 0.375 : 0.0;
}
// transposed taps: fine nodes feeding coarse node y (DefectRestriction = P^T)
template <int ORDER>
__device__ __forceinline__ void restrict_taps(int y, int Mf, int *fi, double *w) {
  constexpr int R = TransferTaps<ORDER>::R;
  int off[R];
  double ww[R];
  if (ORDER == 1) {
    off[0] = -1; off[1] = 0; off[2] = 1;
    ww[0] = 0.5; ww[1] = 1.0; ww[2] = 0.5;
  } else {
    const bool even = (y & 1) == 0;
    off[0] = -3; off[1] = -1; off[2] = 0; off[3] = 1; off[4] = 3;
    ww[0] = even ? -0.125 : 0.0; ww[1] = even ? 0.375 : 0.75; ww[2] = 1.0; ww[3] = even ? 0.375 : 0.75;
    ww[4] = even ? -0.125 : 0.0;
  }
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int x = 2 * y + off[k];
    const bool in = x >= 0 && x < Mf;
    fi[k] = in ? x : 0;
    w[k] = in ? ww[k] : 0.0;
  }
}

// ADD = 0: xf = P xc.  ADD = 1: xf += damp (P xc with 0 on the lattice
// surface), i.e. prolongation, CorrectNodes and the damped update in one
// pass (the Dirichlet nodes of every layout are its lattice surface)
template <typename T, int ORDER, int ADD>
__global__ __launch_bounds__(kBlock) void k_prolong(const T *__restrict__ xc, T *__restrict__ xf, int Mc, int Mf,
                                                    double damp) {
  constexpr int P = TransferTaps<ORDER>::P;
  // 32-bit index arithmetic (the launcher checks that the lattice fits)
  const unsigned id = blockIdx.x * kBlock + threadIdx.x;
  const unsigned Nf = (unsigned)Mf * Mf * Mf;
  if (id >= Nf) return;
  const unsigned yz = id / (unsigned)Mf;
  const int x = id - yz * Mf, y = yz % (unsigned)Mf, z = yz / (unsigned)Mf;
  const int nc = (Mc - 1) / ORDER;
  int ix[P], iy[P], iz[P];
  double wx[P], wy[P], wz[P];
  prolong_taps<ORDER>(x, nc, ix, wx);
  prolong_taps<ORDER>(y, nc, iy, wy);
  prolong_taps<ORDER>(z, nc, iz, wz);
  T v[P][P][P];
#pragma unroll
  for (int c = 0; c < P; c++)
#pragma unroll
    for (int b = 0; b < P; b++) {
      const T *row = xc + (unsigned)Mc * (iy[b] + (unsigned)Mc * iz[c]);
#pragma unroll
      for (int a = 0; a < P; a++) v[c][b][a] = row[ix[a]];
    }
  // arithmetic in T: the tap weights and their products are exact in FP32
  T s = 0;
#pragma unroll
  for (int c = 0; c < P; c++)
#pragma unroll
    for (int b = 0; b < P; b++) {
      const T wzy = (T)wz[c] * (T)wy[b];
#pragma unroll
      for (int a = 0; a < P; a++) {
        const T t = wzy * (T)wx[a] * v[c][b][a];
        s += (wz[c] != 0.0 && wy[b] != 0.0 && wx[a] != 0.0) ? t : T(0);
      }
    }
  if (ADD) {
    const bool surface = x == 0 || y == 0 || z == 0 || x == Mf - 1 || y == Mf - 1 || z == Mf - 1;
    xf[id] += (T)damp * (surface ? T(0) : s);
  } else {
    xf[id] = s;
  }
}
// xc: 0 on the coarse lattice surface and xc = 0 (CorrectDefect and Reset fused)
template <typename T, int ORDER>
__global__ __launch_bounds__(kBlock) void k_restrict(T *__restrict__ rc, const T *__restrict__ rf, int Mc, int Mf,
                                                     T *__restrict__ xc) {
  constexpr int R = TransferTaps<ORDER>::R;
  const unsigned id = blockIdx.x * kBlock + threadIdx.x;
  const unsigned Nc = (unsigned)Mc * Mc * Mc;
  if (id >= Nc) return;
  const unsigned yz = id / (unsigned)Mc;
  const int x = id - yz * Mc, y = yz % (unsigned)Mc, z = yz / (unsigned)Mc;
  int ix[R], iy[R], iz[R];
  double wx[R], wy[R], wz[R];
  restrict_taps<ORDER>(x, Mf, ix, wx);
  restrict_taps<ORDER>(y, Mf, iy, wy);
  restrict_taps<ORDER>(z, Mf, iz, wz);
  T s = 0;
#pragma unroll
  for (int c = 0; c < R; c++)
#pragma unroll
    for (int b = 0; b < R; b++) {
      const T wzy = (T)wz[c] * (T)wy[b];
      const T *row = rf + (unsigned)Mf * (iy[b] + (unsigned)Mf * iz[c]);
#pragma unroll
      for (int a = 0; a < R; a++) {
        const T t = wzy * (T)wx[a] * row[ix[a]];
        s += (wz[c] != 0.0 && wy[b] != 0.0 && wx[a] != 0.0) ? t : T(0);
      }
    }
  if (xc) xc[id] = T(0);
  if (xc && (x == 0 || y == 0 || z == 0 || x == Mc - 1 || y == Mc - 1 || z == Mc - 1)) s = 0;
  rc[id] = s;
}

// ============================================================ assembly
// Coefficients at quadrature point q of cell (cx, cy, cz), in the canonical
// (axis-aligned) frame of the lattice: {w|detJ|, eps, b0, b1, b2, c, f, delta}.
// with_delta = false: the record without its stabilisation parameter
// (o[7] = 0), for callers that read it from the per-point buffer of
// k_qp_delta
template <bool CHEAP = false>
__device__ __forceinline__ void qp_coeffs(const double *__restrict__ prm, const double *__restrict__ qref, int n,
                                          int cx, int cy, int cz, int q, int form, double *o,
                                          const uint8_t *__restrict__ corner = nullptr, bool with_delta = true) {
  const double h = 1.0 / n;
  const double xi = qref[4 * q], eta = qref[4 * q + 1], zeta = qref[4 * q + 2], w = qref[4 * q + 3];
  // THexaAffin::GetOrigFromRef: X = xc0 + xc1 xi + ... with xc0 the cell centre
  const double X = (cx * h + 0.5 * h) + 0.5 * h * xi;
  const double Y = (cy * h + 0.5 * h) + 0.5 * h * eta;
  const double Z = (cz * h + 0.5 * h) + 0.5 * h * zeta;
  const QpCoeffs c = example_coeffs<CHEAP>(prm, X, Y, Z);
  if (!with_delta) {
    o[0] = w * (h * h * h / 8.0);
    o[1] = c.eps; o[2] = c.b0; o[3] = c.b1; o[4] = c.b2; o[5] = c.c; o[6] = c.f; o[7] = 0.0;
    return;
  }
  if (corner && (int)prm[PMX_PRM_CELL_MEASURE] == 4) {
    // the coefficients at the reference's first point of the cell, (a, a, a)
    // with a = qref[0] in the cell's own frame: centre + (h/2) a (e1 + e2 + e3)
    const int code = corner[cx + (int64_t)n * (cy + (int64_t)n * cz)];
    const double a = 0.5 * h * qref[0];
    const QpCoeffs c0 = example_coeffs(prm, (cx * h + 0.5 * h) + ((code & 1) ? a : -a),
                                       (cy * h + 0.5 * h) + ((code & 2) ? a : -a),
                                       (cz * h + 0.5 * h) + ((code & 4) ? a : -a));
    qp_record(prm, form, h, w, c, o, &c0);
  } else {
    qp_record(prm, form, h, w, c, o);
  }
}
// Stage 1 (coefficient functions that are expensive to evaluate): the
// coefficients of every quadrature point of every cell, once.
__global__ __launch_bounds__(kBlock) void k_qp_data(const double *__restrict__ prm, const double *__restrict__ qref,
                                                    int nq, int n, double *__restrict__ out,
                                                    const uint8_t *__restrict__ corner) {
  const int64_t id = blockIdx.x * (int64_t)kBlock + threadIdx.x;
  const int64_t ncell = (int64_t)n * n * n;
  if (id >= ncell * nq) return;
  const int q = id % nq;
  const int64_t cell = id / nq;
  const int cx = cell % n, cy = (cell / n) % n, cz = cell / ((int64_t)n * n);
  qp_coeffs(prm, qref, n, cx, cy, cz, q, (int)prm[PMX_PRM_FORM], out + id * 8, corner);
}
// The stabilisation parameter alone (record entry 7) of every quadrature
// point of every cell, once: the per-row evaluation of the inline
// coefficient functions would otherwise compute it (a square root, a
// hyperbolic tangent and divisions) once for each of the up to 8 rows that
// share a cell.  Point-major, dl[q * n^3 + cell], so that the rows of a
// wavefront (cells two apart along x) read nearby entries.  Grid: x over the
// cells of one z-plane, y = q * n + cz.
__global__ __launch_bounds__(kBlock) void k_qp_delta(const double *__restrict__ prm, const double *__restrict__ qref,
                                                     int n, double *__restrict__ dl) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * n) return;
  const int cx = t % n, cy = t / n;
  const int cz = blockIdx.y % n, q = blockIdx.y / n;
  double o[8];
  qp_coeffs<true>(prm, qref, n, cx, cy, cz, q, (int)prm[PMX_PRM_FORM], o);
  dl[(int64_t)q * n * n * n + t + (int64_t)n * n * cz] = o[7];
}
// forms whose records carry a stabilisation parameter
__host__ __device__ inline bool form_has_delta(int form) {
  return form == PMX_FORM_SDFEM || form == PMX_FORM_MASS_SUPG || form == PMX_FORM_RHS_SUPG ||
         form == PMX_FORM_TCD_SUPG_AK;
}
// The curl-Fourier convection (fourier_b) without a cosine per mode and
// point.  The quadrature rules are tensor products (point q = ix + np (iy +
// np iz) at (xi_ix, xi_iy, xi_iz)), so the phase of mode m at point q of cell
// (cx, cy, cz), 2 pi k . X + phi, is a_x(cx, ix) + a_y(cy, iy) + a_z(cz, iz)
// with a_d = 2 pi k_d X_d along one axis (phi in a_x), and
// cos(phase) = Re(e^{i a_x} e^{i a_y} e^{i a_z}).  The per-axis factors are
// one table per level (mode, axis, cell index, 1D point); a point then costs
// two complex products per mode instead of a cosine, and the three loads of
// a mode touch one cache line per wavefront.  The values differ from the
// direct evaluation by rounding only.
__host__ __device__ inline int rule_points_1d(int nq) { return nq <= 8 ? 2 : (nq <= 27 ? 3 : 4); }
template <bool GRF>
__global__ __launch_bounds__(kBlock) void k_phase_tables(const double *__restrict__ prm,
                                                           const double *__restrict__ qref, int nq, int n,
                                                           double *__restrict__ tab) {
  const int np = rule_points_1d(nq);
  const int id = blockIdx.x * kBlock + threadIdx.x;
  if (id >= (GRF ? kGrfModes : kFourierModes) * 3 * n * np) return;
  const int ci = id % (n * np), d = (id / (n * np)) % 3, m = id / (3 * n * np);
  const int c = ci / np, i = ci % np;
  const double twopi = 6.283185307179586476925286766559;
  const double h = 1.0 / n;
  const double *t = GRF ? prm + PMX_PRM_GRF + m * 4 : prm + PMX_PRM_FOURIER + m * 5;
  // point i of the 1D rule is the first coordinate of point q = i
  const double X = (c * h + 0.5 * h) + 0.5 * h * qref[4 * i];
  const double a = GRF ? t[d] * X + (d == 0 ? t[3] : 0.0) : twopi * t[1 + d] * X + (d == 0 ? t[4] : 0.0);
  tab[2 * id] = cos(a);
  tab[2 * id + 1] = sin(a);
}
// The curl-Fourier coefficients (eps, b, c = 0, f = 1 as example_coeffs) at
// the 1D points (ix, iy, iz) of cell (cx, cy, cz) from the table above.
__device__ __forceinline__ QpCoeffs fourier_coeffs_tab(const double *__restrict__ prm,
                                                       const double *__restrict__ tab, int n, int np, int cx, int cy,
                                                       int cz, int ix, int iy, int iz) {
  const double twopi = 6.283185307179586476925286766559;
  const int64_t L = (int64_t)n * np;  // entries per (mode, axis)
  double dA[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll 4
  for (int m = 0; m < kFourierModes; m++) {
    const double *t = prm + PMX_PRM_FOURIER + m * 5;
    const double *fx = tab + 2 * ((m * 3 + 0) * L + cx * np + ix);
    const double *fy = tab + 2 * ((m * 3 + 1) * L + cy * np + iy);
    const double *fz = tab + 2 * ((m * 3 + 2) * L + cz * np + iz);
    const double r1 = fx[0] * fy[0] - fx[1] * fy[1], i1 = fx[0] * fy[1] + fx[1] * fy[0];
    const double cs = t[0] * (r1 * fz[0] - i1 * fz[1]) * twopi;
    const int c = m / 8;
    dA[c][0] += cs * t[1];
    dA[c][1] += cs * t[2];
    dA[c][2] += cs * t[3];
  }
  const double sc = prm[PMX_PRM_BSCALE];
  QpCoeffs k;
  k.eps = prm[PMX_PRM_EPS];
  k.b0 = sc * (dA[2][1] - dA[1][2]);
  k.b1 = sc * (dA[0][2] - dA[2][0]);
  k.b2 = sc * (dA[1][0] - dA[0][1]);
  k.c = 0;
  k.f = 1.0;
  return k;
}
// Stage 1 for the curl-Fourier example: the records of k_qp_data with the
// coefficients from the table above.  A thread takes the np points of one
// x-line (iy, iz) of a cell: per mode it reads the y and z factors once and
// the np x factors, so the table reads per point (the bound of this kernel:
// 24 modes x 3 complex factors per point) drop from 3 to 1 + 2/np complex
// values.  Per point and mode the products and sums are those of
// fourier_coeffs_tab, in the same order.
// Grid: x over the (cx, iy, iz) lines of one row of cells, y = cy + n cz;
// the rule size is a template parameter so that no index needs a runtime
// division.
template <int NQ>
__global__ __launch_bounds__(kBlock) void k_qp_data_fourier(const double *__restrict__ prm,
                                                            const double *__restrict__ qref, int n,
                                                            const double *__restrict__ tab, double *__restrict__ out,
                                                            const uint8_t *__restrict__ corner) {
  constexpr int np = NQ == 8 ? 2 : (NQ == 27 ? 3 : 4);
  static_assert(np * np * np == NQ, "tensor rule");
  constexpr int NL = np * np;  // x-lines per cell
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * NL) return;
  const int cx = t / NL, r = t % NL, iy = r % np, iz = r / np;
  const int cy = blockIdx.y % n, cz = blockIdx.y / n;
  const double twopi = 6.283185307179586476925286766559;
  const int64_t L = (int64_t)n * np;  // entries per (mode, axis)
  double dA[np][3][3];
#pragma unroll
  for (int i = 0; i < np; i++)
#pragma unroll
    for (int c = 0; c < 3; c++) dA[i][c][0] = dA[i][c][1] = dA[i][c][2] = 0.0;
  // modes 8 c .. 8 c + 7 belong to component c of the potential (the
  // component loop is unrolled so that every accumulator index is a constant)
#pragma unroll
  for (int c = 0; c < 3; c++) {
#pragma unroll 2
    for (int mm = 0; mm < kFourierModes / 3; mm++) {
      const int m = (kFourierModes / 3) * c + mm;
      const double *tm = prm + PMX_PRM_FOURIER + m * 5;
      const double *fx = tab + 2 * ((m * 3 + 0) * L + cx * np);
      const double *fy = tab + 2 * ((m * 3 + 1) * L + cy * np + iy);
      const double *fz = tab + 2 * ((m * 3 + 2) * L + cz * np + iz);
      const double fy0 = fy[0], fy1 = fy[1], fz0 = fz[0], fz1 = fz[1];
      const double t0 = tm[0], t1 = tm[1], t2 = tm[2], t3 = tm[3];
#pragma unroll
      for (int ix = 0; ix < np; ix++) {
        const double fx0 = fx[2 * ix], fx1 = fx[2 * ix + 1];
        const double r1 = fx0 * fy0 - fx1 * fy1, i1 = fx0 * fy1 + fx1 * fy0;
        const double cs = t0 * (r1 * fz0 - i1 * fz1) * twopi;
        dA[ix][c][0] += cs * t1;
        dA[ix][c][1] += cs * t2;
        dA[ix][c][2] += cs * t3;
      }
    }
  }
  const double sc = prm[PMX_PRM_BSCALE];
  const bool cm4 = corner && (int)prm[PMX_PRM_CELL_MEASURE] == 4;
  QpCoeffs k0;
  if (cm4) {
    // the coefficients at the reference's first point of the cell, (a, a, a)
    // in its own frame: 1D point 0 (a) along an axis where the frame points
    // forward, np - 1 (-a; the rules are symmetric) where it points back
    const int code = corner[cx + (int64_t)n * (cy + (int64_t)n * cz)];
    k0 = fourier_coeffs_tab(prm, tab, n, np, cx, cy, cz, (code & 1) ? 0 : np - 1, (code & 2) ? 0 : np - 1,
                            (code & 4) ? 0 : np - 1);
  }
  const int64_t cell = cx + (int64_t)n * (blockIdx.y);
#pragma unroll
  for (int ix = 0; ix < np; ix++) {
    QpCoeffs k;
    k.eps = prm[PMX_PRM_EPS];
    k.b0 = sc * (dA[ix][2][1] - dA[ix][1][2]);
    k.b1 = sc * (dA[ix][0][2] - dA[ix][2][0]);
    k.b2 = sc * (dA[ix][1][0] - dA[ix][0][1]);
    k.c = 0;
    k.f = 1.0;
    const int q = ix + np * r;
    double *o = out + (cell * NQ + q) * 8;
    if (cm4) qp_record(prm, (int)prm[PMX_PRM_FORM], 1.0 / n, qref[4 * q + 3], k, o, &k0);
    else qp_record(prm, (int)prm[PMX_PRM_FORM], 1.0 / n, qref[4 * q + 3], k, o);
  }
}
// ... and for the log-normal example, eps exp(sigma g) with the field g of
// grf_field, a sum of cosines at 64 frequencies: a cosine of the sum of three
// phases is the real part of the product of the tables' factors, 2 operations per
// point and mode behind the product of a line's y and z factors.  (Evaluating the
// cosines was all of an assembly: 13.2 ms of 15.5 at 128^3 cells, 27 points.)
// 64^3 cells and the levels below: 1.37 -> 0.34 ms.
template <int NQ>
__global__ __launch_bounds__(kBlock) void k_qp_data_grf(const double *__restrict__ prm,
                                                        const double *__restrict__ qref, int n,
                                                        const double *__restrict__ tab, double *__restrict__ out) {
  constexpr int np = NQ == 8 ? 2 : (NQ == 27 ? 3 : 4);
  // a thread takes the np x np points of a cell with one z
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * np) return;
  const int cx = t / np, iz = t % np;
  const int cy = blockIdx.y % n, cz = blockIdx.y / n;
  const int64_t L = (int64_t)n * np;  // entries per (mode, axis)
  double s[np][np];
#pragma unroll
  for (int i = 0; i < np * np; i++) s[i / np][i % np] = 0;
#pragma unroll 2
  for (int m = 0; m < kGrfModes; m++) {
    const double *fx = tab + 2 * ((m * 3 + 0) * L + cx * np);
    const double *fy = tab + 2 * ((m * 3 + 1) * L + cy * np);
    const double *fz = tab + 2 * ((m * 3 + 2) * L + cz * np + iz);
#pragma unroll
    for (int y = 0; y < np; y++) {
      const double pr = fy[2 * y] * fz[0] - fy[2 * y + 1] * fz[1], pi = fy[2 * y] * fz[1] + fy[2 * y + 1] * fz[0];
#pragma unroll
      for (int i = 0; i < np; i++) s[y][i] += fx[2 * i] * pr - fx[2 * i + 1] * pi;
    }
  }
  const int64_t cell = cx + (int64_t)n * blockIdx.y;
  QpCoeffs k;
  k.c = prm[PMX_PRM_C];
  k.b0 = prm[PMX_PRM_B0];
  k.b1 = prm[PMX_PRM_B1];
  k.b2 = prm[PMX_PRM_B2];
  k.f = 1.0;
#pragma unroll 1
  for (int y = 0; y < np; y++)
#pragma unroll
    for (int i = 0; i < np; i++) {
      double g = s[0][i];
#pragma unroll
      for (int c = 1; c < np; c++) g = y == c ? s[c][i] : g;
      k.eps = prm[PMX_PRM_EPS] * exp(prm[PMX_PRM_GRF_SIGMA] * (g * kGrfScale));
      const int q = i + np * (y + np * iz);
      qp_record(prm, (int)prm[PMX_PRM_FORM], 1.0 / n, qref[4 * q + 3], k, out + (cell * NQ + q) * 8);
    }
}
// examples whose coefficients are cheaper to evaluate again than to read back
__host__ __device__ inline bool coeffs_inline(int example) {
  return example == PMX_EX_LAPLACE || example == PMX_EX_SINE_CD || example == PMX_EX_HEAT_AMC ||
         example == PMX_EX_ROTATING;
}

// Stage 2: row gather.  The thread of active node p visits the cells that
// contain p, forms row a of each local matrix
//   K_ab = sum_q w [ u0 phi_b + u . grad phi_b ]
// with s_a = phi_a + delta b.grad phi_a, u0 = c s_a, u = eps grad phi_a + b s_a
// (BilinearAssemble / _SD, ConvDiff3D.C:118-145,182-213; mass and TCD forms,
// TCD3D.C:37-322), and adds it into its own row of values.  No two threads write
// the same row, so no atomics and no colouring of cells are needed, and the
// writes of a wavefront are coalesced.
// The incident cells per direction are compile-time (a Q2 node with an odd
// coordinate lies in one cell along it, every other node in two), so the
// loops are uniform across the wavefront and the basis tables are read with
// scalar loads; val2 is the second matrix of the SUPG TCD form.
struct RowPoint {
  double u0, ux, uy, uz, k0, f;  // of K_ab, of the second matrix, of the rhs
};
// a quadrature point's factors of a row, with the row's basis function (value
// fa and physical derivatives) there
__device__ __forceinline__ RowPoint row_point(const double *Qq, double fa, double gax, double gay, double gaz, int form,
                                              double g) {
  const double w = Qq[0], eps = Qq[1], b0 = Qq[2], b1 = Qq[3], b2 = Qq[4];
  const double cc = Qq[5], ff = Qq[6], dl = Qq[7];
  const double bga = b0 * gax + b1 * gay + b2 * gaz;
  RowPoint r;
  // the rhs is f (phi_a + delta b.grad phi_a), with delta = 0 for the Galerkin
  // rhs and for MatrixMRhsAssemble (TCD3D.C:64, 117)
  const double sa = fa + dl * bga;
  r.f = w * ff * sa;
  if (form == PMX_FORM_MASS || form == PMX_FORM_MASS_SUPG) {
    r.u0 = fa;
    r.ux = r.uy = r.uz = r.k0 = 0;
  } else {
    r.u0 = cc * sa;
    r.ux = eps * gax + b0 * sa;
    r.uy = eps * gay + b1 * sa;
    r.uz = eps * gaz + b2 * sa;
    r.k0 = dl * bga;
  }
  r.u0 *= w;
  r.ux *= w * g;
  r.uy *= w * g;
  r.uz *= w * g;
  r.k0 *= w;
  return r;
}
template <int ORDER, int EX, int EY, int EZ, bool INL, bool RONLY>
__device__ __forceinline__ void assemble_row(int px, int py, int pz, int M, int n, int nq, int form,
                                             const double *__restrict__ prm, const double *__restrict__ qref,
                                             const double *__restrict__ qp, const double *__restrict__ tab,
                                             double *__restrict__ val, double *__restrict__ val2,
                                             double *__restrict__ rhs) {
  constexpr int NCX = (ORDER == 2 && EX == 1) ? 1 : 2;
  constexpr int NCY = (ORDER == 2 && EY == 1) ? 1 : 2;
  constexpr int NCZ = (ORDER == 2 && EZ == 1) ? 1 : 2;
  constexpr int K = ORDER + 1, NB = K * K * K;
  const int p = px + M * (py + M * pz);
  const double g = 2.0 * n;  // reference -> physical derivative factor 2/h
  // the row's entries: group position of (dy, dz), slot of dx
  const int P = (M - 1) / 2;
  const int64_t v0 = line_values<ORDER>(P, py, pz);
  const GroupOrder<ORDER> go(__builtin_amdgcn_readfirstlane(py), __builtin_amdgcn_readfirstlane(pz));
  auto at = [&](int dx, int dy, int dz) {
    return v0 + go.position(dy, dz) * (Lines<ORDER>::VL * P) +
           Slots<double, ORDER>::at(P, (px - 1) >> 1, Lines<ORDER>::slot(px, dx));
  };
  double frhs = 0;
  // incident cells per direction: lattice coordinate x lies in cells
  // floor((x-1)/ORDER) .. floor(x/ORDER) (two cells at a vertex plane)
  constexpr int UNR = ORDER == 1 ? 2 : 1;  // (right-hand sides of Q1: the 8 cells; 4.7 -> 4.4 ms there)
  const int cx0 = (px - 1) / ORDER, cy0 = (py - 1) / ORDER, cz0 = (pz - 1) / ORDER;
#pragma unroll UNR
  for (int iz = 0; iz < NCZ; iz++)
#pragma unroll UNR
    for (int iy = 0; iy < NCY; iy++)
#pragma unroll UNR
      for (int ix = 0; ix < NCX; ix++) {
        const int cx = cx0 + ix, cy = cy0 + iy, cz = cz0 + iz;
        const int ax = px - ORDER * cx, ay = py - ORDER * cy, az = pz - ORDER * cz;
        const int a = ax + K * (ay + K * az);
        const int64_t cell = cx + (int64_t)n * (cy + (int64_t)n * cz);
        const double *Q = qp + cell * nq * 8;
        double acc[NB], acc2[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) acc[b] = acc2[b] = 0;
        // inline coefficients: qp holds the per-point stabilisation
        // parameters of k_qp_delta (nullptr for the forms without one), read
        // one point ahead
        const int64_t ncell = (int64_t)n * n * n;
        double dl_next = (INL && qp) ? qp[cell] : 0.0;
        for (int q = 0; q < nq; q++) {
          double Qq[8];
          if (INL) {
            qp_coeffs<true>(prm, qref, n, cx, cy, cz, q, form, Qq, nullptr, false);
            Qq[7] = dl_next;
            if (qp) dl_next = qp[(q + 1 < nq ? q + 1 : q) * ncell + cell];
          } else {
#pragma unroll
            for (int e = 0; e < 8; e++) Qq[e] = Q[8 * q + e];
          }
          const double *Ta = tab + (q * NB + a) * 4;
          const RowPoint r = row_point(Qq, Ta[0], g * Ta[1], g * Ta[2], g * Ta[3], form, g);
          frhs += r.f;
          if (RONLY) continue;
          const double *Tq = tab + q * NB * 4;
#pragma unroll
          for (int b = 0; b < NB; b++) {
            const double *Tb = Tq + 4 * b;
            acc[b] += r.u0 * Tb[0] + r.ux * Tb[1] + r.uy * Tb[2] + r.uz * Tb[3];
            acc2[b] += r.k0 * Tb[0];
          }
        }
        if (RONLY) continue;
        // add the row into the value slots of node p
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const int bx = b % K, by = (b / K) % K, bz = b / (K * K);
          const int dx = ORDER * cx + bx - px, dy = ORDER * cy + by - py, dz = ORDER * cz + bz - pz;
          val[at(dx, dy, dz)] += acc[b];
          val2[at(dx, dy, dz)] += acc2[b];
        }
      }
  rhs[p] = frhs;
}

// Rows of the one-thread-per-row assembly kernels: 64 row pairs of a unit's
// lines (unit_lines), the odd rows in one workgroup and the even rows in
// another, so that a wavefront's rows have one stencil shape and its stores of a
// slot are contiguous.
// Q2: a row has 1, 2, 4 or 8 cells, by the parities of its coordinates.
// Workgroups go to the shader engines in turn, so that shapes which alternate
// with a short period put all the long rows on the same ones.  Units therefore
// come in runs of kShapeRun, and a run's workgroups part by part and (one line
// per unit) parity of y by parity of y.  Two-matrix form of the sine example, 64
// points, 64^3 / 32^3: parts alternating 34.5 / 4.2 ms, runs of 8 22.1 / 3.6 ms,
// of 16 22.5 / 3.6 ms, of 64 23.7 / 3.6 ms.
struct RowBlock {
  int part;  // parity of x, segment of the line
  UnitLines u;
};
constexpr int kShapeRun = 8;
template <int O> __device__ __forceinline__ RowBlock row_block(const LineSet &set, int M, int lg) {
  const int b = xcd_remap(blockIdx.x, gridDim.x), parts = lg > 6 ? (1 << lg) / 32 : 2;
  if (O == 1) return RowBlock{b % parts, unit_lines<O>(set, M, lg, b / parts)};
  const int kz = b / (parts * set.upz), r = b - kz * (parts * set.upz);
  const int first = r / (parts * kShapeRun) * kShapeRun, i = r - parts * first;
  const int n = set.upz - first < kShapeRun ? set.upz - first : kShapeRun;
  const int part = i / n;
  int j = i - part * n;
  if (lg >= 6) {
    const int h = (n + 1) >> 1;
    j = j < h ? 2 * j : 2 * (j - h) + 1;
  }
  return RowBlock{part, unit_lines<O>(set, M, lg, kz * set.upz + first + j)};
}
// False: no row.
template <int O>
__device__ __forceinline__ bool unit_row(const RowBlock &b, int M, int lg, int lane, int *px, int *py, int *pz) {
  const int P = 1 << lg, t = lane + 64 * (b.part >> 1), m = t & (P - 1);
  *px = 2 * m + 1 + (b.part & 1);
  *py = b.u.y0 + Lines<O>::S * (t >> lg);
  *pz = b.u.z;
  return *py <= M - 2 && *px <= M - 2;
}
// the same shape for the whole wavefront
template <int O> __device__ __forceinline__ int unit_shape(const RowBlock &b) {
  return __builtin_amdgcn_readfirstlane(Lines<O>::ext(1 + (b.part & 1)) * 100 + Lines<O>::ext(b.u.y0) * 10 +
                                        Lines<O>::ext(b.u.z));
}
static unsigned row_blocks(const DevLayout &D, int units) {
  return (unsigned)units * 2 * (D.lg > 6 ? (1u << D.lg) / 64 : 1);
}

template <int ORDER, bool INL, bool RONLY>
__global__ __launch_bounds__(kRowsPerBlock) void k_assemble(LineSet set, int lg, int M, int n, int nq,
                                                     const double *__restrict__ prm, const double *__restrict__ qref,
                                                     const double *__restrict__ qp, const double *__restrict__ tab,
                                                     double *__restrict__ val, double *__restrict__ val2,
                                                     double *__restrict__ rhs) {
  int px, py, pz;
  const RowBlock rb = row_block<ORDER>(set, M, lg);
  const bool ok = unit_row<ORDER>(rb, M, lg, threadIdx.x, &px, &py, &pz);
  const int code = unit_shape<ORDER>(rb);
  if (!ok) return;
  // (known to be uniform, they and what follows from them take the scalar
  // registers that the coefficients' constants need in the loop over the points;
  // right-hand side of the sine example at 128^3 Q1 4.41 -> 4.24 ms)
  asm volatile("" : "+v"(py), "+v"(pz));
  const int form = (int)prm[PMX_PRM_FORM];
#define PMX_AROW(O, EX, EY, EZ) \
  assemble_row<O, EX, EY, EZ, INL, RONLY>(px, py, pz, M, n, nq, form, prm, qref, qp, tab, val, val2, rhs)
  if (ORDER == 1) {
    PMX_AROW(1, 1, 1, 1);
    return;
  }
  switch (code) {
    case 111: PMX_AROW(2, 1, 1, 1); break;
    case 211: PMX_AROW(2, 2, 1, 1); break;
    case 121: PMX_AROW(2, 1, 2, 1); break;
    case 221: PMX_AROW(2, 2, 2, 1); break;
    case 112: PMX_AROW(2, 1, 1, 2); break;
    case 212: PMX_AROW(2, 2, 1, 2); break;
    case 122: PMX_AROW(2, 1, 2, 2); break;
    default: PMX_AROW(2, 2, 2, 2); break;
  }
#undef PMX_AROW
}
// a value that is the same in all lanes, in scalar registers
__device__ __forceinline__ double uniform(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned)u), hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
struct AxisPoint {
  double x, s, c;  // coordinate, sin(pi x), cos(pi x)
};
// Q1 rows with matrices: a workgroup takes the 64 rows of unit_row, its
// wavefront j the j-th of the rows' 8 cells (ix + 2 iy + 4 iz); the cells'
// rows of the local matrices meet in LDS and are added in the order of j, a
// slot of the 64 rows per wavefront and turn.
//
// Bound by the FP64 operations of the points and, on small levels, by the
// chain of a thread, which is 8 times shorter than with all cells of a row on
// one thread.  The rule and the basis are tensor products (NP points per
// axis), so a row is summed axis by axis (14 products per point instead of 32,
// no table of basis values).
// SRC: where the coefficients come from.  kInline: constant coefficients and a
// source of sines and cosines, two products per point from the factors of the
// axes (sine_coeffs); the rotating flow has a kernel without them.
// A workgroup has two wavefronts per SIMD, so a second one on the CU (68 KB of
// LDS with both matrices) needs at most 128 registers: a thread's sums over the
// points along x are kept in LDS, where they are needed at the end, and the
// points along z are a loop (rotating flow, both matrices 174 -> 118 registers;
// inline source 223 -> 126; both matrices with it take 148 and stay at one).
// 128^3, rotating flow: both matrices 2.36 -> 1.70 -> 1.29 ms (a row per thread,
// axis by axis, two workgroups), one 1.43 -> 1.10 ms.  8^3 and 16^3 cells, inline
// source: 331 -> 19.9 -> 17.2 us.
enum { kRecords = 0, kInline = 1, kRotating = 2 };
template <int NP, bool TWO, int SRC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(TWO && SRC == kInline ? 2 : 4)))
void k_assemble_q1(LineSet set, int lg, int M, int n, const double *__restrict__ prm, const double *__restrict__ qref,
                   const double *__restrict__ qp, double *__restrict__ val, double *__restrict__ val2,
                   double *__restrict__ rhs) {
  constexpr int NB = 8, R = kRowsPerBlock, NQ = NP * NP * NP;
  constexpr bool INL = SRC != kRecords;
  __shared__ double sh[(TWO ? 2 : 1) * 8 * NB * R], sf[8 * R];
  const int t = threadIdx.x & (R - 1), j = __builtin_amdgcn_readfirstlane(threadIdx.x / R);
  int px, py, pz;
  const bool ok = unit_row<1>(row_block<1>(set, M, lg), M, lg, t, &px, &py, &pz);
  // (a row that exists for the lanes without one)
  if (!ok) px = py = 1;
  const int form = (int)prm[PMX_PRM_FORM];
  {
    const int ix = j & 1, iy = (j >> 1) & 1, iz = j >> 2;
    const int cx = px - 1 + ix, cy = py - 1 + iy, cz = pz - 1 + iz;
    const int64_t cell = cx + (int64_t)n * (cy + (int64_t)n * cz), ncell = (int64_t)n * n * n;
    const double *Q = qp + cell * NQ * 8;
    const double h = 1.0 / n, g = 2.0 * n;  // reference -> physical derivative factor 2/h
    // (the basis functions of an axis have the derivatives -1/2, 1/2)
    const double gx = ix ? -0.5 * g : 0.5 * g, gy = iy ? -0.5 * g : 0.5 * g, gz = iz ? -0.5 * g : 0.5 * g;
    auto axis_point = [&](int c, double xi) {
      AxisPoint a{(c * h + 0.5 * h) + 0.5 * h * xi, 0, 0};
      if (SRC == kInline) sincospi(a.x, &a.s, &a.c);
      return a;
    };
    // kInline: constant coefficients and the factors of the source's terms; the
    // lines of a workgroup lie in one plane, so all of this is uniform
    SineCoeffs sc{};
    double zs[NP], zc[NP];
    if (SRC == kInline) {
      sc = sine_coeffs(prm);
      for (double *v : {&sc.sss, &sc.css, &sc.scs, &sc.ssc, &sc.scc}) *v = uniform(*v);
    }
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const AxisPoint Z = SRC == kInline ? axis_point(cz, qref[4 * i]) : AxisPoint{0, 0, 0};
      zs[i] = uniform(Z.s);
      zc[i] = uniform(Z.c);
    }
    double *acc = sh + j * NB * R + t, *acc2 = acc + 8 * NB * R, frhs = 0;  // this thread's: no barrier
    // inline coefficients: qp holds the per-point stabilisation parameters of
    // k_qp_delta (nullptr for the forms without one)
#pragma unroll 1
    for (int qx = 0; qx < NP; qx++) {
      const double xi = qref[4 * qx], x0 = uniform(0.5 * (1 - xi)), x1 = uniform(0.5 * (1 + xi)), fx = ix ? x0 : x1;
      const AxisPoint X = INL ? axis_point(cx, xi) : AxisPoint{0, 0, 0};
      double p[4] = {0, 0, 0, 0}, d[4] = {0, 0, 0, 0}, p2[4] = {0, 0, 0, 0};  // by + 2 bz
#pragma unroll 1
      for (int qy = 0; qy < NP; qy++) {
        const double yi = qref[4 * qy], y0 = uniform(0.5 * (1 - yi)), y1 = uniform(0.5 * (1 + yi)), fy = iy ? y0 : y1;
        const AxisPoint Y = INL ? axis_point(cy, yi) : AxisPoint{0, 0, 0};
        const double fs = (sc.sss * X.s + sc.css * X.c) * Y.s + sc.scs * X.s * Y.c;
        const double fc = X.s * (sc.ssc * Y.s + sc.scc * Y.c);
        const double gxy = gx * fy, gyx = gy * fx, gzxy = gz * (fx * fy), fxy = fx * fy;
        double dl[NP];
#pragma unroll
        for (int qz = 0; qz < NP; qz++)
          dl[qz] = (INL && qp) ? qp[(qx + NP * (qy + NP * qz)) * ncell + cell] : 0.0;
        double a[2] = {0, 0}, ax[2] = {0, 0}, ay[2] = {0, 0}, a2[2] = {0, 0};  // bz
#pragma unroll 1
        for (int qz = 0; qz < NP; qz++) {
          const int q = qx + NP * (qy + NP * qz);
          const double zi = qref[4 * qz], z0 = uniform(0.5 * (1 - zi)), z1 = uniform(0.5 * (1 + zi)), fz = iz ? z0 : z1;
          double Qq[8];
          if (INL) {
            QpCoeffs c;
            if constexpr (SRC == kRotating) c = rotating_coeffs(prm[PMX_PRM_EPS], X.x, Y.x);
            else c = QpCoeffs{sc.eps, sc.b0, sc.b1, sc.b2, sc.c, fs * zs[0] + fc * zc[0]};
            // (the next point's to the front; back in order after NP turns)
            const double zs0 = zs[0], zc0 = zc[0];
#pragma unroll
            for (int i = 0; i < NP; i++) {
              zs[i] = i + 1 < NP ? zs[i + 1] : zs0;
              zc[i] = i + 1 < NP ? zc[i + 1] : zc0;
            }
            Qq[0] = qref[4 * q + 3] * (h * h * h / 8.0);
            Qq[1] = c.eps; Qq[2] = c.b0; Qq[3] = c.b1; Qq[4] = c.b2; Qq[5] = c.c; Qq[6] = c.f;
            Qq[7] = dl[0];
#pragma unroll
            for (int i = 0; i + 1 < NP; i++) dl[i] = dl[i + 1];
          } else {
#pragma unroll
            for (int e = 0; e < 8; e++) Qq[e] = Q[8 * q + e];
          }
          const RowPoint r = row_point(Qq, fxy * fz, gxy * fz, gyx * fz, gzxy, form, g);
          frhs += r.f;
          a[0] = fma(r.u0, z0, fma(r.uz, -0.5, a[0]));
          a[1] = fma(r.u0, z1, fma(r.uz, 0.5, a[1]));
          ax[0] = fma(r.ux, z0, ax[0]);
          ax[1] = fma(r.ux, z1, ax[1]);
          ay[0] = fma(r.uy, z0, ay[0]);
          ay[1] = fma(r.uy, z1, ay[1]);
          if (TWO) {
            a2[0] = fma(r.k0, z0, a2[0]);
            a2[1] = fma(r.k0, z1, a2[1]);
          }
        }
#pragma unroll
        for (int bz = 0; bz < 2; bz++) {
          p[2 * bz] = fma(a[bz], y0, fma(ay[bz], -0.5, p[2 * bz]));
          p[2 * bz + 1] = fma(a[bz], y1, fma(ay[bz], 0.5, p[2 * bz + 1]));
          d[2 * bz] = fma(ax[bz], y0, d[2 * bz]);
          d[2 * bz + 1] = fma(ax[bz], y1, d[2 * bz + 1]);
          if (TWO) {
            p2[2 * bz] = fma(a2[bz], y0, p2[2 * bz]);
            p2[2 * bz + 1] = fma(a2[bz], y1, p2[2 * bz + 1]);
          }
        }
      }
#pragma unroll
      for (int b = 0; b < 4; b++) {
        double *o = acc + 2 * b * R, *o2 = acc2 + 2 * b * R;
        o[0] = fma(p[b], x0, fma(d[b], -0.5, qx ? o[0] : 0.0));
        o[R] = fma(p[b], x1, fma(d[b], 0.5, qx ? o[R] : 0.0));
        if (TWO) {
          o2[0] = fma(p2[b], x0, qx ? o2[0] : 0.0);
          o2[R] = fma(p2[b], x1, qx ? o2[R] : 0.0);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the compiler would keep the sums in registers)
    }
    sf[j * R + t] = frhs;
  }
  __syncthreads();
  if (!ok) return;
  const int P = (M - 1) / 2;
  const int64_t v0 = line_values<1>(P, py, pz);
  const GroupOrder<1> go(__builtin_amdgcn_readfirstlane(py), __builtin_amdgcn_readfirstlane(pz));
  for (int q = j; q < 27; q += 8) {
    // column dx lies in the cells ix = 0 (dx <= 0) and 1 (dx >= 0) along x as
    // their node dx + 1 - ix
    const int dx = q % 3 - 1, dy = (q / 3) % 3 - 1, dz = q / 9 - 1;
    double s = 0, s2 = 0;
    for (int iz = dz > 0; iz <= (dz >= 0); iz++)
      for (int iy = dy > 0; iy <= (dy >= 0); iy++)
        for (int ix = dx > 0; ix <= (dx >= 0); ix++) {
          const int c = ix + 2 * iy + 4 * iz, b = (dx + 1 - ix) + 2 * (dy + 1 - iy) + 4 * (dz + 1 - iz);
          s += sh[(c * NB + b) * R + t];
          if (TWO) s2 += sh[((8 + c) * NB + b) * R + t];
        }
    const int64_t at =
        v0 + go.position(dy, dz) * (Lines<1>::VL * P) + Slots<double, 1>::at(P, (px - 1) >> 1, Lines<1>::slot(px, dx));
    val[at] = s;
    if (TWO) val2[at] = s2;
  }
  if (j == 3) {  // (the others have four slots)
    double f = 0;
#pragma unroll
    for (int c = 0; c < 8; c++) f += sf[c * R + t];
    rhs[px + M * (py + M * pz)] = f;
  }
}
__global__ void k_scatter(double *__restrict__ y, const int *__restrict__ idx, const double *__restrict__ v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[idx[i]] = v[i];
}
void scatter(double *y, const int *idx, const double *v, int n, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(k_scatter, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, y, idx, v, n);
}
// Dirichlet rhs: RHS[dof] = g(node) (AssembleMat3D.C:1031-1096)
__global__ void k_boundary_rhs(const int *__restrict__ bnd, int nbd, int M, const double *__restrict__ prm,
                               double *__restrict__ rhs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nbd) return;
  const int p = bnd[i];
  const double h = 1.0 / (M - 1);
  const int x = p % M, y = (p / M) % M, z = p / (M * M);
  rhs[p] = example_bound_value(prm, x * h, y * h, z * h);
}

// ============================================================ CSR export
// entries in the reference CSR (sorted rows, Dirichlet rows = 1) from the
// line layout's values (FP16: the row-scaled smoother values)
template <typename T, int O>
__global__ void k_values_to_csr(const int *__restrict__ rowptr, const int *__restrict__ kcol,
                                const int *__restrict__ dof2lat, int64_t N, int64_t active, int M,
                                const T *__restrict__ val, double *__restrict__ out) {
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= N) return;
  const int b = rowptr[r], e = rowptr[r + 1], P = (M - 1) / 2;
  if (r >= active) { out[b] = 1.0; return; }
  const int p = dof2lat[r];
  const int x = p % M, y = (p / M) % M, z = p / (M * M);
  for (int n = b; n < e; n++) {
    const int q = dof2lat[kcol[n]];
    const int dx = q % M - x, dy = (q / M) % M - y, dz = q / (M * M) - z;
    out[n] = (double)val[value_index<T, O>(P, x, y, z, dx, dy, dz)];
  }
}

// The inverse of k_values_to_csr for the active rows: the entries of a CSR
// matrix with the level's pattern (reference numbering) into the line layout.
template <int O>
__global__ void k_csr_to_values(const int *__restrict__ rowptr, const int *__restrict__ kcol,
                                const int *__restrict__ dof2lat, int64_t active, int M,
                                const double *__restrict__ in, double *__restrict__ val) {
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= active) return;
  const int b = rowptr[r], e = rowptr[r + 1], P = (M - 1) / 2;
  const int p = dof2lat[r];
  const int x = p % M, y = (p / M) % M, z = p / (M * M);
  for (int n = b; n < e; n++) {
    const int q = dof2lat[kcol[n]];
    const int dx = q % M - x, dy = (q / M) % M - y, dz = q / (M * M) - z;
    val[value_index<double, O>(P, x, y, z, dx, dy, dz)] = in[n];
  }
}

// ============================================================ permutations
template <typename T, typename U>
__global__ void k_gather(T *__restrict__ out, const U *__restrict__ in, const int *__restrict__ map, int64_t n) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) out[i] = (T)in[map[i]];
}

// ============================================================ generic CSR
// y = A x on a caller CSR matrix (MatVect on any TSquareMatrix3D): 16 lanes per row
template <typename T>
__global__ __launch_bounds__(kBlock) void k_csr_spmv(int n, const int *__restrict__ rowptr,
                                                     const int *__restrict__ kcol, const T *__restrict__ val,
                                                     const T *__restrict__ x, T *__restrict__ y,
                                                     const T *__restrict__ b) {
  const int lane = threadIdx.x & 15;
  const int row = (blockIdx.x * kBlock + threadIdx.x) >> 4;
  if (row >= n) return;
  double s = 0;
  for (int j = rowptr[row] + lane; j < rowptr[row + 1]; j += 16) s += (double)val[j] * (double)x[kcol[j]];
  for (int o = 8; o > 0; o >>= 1) s += __shfl_down(s, o, 16);
  if (lane == 0) y[row] = b ? (T)((double)b[row] - s) : (T)s;
}

// ============================================================ dense coarse solve
// The coarsest operator is A = [A_II A_IB; 0 I] (interior rows I, Dirichlet
// rows B identity), so A^-1 f = [A_II^-1 (f_I - A_IB f_B); f_B].  The device
// keeps W = A_II^-1 [I_I, -A_IB] as an n_I x N matrix in lattice column order:
// y_I = W f (one wavefront per row, FP64), y_B = f_B.
// Bound by latency: a row of 729 columns is 12 loads of a lane.  kGemvLoads of
// them are in flight at a time (past the end the last column again, not added),
// and a workgroup has one row, so that the rows of a few hundred spread over the CUs.  343 rows of 729
// columns: FP32 vectors 8.4 -> 3.4 us, FP64 8.4 -> 3.0 us (four rows per workgroup,
// one load waited for after another).
constexpr int kGemvLoads = 8;
template <typename T>
__global__ __launch_bounds__(64) void k_gemv_coarse(int N, const double *__restrict__ W, const int *__restrict__ iidx,
                                                    const T *__restrict__ x, T *__restrict__ y) {
  const int lane = threadIdx.x, row = blockIdx.x;
  double s = 0;
  const double *a = W + (int64_t)row * N;
  for (int j0 = lane; j0 < N; j0 += 64 * kGemvLoads) {
    double av[kGemvLoads];
    T xv[kGemvLoads];
#pragma unroll
    for (int u = 0; u < kGemvLoads; u++) {
      const int j = j0 + 64 * u < N ? j0 + 64 * u : N - 1;
      av[u] = a[j];
      xv[u] = x[j];
    }
#pragma unroll
    for (int u = 0; u < kGemvLoads; u++)
      if (j0 + 64 * u < N) s += av[u] * (double)xv[u];
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if (lane == 0) y[iidx[row]] = (T)s;
}

// ============================================================ coarse inverse
// Augmented [A_II | R] (n_I x (n_I + N), row-major), R[i][p] = 1 for the
// interior node p of row i, -a(i, p) for Dirichlet columns p.
template <int O>
__global__ void k_values_to_aug(int M, const int *__restrict__ iidx, const int *__restrict__ cidx, int nI,
                                const double *__restrict__ val, double *__restrict__ aug, int64_t ld) {
  using L = Lines<O>;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nI) return;
  const int p = iidx[r], x = p % M, y = (p / M) % M, z = p / (M * M), P = (M - 1) / 2;
  double *row = aug + (int64_t)r * ld;
  row[nI + p] = 1.0;
  const int ex = L::ext(x), ey = L::ext(y), ez = L::ext(z);
  for (int dz = -ez; dz <= ez; dz++)
    for (int dy = -ey; dy <= ey; dy++)
      for (int dx = -ex; dx <= ex; dx++) {
        const int q = (x + dx) + M * ((y + dy) + M * (z + dz));
        const double v = val[value_index<double, O>(P, x, y, z, dx, dy, dz)];
        const int cq = cidx[q];
        if (cq >= 0) row[cq] = v;
        else row[nI + q] = -v;
      }
}
// Gauss-Jordan step c with partial pivoting, in one launch: every block finds
// the same pivot row (largest |a(r, c)| among rows not yet used as pivots,
// lowest index on ties), then eliminates column c from the other rows of its
// share.  Rows are not swapped or scaled (the pivot row and column c are
// read-only during the step); piv[c] records the pivot row.
__global__ __launch_bounds__(256) void k_gj_step(double *__restrict__ aug, int nI, int64_t ld, int c,
                                                 int *__restrict__ piv) {
  __shared__ unsigned char used[8192];
  __shared__ double bv[256];
  __shared__ int bix[256];
  for (int r = threadIdx.x; r < nI; r += 256) used[r] = 0;
  __syncthreads();
  for (int k = threadIdx.x; k < c; k += 256) used[piv[k]] = 1;
  __syncthreads();
  double best = -1.0;
  int arg = nI;
  for (int r = threadIdx.x; r < nI; r += 256) {
    if (used[r]) continue;
    const double a = fabs(aug[(int64_t)r * ld + c]);
    if (a > best) { best = a; arg = r; }
  }
  bv[threadIdx.x] = best;
  bix[threadIdx.x] = arg;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      const double b2 = bv[threadIdx.x + o];
      const int i2 = bix[threadIdx.x + o];
      if (b2 > bv[threadIdx.x] || (b2 == bv[threadIdx.x] && i2 < bix[threadIdx.x])) {
        bv[threadIdx.x] = b2;
        bix[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  const int pr = bix[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) piv[c] = pr;
  const double *prow = aug + (int64_t)pr * ld;
  const double pinv = 1.0 / prow[c];
  // this block's rows: r = blockIdx.x * 4 + 0..3, columns c+1 .. ld-1
  const int64_t w = ld - (c + 1);
  for (int q = 0; q < 4; q++) {
    const int r = blockIdx.x * 4 + q;
    if (r >= nI || r == pr) continue;
    double *row = aug + (int64_t)r * ld;
    const double f = row[c] * pinv;
    if (f == 0.0) continue;
    for (int64_t j = threadIdx.x; j < w; j += 256) row[c + 1 + j] -= f * prow[c + 1 + j];
  }
}
// kGjPanel Gauss-Jordan steps at once (nI <= kGjRows): k_gj_panel does them on
// the panel's columns alone, a row per thread, and leaves what they do to a row as the
// factors T of the panel's pivot rows, row += sum_k T[row][k] (pivot row k);
// k_gj_update does that to the columns behind the panel, from one copy of the
// matrix to the other.  Elimination and pivots (up to ties of 42 bits) are those
// of k_gj_step.  In the
// panel a column that has been eliminated holds the factors of its pivot row.
// Bound by the chain of the panel's steps; 343 rows: 2.65 ms by steps,
// 0.71 ms (27 + 6 us per panel).
constexpr int kGjPanel = 16, kGjRows = 1024;
__global__ __launch_bounds__(kGjRows) void k_gj_panel(const double *__restrict__ aug, int nI, int64_t ld, int c0, int nc,
                                                      int *__restrict__ piv, double *__restrict__ pval,
                                                      double *__restrict__ T) {
  constexpr int B = kGjPanel, W = kGjRows / 64;
  __shared__ unsigned long long best[2][W];
  __shared__ double prow[2][B];
  __shared__ unsigned char taken[kGjRows];
  const int r = threadIdx.x;
  // a row per thread
  double a[B];
#pragma unroll
  for (int j = 0; j < B; j++) a[j] = r < nI && j < nc ? aug[(int64_t)r * ld + c0 + j] : 0.0;
  if (r < W) best[0][r] = best[1][r] = 0;  // (of wavefronts that are not there)
  taken[r] = 0;
  __syncthreads();
  for (int k = r; k < c0; k += blockDim.x) taken[piv[k]] = 1;
  __syncthreads();
  bool used = taken[r] != 0;
#pragma unroll
  for (int k = 0; k < B; k++) {
    if (k >= nc) break;
    // the largest entry among the rows not yet used, the lowest row on ties:
    // the last 10 bits of the entry make room for the row
    const double m = fabs(a[k]);
    const unsigned long long low = kGjRows - 1;
    unsigned long long v = 0;
    if (r < nI && !used) v = ((m >= 0 ? __builtin_bit_cast(unsigned long long, m) : 0) & ~low) | (low - r);
    for (int o = 32; o > 0; o >>= 1) {
      const unsigned long long v2 = __shfl_down(v, o, 64);
      v = v2 > v ? v2 : v;
    }
    if ((r & 63) == 0) best[k & 1][r >> 6] = v;
    __syncthreads();
    v = best[k & 1][0];
#pragma unroll
    for (int i = 1; i < W; i++) v = best[k & 1][i] > v ? best[k & 1][i] : v;
    const int pr = (int)(low - (v & low));
    if (r == pr) {
#pragma unroll
      for (int j = 0; j < B; j++) prow[k & 1][j] = a[j];
      piv[c0 + k] = pr;
      pval[c0 + k] = a[k];
      used = true;
    }
    __syncthreads();
    const double f = r == pr ? 0.0 : a[k] * (1.0 / prow[k & 1][k]);
#pragma unroll
    for (int j = 0; j < B; j++)
      if (j != k) a[j] -= f * prow[k & 1][j];
    a[k] = -f;
  }
  if (r >= nI) return;
#pragma unroll
  for (int j = 0; j < B; j++) T[(int64_t)r * B + j] = j < nc ? a[j] : 0.0;
}
// columns c1 .. ld - 1 of `to` = those of `from` + T (pivot rows); 64 columns x 16 rows
__global__ __launch_bounds__(256) void k_gj_update(const double *__restrict__ from, double *__restrict__ to, int nI,
                                                   int64_t ld, int c0, int c1, const int *__restrict__ piv,
                                                   const double *__restrict__ T) {
  constexpr int B = kGjPanel;
  __shared__ double ts[16 * B];
  const int64_t j = c1 + (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
  const int r0 = blockIdx.y * 16, w = threadIdx.x >> 6;
  ts[threadIdx.x] = r0 + (int)threadIdx.x / B < nI ? T[(int64_t)r0 * B + threadIdx.x] : 0.0;
  double p[B];
#pragma unroll
  for (int k = 0; k < B; k++) p[k] = c0 + k < c1 && j < ld ? from[(int64_t)piv[c0 + k < c1 ? c0 + k : c0] * ld + j] : 0.0;
  __syncthreads();
  if (j >= ld) return;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int r = r0 + 4 * q + w;
    if (r >= nI) break;
    double v = from[(int64_t)r * ld + j];
#pragma unroll
    for (int k = 0; k < B; k++) v += ts[(4 * q + w) * B + k] * p[k];
    to[(int64_t)r * ld + j] = v;
  }
}
// W[i][p] = aug[piv[i]][nI + p] / (pivot i), the pivot aug[piv[i]][i] or pval[i]
__global__ void k_gj_finish(const double *__restrict__ aug, int nI, int N, int64_t ld, const int *__restrict__ piv,
                            const double *__restrict__ pval, double *__restrict__ W) {
  const int64_t id = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (id >= (int64_t)nI * N) return;
  const int i = (int)(id / N), p = (int)(id % N);
  const double *row = aug + (int64_t)piv[i] * ld;
  W[id] = row[nI + p] / (pval ? pval[i] : row[i]);
}

// ============================================================ FGMRES scalars
// Givens update of column i of H and of s (FgmresIte.C:194-222, 447-459),
// H stored column-major with leading dimension m+1; writes |s[i+1]| to res.
__global__ void k_givens(double *H, double *cs, double *sn, double *s, int i, int ld, double *res) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double *h = H + (int64_t)i * ld;
  for (int k = 0; k < i; k++) {
    const double t = cs[k] * h[k] + sn[k] * h[k + 1];
    h[k + 1] = -sn[k] * h[k] + cs[k] * h[k + 1];
    h[k] = t;
  }
  const double dx = h[i], dy = h[i + 1];
  double c, sg;
  if (dy == 0.0) { c = 1.0; sg = 0.0; }
  else if (fabs(dy) > fabs(dx)) { const double t = dx / dy; sg = 1.0 / sqrt(1.0 + t * t); c = t * sg; }
  else { const double t = dy / dx; c = 1.0 / sqrt(1.0 + t * t); sg = t * c; }
  cs[i] = c; sn[i] = sg;
  {
    const double t = c * h[i] + sg * h[i + 1];
    h[i + 1] = -sg * h[i] + c * h[i + 1];
    h[i] = t;
  }
  {
    const double t = c * s[i] + sg * s[i + 1];
    s[i + 1] = -sg * s[i] + c * s[i + 1];
    s[i] = t;
  }
  res[0] = fabs(s[i + 1]);
}
// back substitution of UpdateGmresIterate (FgmresIte.C:224-243): y = H^{-1} s
__global__ void k_backsolve(const double *H, const double *s, double *y, int k, int ld) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  for (int i = 0; i <= k; i++) y[i] = s[i];
  for (int i = k; i >= 0; i--) {
    y[i] /= H[(int64_t)i * ld + i];
    for (int j = i - 1; j >= 0; j--) y[j] -= H[(int64_t)i * ld + j] * y[i];
  }
}
// x += sum_j y[j] z_j over k+1 vectors (z stored contiguously, stride n)
template <typename T, typename X>
__global__ __launch_bounds__(kBlock) void k_multi_axpy(X *__restrict__ x, const T *__restrict__ z,
                                                       const double *__restrict__ y, int k1, int64_t n,
                                                       int64_t stride) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    double s = 0;
    for (int j = 0; j < k1; j++) s += y[j] * (double)z[j * stride + i];
    x[i] += (X)s;
  }
}
// write a scalar into H(i,j) from a reduction result
__global__ void k_set_scalar(double *dst, const double *src, double scale) {
  if (threadIdx.x == 0 && blockIdx.x == 0) dst[0] = scale * src[0];
}

// ================================================================ launchers
static inline int grid_for(int64_t n) {
  int64_t g = (n + kBlock - 1) / kBlock;
  if (g > 65535 * 8) g = 65535 * 8;
  return (int)(g < 1 ? 1 : g);
}

void check(hipError_t e, const char *what) {
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

template <typename T>
void fill(T *x, T v, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_fill<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, x, v, n);
}
bool bits_equal(const double *a, const double *b, int64_t n, int *flag, hipStream_t st) {
  fill<int>(flag, 0, 1, st);
  hipLaunchKernelGGL(k_bits_differ, dim3(grid_for(n)), dim3(kBlock), 0, st, a, b, n, flag);
  int h = 1;
  if (hipMemcpyAsync(&h, flag, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    throw std::runtime_error("bits_equal: copy failed");
  return h == 0;
}
// z = x and, on the lattice surface, y = x: the Dirichlet rows of y = A z in
// the copy that leaves z, a launch less per Krylov step (129^3 FP32: 6.5 us, in two
// launches 5.5 + 5.1)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_copy_surface(int M, T *__restrict__ z, const T *__restrict__ x,
                                                         T *__restrict__ y, unsigned n) {
  const unsigned i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const T v = x[i];
  z[i] = v;
  const unsigned yz = i / (unsigned)M, e = M - 1, ix = i - yz * M, iy = yz % (unsigned)M, iz = yz / (unsigned)M;
  if (ix == 0 || iy == 0 || iz == 0 || ix == e || iy == e || iz == e) y[i] = v;
}
template <typename T>
void copy_surface(const DevLayout &D, T *z, const T *x, T *y, hipStream_t st) {
  hipLaunchKernelGGL(k_copy_surface<T>, dim3((unsigned)((D.N + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, D.M, z, x, y,
                     (unsigned)D.N);
}
template <typename T>
void copy(T *y, const T *x, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_copy<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, y, x, n);
}
template <typename T>
void axpy(T *y, const T *x, const double *alpha_dev, double sgn, double ac, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_axpy<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, y, x, alpha_dev, sgn, ac, n);
}
template <typename T, typename U>
void convert(T *y, const U *x, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL((k_convert<T, U>), dim3(grid_for(n)), dim3(kBlock), 0, st, y, x, n);
}
template <typename T, typename U>
void add_convert(T *y, const U *x, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL((k_add_convert<T, U>), dim3(grid_for(n)), dim3(kBlock), 0, st, y, x, n);
}
template <typename T>
void scale_inv(T *y, const T *x, const double *nrm, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_scale_inv<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, y, x, nrm, n);
}
// The end of a defect r = f - A x: its Dirichlet rows, f - x on the lattice
// surface, and the norm, one workgroup of BLOCK threads per kDotChunk (up to
// kDefectSmall, 17^3: all) elements without a grid-stride loop, so that the number of
// partial sums grows with n; a single workgroup writes the norm itself.
// Bound by the launches: the surface, the sum and its last step as launches of
// their own took 5.6 us more at 9^3 (13.6 us per call).
// With the loads behind a branch per element a thread waited for each: calls
// among others at 33^3 (Q2) 15.7 -> 11.1 us, 65^3 (Q1) 20.5 -> 15.9 us, 65^3 (Q2)
// 39.2 -> 34.6 us.
constexpr int64_t kDefectSmall = 8 * 1024;
template <int BLOCK, int PER>
__global__ __launch_bounds__(BLOCK) void k_defect_norm(int M, double *r, const double *x, const double *f,
                                                       double *__restrict__ part, int64_t n, int last) {
  __shared__ double sh[BLOCK / 64];
  const int64_t base = (int64_t)blockIdx.x * (BLOCK * PER);
  // all loads are issued before the first is used (a branch around each would
  // wait for it): a lane of an interior row reads r in the place of f and x
  double a[PER], b[PER];
  bool surface[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const int64_t j = base + k * BLOCK + threadIdx.x, i = j < n ? j : n - 1;
    const unsigned yz = (unsigned)i / (unsigned)M;
    const int ix = (int)((unsigned)i - yz * M), iy = (int)(yz % (unsigned)M), iz = (int)(yz / (unsigned)M);
    surface[k] = ix == 0 || iy == 0 || iz == 0 || ix == M - 1 || iy == M - 1 || iz == M - 1;
    const double *pa = surface[k] ? f : r, *pb = surface[k] ? x : r;
    a[k] = pa[i];
    b[k] = pb[i];
  }
  double s = 0;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const int64_t i = base + k * BLOCK + threadIdx.x;
    const double v = surface[k] ? a[k] - b[k] : a[k];
    if (i >= n) continue;
    if (surface[k]) r[i] = v;
    s += v * v;
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    s = 0;
    for (int k = 0; k < BLOCK / 64; k++) s += sh[k];
    part[blockIdx.x] = last ? sqrt(s) : s;
  }
}
void defect_norm(const DevLayout &D, double *r, const double *x, const double *f, double *part, double *out,
                 hipStream_t st) {
  const int64_t n = D.N, nb = (n + kDotChunk - 1) / kDotChunk;
  if (n <= kDefectSmall) {
    auto *k = n <= 1024 ? k_defect_norm<1024, 1> : k_defect_norm<1024, kDefectSmall / 1024>;
    hipLaunchKernelGGL(k, dim3(1), dim3(1024), 0, st, D.M, r, x, f, out, n, 1);
    return;
  }
  hipLaunchKernelGGL((k_defect_norm<kBlock, kDotChunk / kBlock>), dim3((unsigned)nb), dim3(kBlock), 0, st, D.M, r, x, f,
                     part, n, 0);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kBlock), 0, st, part, (int)nb, out, 1);
}
template <typename T>
void dot(const T *x, const T *y, int64_t n, double *part, double *out, int do_sqrt, hipStream_t st) {
  int g = (int)((n + kBlock - 1) / kBlock);
  if (g > kRedBlocks) g = kRedBlocks;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(k_dot_partial<T>, dim3(g), dim3(kBlock), 0, st, x, y, part, n);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kBlock), 0, st, part, g, out, do_sqrt);
}

// ------------------------------------------------------- start of a cycle
template <typename T>
__global__ void k_start_zero(T *__restrict__ f, T *__restrict__ x, const T *__restrict__ v, int *__restrict__ bnd_set,
                             int64_t n) {
  const int64_t i0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i0 == 0) *bnd_set = 0;
  for (int64_t i = i0; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    f[i] = v[i];
    x[i] = T(0);
  }
}
template <typename T>
__global__ void k_start_boundary(const int *__restrict__ bnd, int nb, T *__restrict__ x, const T *__restrict__ f,
                                 int *__restrict__ bnd_set) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb) return;
  const T v = f[bnd[i]];
  x[bnd[i]] = v;
  if (v != T(0)) *bnd_set = 1;  // (every writer stores the same value; NaN counts)
}
template <typename T>
void start_zero(T *f, T *x, const T *v, int *bnd_set, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_start_zero<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, f, x, v, bnd_set, n);
}
template <typename T>
void start_boundary(const DevLayout &D, T *x, const T *f, int *bnd_set, hipStream_t st) {
  hipLaunchKernelGGL(k_start_boundary<T>, dim3((D.nboundary + kBlock - 1) / kBlock), dim3(kBlock), 0, st, D.boundary,
                     D.nboundary, x, f, bnd_set);
}

// ------------------------------------------------------- step length control
template <typename T>
__global__ void k_diff(T *__restrict__ e, const T *__restrict__ u, const T *__restrict__ uold, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    e[i] = u[i] - uold[i];
}
// omega = num / nom (param0 if nom <= 0 or |omega| < 0.1), u = uold + omega (u - uold)
template <typename T>
__global__ void k_step_length(T *__restrict__ u, const T *__restrict__ uold, const double *__restrict__ num_nom,
                              double param0, int64_t n) {
  const double num = num_nom[0], nom = num_nom[1];
  double omega = nom > 0 ? num / nom : param0;
  if (fabs(omega) < 0.1) omega = param0;
  const T a = (T)omega;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    u[i] = uold[i] + a * (u[i] - uold[i]);
}
template <typename T>
void axpy_diff(T *e, const T *u, const T *uold, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_diff<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, e, u, uold, n);
}
template <typename T>
void step_length_update(T *u, const T *uold, const double *num_nom, double param0, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_step_length<T>, dim3(grid_for(n)), dim3(kBlock), 0, st, u, uold, num_nom, param0, n);
}

// ------------------------------------------------------- Gram-Schmidt
// sum of the np partials in k_reduce_final's order, in every workgroup (the
// same bits everywhere), broadcast to the workgroup
__device__ __forceinline__ double sum_partials(const double *__restrict__ part, int np) {
  __shared__ double sh_total;
  double s = 0;
  for (int i = threadIdx.x; i < np; i += kBlock) s += part[i];
  s = block_sum<double>(s);
  if (threadIdx.x == 0) sh_total = s;
  __syncthreads();
  return sh_total;
}
// one modified Gram-Schmidt step: h = (w, v) from the partials of the
// previous launch (stored to *h by workgroup 0), w -= h v, and the partials
// of (w, next) for the following step (next = w: the squared norm).  The
// thread's first kPrefetch elements are loaded before the partials are
// summed, so their latency overlaps that reduction; elements and their
// order per thread are those of the plain grid-stride loop.
constexpr int kPrefetch = 8;
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mgs_step(T *w, const T *__restrict__ v, const T *next,
                                                     const double *__restrict__ part_in, int np,
                                                     double *__restrict__ part_out, double *__restrict__ h,
                                                     int64_t n) {
  const int64_t i0 = blockIdx.x * (int64_t)kBlock + threadIdx.x, stride = (int64_t)gridDim.x * kBlock;
  const bool self = next == w;
  T wv[kPrefetch], vv[kPrefetch], nv[kPrefetch];
#pragma unroll
  for (int k = 0; k < kPrefetch; k++) {
    const int64_t i = i0 + k * stride;
    wv[k] = vv[k] = nv[k] = T(0);
    if (i < n) {
      wv[k] = w[i];
      vv[k] = v[i];
      if (!self) nv[k] = next[i];
    }
  }
  const double hv = sum_partials(part_in, np);
  if (blockIdx.x == 0 && threadIdx.x == 0) h[0] = hv;
  const T at = (T)(-hv);
  double s = 0;
#pragma unroll
  for (int k = 0; k < kPrefetch; k++) {
    const int64_t i = i0 + k * stride;
    if (i < n) {
      T wi = wv[k];
      wi += at * vv[k];
      w[i] = wi;
      s += (double)wi * (double)(self ? wi : nv[k]);
    }
  }
  for (int64_t i = i0 + kPrefetch * stride; i < n; i += stride) {
    T wi = w[i];
    wi += at * v[i];
    w[i] = wi;
    s += (double)wi * (double)(self ? wi : next[i]);
  }
  s = block_sum<T>(s);
  if (threadIdx.x == 0) part_out[blockIdx.x] = s;
}
// *h = ||w|| from the partials of (w, w), y = w / ||w|| (prefetch as above)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_norm_scale(const T *__restrict__ w, const double *__restrict__ part,
                                                       int np, double *__restrict__ h, T *__restrict__ y, int64_t n) {
  const int64_t i0 = blockIdx.x * (int64_t)kBlock + threadIdx.x, stride = (int64_t)gridDim.x * kBlock;
  T wv[kPrefetch];
#pragma unroll
  for (int k = 0; k < kPrefetch; k++) {
    const int64_t i = i0 + k * stride;
    wv[k] = i < n ? w[i] : T(0);
  }
  const double nv = sqrt(sum_partials(part, np));
  if (blockIdx.x == 0 && threadIdx.x == 0) h[0] = nv;
  const T sc = (T)(1.0 / nv);
#pragma unroll
  for (int k = 0; k < kPrefetch; k++) {
    const int64_t i = i0 + k * stride;
    if (i < n) y[i] = wv[k] * sc;
  }
  for (int64_t i = i0 + kPrefetch * stride; i < n; i += stride) y[i] = w[i] * sc;
}
// All steps of an Arnoldi vector of a small space in one workgroup, which keeps
// w and the next basis vector in registers.  Bound by the chain of the
// reductions; a launch per step costs 4 us whatever the size (n = 4913, FP64, 3 basis vectors on
// average: 8.3 us, by launches 23 us; a second pass over V for more elements than
// fit the registers would take as long as the launches).
constexpr int kMgsWg = 1024, kMgsWgMax = 8 * kMgsWg;
__device__ __forceinline__ double mgs_total(double s, double *sh) {
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  s = 0;
#pragma unroll
  for (int i = 0; i < kMgsWg / 64; i++) s += sh[i];
  return s;
}
template <typename T, int PER>
__global__ __launch_bounds__(kMgsWg) void k_mgs_wg(T *__restrict__ w, const T *__restrict__ V, int64_t n, int k1,
                                                   double *__restrict__ h, T *__restrict__ y) {
  __shared__ double sh[2][kMgsWg / 64];  // (two: the one of the step before may still be read)
  T wv[PER], v[PER], next[PER];
  auto load = [&](const T *q, T *r) {
#pragma unroll
    for (int i = 0; i < PER; i++) r[i] = threadIdx.x + i * kMgsWg < n ? q[threadIdx.x + i * kMgsWg] : T(0);
  };
  load(w, wv);
  load(V, v);
  for (int k = 0; k < k1; k++) {
    load(V + (k + 1 < k1 ? k + 1 : k) * n, next);
    double s = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) s += (double)wv[i] * (double)v[i];
    s = mgs_total(s, sh[k & 1]);
    if (threadIdx.x == 0) h[k] = s;
    const T at = (T)(-s);
#pragma unroll
    for (int i = 0; i < PER; i++) {
      wv[i] += at * v[i];
      v[i] = next[i];
    }
  }
  double s = 0;
#pragma unroll
  for (int i = 0; i < PER; i++) s += (double)wv[i] * (double)wv[i];
  s = sqrt(mgs_total(s, sh[k1 & 1]));
  if (threadIdx.x == 0) h[k1] = s;
  const T sc = (T)(1.0 / s);
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int64_t p = threadIdx.x + i * kMgsWg;
    if (p < n) {
      w[p] = wv[i];
      y[p] = wv[i] * sc;
    }
  }
}
template <typename T>
void mgs_arnoldi(T *w, const T *V, int64_t n, int k1, double *h, T *vnext, double *part, hipStream_t st) {
  if (n <= kMgsWgMax) {
    auto *k = n <= kMgsWg ? k_mgs_wg<T, 1> : k_mgs_wg<T, 8>;  // (levels have 729 nodes or less, or 4913)
    hipLaunchKernelGGL(k, dim3(1), dim3(kMgsWg), 0, st, w, V, n, k1, h, vnext);
    return;
  }
  int g = (int)((n + kBlock - 1) / kBlock);
  if (g > kRedBlocks) g = kRedBlocks;
  if (g < 1) g = 1;
  double *pa = part, *pb = part + kRedBlocks;
  hipLaunchKernelGGL(k_dot_partial<T>, dim3(g), dim3(kBlock), 0, st, w, V, pa, n);
  for (int k = 0; k < k1; k++) {
    const T *next = k + 1 < k1 ? V + (size_t)(k + 1) * n : w;
    hipLaunchKernelGGL(k_mgs_step<T>, dim3(g), dim3(kBlock), 0, st, w, V + (size_t)k * n, next, pa, g, pb, h + k, n);
    std::swap(pa, pb);
  }
  hipLaunchKernelGGL(k_norm_scale<T>, dim3(g), dim3(kBlock), 0, st, w, pa, g, h + k1, vnext, n);
}

template <typename T>
void boundary(const DevLayout &D, int mode, T *y, const T *x, const T *f, hipStream_t st) {
  const int g = (D.nboundary + kBlock - 1) / kBlock;
  switch (mode) {
    case 0: hipLaunchKernelGGL((k_boundary<T, 0>), dim3(g), dim3(kBlock), 0, st, D.boundary, D.nboundary, y, x, f); break;
    case 1: hipLaunchKernelGGL((k_boundary<T, 1>), dim3(g), dim3(kBlock), 0, st, D.boundary, D.nboundary, y, x, f); break;
    case 2: hipLaunchKernelGGL((k_boundary<T, 2>), dim3(g), dim3(kBlock), 0, st, D.boundary, D.nboundary, y, x, f); break;
    default: hipLaunchKernelGGL((k_boundary<T, 3>), dim3(g), dim3(kBlock), 0, st, D.boundary, D.nboundary, y, x, f); break;
  }
}
template <typename T>
void prolongate(const DevLayout &C, const DevLayout &F, const T *xc, T *xf, hipStream_t st) {
  if (F.N >= (int64_t(1) << 31)) throw std::runtime_error("prolongate: lattice too large for 32-bit indices");
  if (F.order == 2)
    hipLaunchKernelGGL((k_prolong<T, 2, 0>), dim3(grid_for(F.N)), dim3(kBlock), 0, st, xc, xf, C.M, F.M, 1.0);
  else
    hipLaunchKernelGGL((k_prolong<T, 1, 0>), dim3(grid_for(F.N)), dim3(kBlock), 0, st, xc, xf, C.M, F.M, 1.0);
}
template <typename T>
void prolongate_add(const DevLayout &C, const DevLayout &F, const T *xc, T *xf, double damp, hipStream_t st) {
  if (F.N >= (int64_t(1) << 31)) throw std::runtime_error("prolongate: lattice too large for 32-bit indices");
  if (F.order == 2)
    hipLaunchKernelGGL((k_prolong<T, 2, 1>), dim3(grid_for(F.N)), dim3(kBlock), 0, st, xc, xf, C.M, F.M, damp);
  else
    hipLaunchKernelGGL((k_prolong<T, 1, 1>), dim3(grid_for(F.N)), dim3(kBlock), 0, st, xc, xf, C.M, F.M, damp);
}
template <typename T>
void restrict_(const DevLayout &C, const DevLayout &F, T *rc, const T *rf, hipStream_t st, T *xc) {
  if (F.N >= (int64_t(1) << 31)) throw std::runtime_error("restrict: lattice too large for 32-bit indices");
  if (F.order == 2)
    hipLaunchKernelGGL((k_restrict<T, 2>), dim3(grid_for(C.N)), dim3(kBlock), 0, st, rc, rf, C.M, F.M, xc);
  else
    hipLaunchKernelGGL((k_restrict<T, 1>), dim3(grid_for(C.N)), dim3(kBlock), 0, st, rc, rf, C.M, F.M, xc);
}
template <typename T>
void gemv_coarse(int nI, int N, const double *W, const int *iidx, const T *x, T *y, hipStream_t st) {
  hipLaunchKernelGGL(k_gemv_coarse<T>, dim3((unsigned)nI), dim3(64), 0, st, N, W, iidx, x, y);
}
// (k_gj_panel has a thread per row)
static bool gj_by_panels(int nI) { return nI <= kGjRows; }
int64_t coarse_inverse_scratch(int nI, int N) {
  const int64_t m = (int64_t)nI * (nI + (int64_t)N);
  return gj_by_panels(nI) ? 2 * m + (int64_t)nI * (kGjPanel + 1) : m;
}
void coarse_inverse_dense(const DevLayout &D, const double *val, const int *iidx, const int *cidx, int nI, double *aug,
                          int *piv, double *W, hipStream_t st) {
  if (nI > 8192) throw std::invalid_argument("coarse inverse: too many interior nodes");
  const int N = (int)D.N;
  const int64_t ld = nI + (int64_t)N;
  fill<double>(aug, 0.0, nI * ld, st);
  const dim3 ga((unsigned)((nI + 63) / 64));
  if (D.order == 2) hipLaunchKernelGGL(k_values_to_aug<2>, ga, dim3(64), 0, st, D.M, iidx, cidx, nI, val, aug, ld);
  else hipLaunchKernelGGL(k_values_to_aug<1>, ga, dim3(64), 0, st, D.M, iidx, cidx, nI, val, aug, ld);
  const dim3 gf((unsigned)(((int64_t)nI * N + 255) / 256));
  if (gj_by_panels(nI)) {
    // scratch behind the matrix: its other copy, the factors, the pivots
    double *other = aug + (int64_t)nI * ld, *T = other + (int64_t)nI * ld, *pval = T + (int64_t)nI * kGjPanel;
    for (int c = 0; c < nI; c += kGjPanel) {
      const int nc = std::min(kGjPanel, nI - c), c1 = c + nc;
      hipLaunchKernelGGL(k_gj_panel, dim3(1), dim3((unsigned)(nI + 63) / 64 * 64), 0, st, aug, nI, ld, c, nc, piv, pval, T);
      hipLaunchKernelGGL(k_gj_update, dim3((unsigned)((ld - c1 + 63) / 64), (unsigned)((nI + 15) / 16)), dim3(256), 0, st,
                         aug, other, nI, ld, c, c1, piv, T);
      std::swap(aug, other);
    }
    hipLaunchKernelGGL(k_gj_finish, gf, dim3(256), 0, st, aug, nI, N, ld, piv, (const double *)pval, W);
    return;
  }
  const unsigned g = (unsigned)((nI + 3) / 4);
  for (int c = 0; c < nI; c++) hipLaunchKernelGGL(k_gj_step, dim3(g), dim3(256), 0, st, aug, nI, ld, c, piv);
  hipLaunchKernelGGL(k_gj_finish, gf, dim3(256), 0, st, aug, nI, N, ld, piv, (const double *)nullptr, W);
}
template <typename T, typename U>
void gather(T *out, const U *in, const int *map, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL((k_gather<T, U>), dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, out, in,
                     map, n);
}
template <typename T>
void csr_spmv(int n, const int *rp, const int *kc, const T *val, const T *x, T *y, hipStream_t st) {
  const int g = (int)(((int64_t)n * 16 + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_csr_spmv<T>, dim3(g), dim3(kBlock), 0, st, n, rp, kc, val, x, y, (const T *)nullptr);
}
template <typename T>
void csr_defect(int n, const int *rp, const int *kc, const T *val, const T *x, const T *b, T *r, hipStream_t st) {
  const int g = (int)(((int64_t)n * 16 + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_csr_spmv<T>, dim3(g), dim3(kBlock), 0, st, n, rp, kc, val, x, r, b);
}
void csr_to_values(const DevLayout &D, const int *rowptr, const int *kcol, const int *dof2lat, int64_t active,
                   const double *in, double *val, hipStream_t st) {
  if (active == 0) return;
  const dim3 g((unsigned)((active + kBlock - 1) / kBlock));
  if (D.order == 2)
    hipLaunchKernelGGL(k_csr_to_values<2>, g, dim3(kBlock), 0, st, rowptr, kcol, dof2lat, active, D.M, in, val);
  else
    hipLaunchKernelGGL(k_csr_to_values<1>, g, dim3(kBlock), 0, st, rowptr, kcol, dof2lat, active, D.M, in, val);
}
template <typename T>
void values_to_csr(const DevLayout &D, const int *rowptr, const int *kcol, const int *dof2lat, int64_t active,
                   const T *val, double *out, hipStream_t st) {
  const dim3 g((unsigned)((D.N + kBlock - 1) / kBlock));
  if (D.order == 2)
    hipLaunchKernelGGL((k_values_to_csr<T, 2>), g, dim3(kBlock), 0, st, rowptr, kcol, dof2lat, D.N, active, D.M, val, out);
  else
    hipLaunchKernelGGL((k_values_to_csr<T, 1>), g, dim3(kBlock), 0, st, rowptr, kcol, dof2lat, D.N, active, D.M, val, out);
}

// ---- Q2 one-matrix forms: local matrices per cell, then a row gather.
// With Phi_q the 4 x 27 table of (phi, dphi/dxi, dphi/deta, dphi/dzeta) at
// point q, every form above is K = sum_q Phi_q^T D_q Phi_q (rows: test
// functions a, columns: trial functions b) with, for the convection-diffusion
// forms (g = 2/h folds the reference derivatives into D, s = delta):
//   D[0][0] = w c          D[0][d] = w g b_d
//   D[e][0] = w g c s b_e  D[e][d] = w g^2 (eps [e == d] + s b_e b_d)
// and the right-hand side f_a = sum_q r_q . Phi_q[:, a] with r = w f (1, g s b);
// the mass form has D[0][0] = w and r = w f (1, g s b).
//
// The rule (NP points per axis) and the basis are tensor products, so the sum
// is taken axis by axis: x, y, z one after the other, a pair of 1D basis
// functions (of a and of b) at a time.  After the x sum the rows and columns
// without a y or z derivative (phi and dphi/dxi) have the same y and z factors
// and are one class (N), so 3 x 3 classes (N, Y, Z) remain of 4 x 4, after the
// y sum 2 x 2.  For 64 points a cell takes 33 thousand products instead of the
// 187 thousand of the plain sum (262 thousand on padded 16 x 16 x 4 matrix
// instructions).  A workgroup takes kCells cells; a thread holds, of one cell,
//   x: a line (y, z) of points and one basis function of a,
//   y: a pair of x functions and one z,
//   z: a pair of x and a pair of y functions,
// and the sums between the axes go through LDS.  64^3 cells, 64 points: 3.75 ms by
// the matrix instructions, 1.05 ms now (the cell buffer is 1.6 GB); 16^3 cells and
// the levels below them, 27 points: 410 -> 64 us with the gather.
constexpr int kKcRow = 28;  // doubles per local row in the cell buffer: 27 entries + rhs
constexpr int kCells = 4, kCellThreads = 192;
template <int NP, bool INL>
__global__ __launch_bounds__(kCellThreads) void k_cell_sum(int n, int form, const double *__restrict__ prm,
                                                           const double *__restrict__ qref,
                                                           const double *__restrict__ qp, double *__restrict__ kc) {
  constexpr int YZ = NP * NP, NQ = NP * YZ, XS = 81 * YZ, YS = 4 * 81 * NP, TS = XS > YS ? XS : YS;
  static_assert(kCells * 3 * YZ <= kCellThreads && kCells * 12 * NP <= kCellThreads, "a thread per task");
  __shared__ double tx[kCells * TS];  // x sums [class][pair][z][y], then y sums [class][pair][pair][z]
  __shared__ double rx[kCells * 9 * YZ], ry[kCells * 18 * NP];  // those of the right-hand side
  const int tid = threadIdx.x;
  const int64_t ncells = (int64_t)n * n * n, cell0 = (int64_t)blockIdx.x * kCells;
  // 1D basis functions and derivatives at the points
  double f[3][NP], d[3][NP];
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const double t = qref[4 * i];
    f[0][i] = uniform(0.5 * t * (t - 1));
    f[1][i] = uniform(1 - t * t);
    f[2][i] = uniform(0.5 * t * (t + 1));
    d[0][i] = uniform(t - 0.5);
    d[1][i] = uniform(-2 * t);
    d[2][i] = uniform(t + 0.5);
  }
  if (tid < kCells * 3 * YZ) {
    const int c = tid / (3 * YZ), ax = (tid / YZ) % 3, yz = tid % YZ;
    // (a cell past the last one repeats it and is not stored)
    const int64_t cell = cell0 + c < ncells ? cell0 + c : ncells - 1;
    const int cx = (int)(cell % n), cy = (int)((cell / n) % n), cz = (int)(cell / ((int64_t)n * n));
    const bool mass = form == PMX_FORM_MASS || form == PMX_FORM_MASS_SUPG;
    const double g = 2.0 * n;
    double t[9][3], r[3] = {0, 0, 0};  // class (row, column), function of b
#pragma unroll
    for (int i = 0; i < 9; i++) t[i][0] = t[i][1] = t[i][2] = 0;
#pragma unroll
    for (int i = 0; i < NP; i++) {
      double Q[8];
      if (INL) {
        qp_coeffs<true>(prm, qref, n, cx, cy, cz, i + NP * yz, form, Q);
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) Q[e] = qp[(cell * NQ + i + NP * yz) * 8 + e];
      }
      const double w = Q[0], xa = ax == 0 ? f[0][i] : ax == 1 ? f[1][i] : f[2][i],
                   da = ax == 0 ? d[0][i] : ax == 1 ? d[1][i] : d[2][i];
      const double wgs = w * g * Q[7], s1 = wgs * Q[2], s2 = wgs * Q[3], s3 = wgs * Q[4];
      // D = s v^T + eps w g^2 on the diagonal of the derivatives, s = (w, s1, s2, s3)
      const double rn = w * xa + s1 * da, rY = s2 * xa, rZ = s3 * xa;
      r[0] += Q[6] * rn;
      r[1] += Q[6] * rY;
      r[2] += Q[6] * rZ;
      const double sn = mass ? w * xa : rn, sY = mass ? 0.0 : rY, sZ = mass ? 0.0 : rZ;
      const double v0 = mass ? 1.0 : Q[5], v1 = mass ? 0.0 : g * Q[2], v2 = mass ? 0.0 : g * Q[3],
                   v3 = mass ? 0.0 : g * Q[4], ee = mass ? 0.0 : w * g * g * Q[1];
      const double m[3][4] = {{sn * v0, sn * v1 + ee * da, sn * v2, sn * v3},
                              {sY * v0, sY * v1, sY * v2 + ee * xa, sY * v3},
                              {sZ * v0, sZ * v1, sZ * v2, sZ * v3 + ee * xa}};
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
          t[3 * k][b] = fma(m[k][0], f[b][i], fma(m[k][1], d[b][i], t[3 * k][b]));
          t[3 * k + 1][b] = fma(m[k][2], f[b][i], t[3 * k + 1][b]);
          t[3 * k + 2][b] = fma(m[k][3], f[b][i], t[3 * k + 2][b]);
        }
    }
#pragma unroll
    for (int k = 0; k < 9; k++)
#pragma unroll
      for (int b = 0; b < 3; b++) tx[c * TS + (k * 9 + 3 * ax + b) * YZ + yz] = t[k][b];
#pragma unroll
    for (int k = 0; k < 3; k++) rx[(c * 9 + 3 * k + ax) * YZ + yz] = r[k];
  }
  __syncthreads();
  {
    const int c = tid / (9 * NP), xp = (tid / NP) % 9, z = tid % NP;
    const bool matrix = tid < kCells * 9 * NP;
    double t[9][4];  // pair of y functions, class (row, column)
#pragma unroll
    for (int i = 0; i < 9; i++) t[i][0] = t[i][1] = t[i][2] = t[i][3] = 0;
    if (matrix) {
#pragma unroll
      for (int y = 0; y < NP; y++) {
        double v[9];
#pragma unroll
        for (int k = 0; k < 9; k++) v[k] = tx[c * TS + (k * 9 + xp) * YZ + z * NP + y];
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const double fa = f[a][y], da = d[a][y];
          const double nn = v[0] * fa + v[3] * da, ny = v[1] * fa + v[4] * da, nz = v[2] * fa + v[5] * da;
          const double zn = v[6] * fa, zy = v[7] * fa, zz = v[8] * fa;
#pragma unroll
          for (int b = 0; b < 3; b++) {
            double *o = t[3 * a + b];
            o[0] = fma(nn, f[b][y], fma(ny, d[b][y], o[0]));
            o[1] = fma(nz, f[b][y], o[1]);
            o[2] = fma(zn, f[b][y], fma(zy, d[b][y], o[2]));
            o[3] = fma(zz, f[b][y], o[3]);
          }
        }
      }
    } else if (tid < kCells * 12 * NP) {
      const int i = tid - kCells * 9 * NP, c = i / (3 * NP), ax = (i / NP) % 3, z = i % NP;
      double o[3][2] = {{0, 0}, {0, 0}, {0, 0}};
#pragma unroll
      for (int y = 0; y < NP; y++) {
        const double v0 = rx[(c * 9 + ax) * YZ + z * NP + y], v1 = rx[(c * 9 + 3 + ax) * YZ + z * NP + y],
                     v2 = rx[(c * 9 + 6 + ax) * YZ + z * NP + y];
#pragma unroll
        for (int a = 0; a < 3; a++) {
          o[a][0] = fma(v0, f[a][y], fma(v1, d[a][y], o[a][0]));
          o[a][1] = fma(v2, f[a][y], o[a][1]);
        }
      }
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int k = 0; k < 2; k++) ry[((c * 2 + k) * 9 + 3 * a + ax) * NP + z] = o[a][k];
    }
    __syncthreads();
    if (matrix) {
#pragma unroll
      for (int y = 0; y < 9; y++)
#pragma unroll
        for (int k = 0; k < 4; k++) tx[c * TS + ((k * 9 + xp) * 9 + y) * NP + z] = t[y][k];
    }
  }
  __syncthreads();
  for (int i = tid; i < kCells * 90; i += kCellThreads) {
    const int c = i / 90, j = i % 90;
    if (cell0 + c >= ncells) break;
    double *K = kc + (cell0 + c) * (27 * kKcRow);
    if (j < 81) {
      // (x, y) functions of a, of b
      const int a9 = j / 9, b9 = j % 9, xp = 3 * (a9 % 3) + b9 % 3, yp = 3 * (a9 / 3) + b9 / 3;
      double o[9];
#pragma unroll
      for (int k = 0; k < 9; k++) o[k] = 0;
#pragma unroll
      for (int z = 0; z < NP; z++) {
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = tx[c * TS + ((k * 9 + xp) * 9 + yp) * NP + z];
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const double nn = v[0] * f[a][z] + v[2] * d[a][z], nz = v[1] * f[a][z] + v[3] * d[a][z];
#pragma unroll
          for (int b = 0; b < 3; b++) o[3 * a + b] = fma(nn, f[b][z], fma(nz, d[b][z], o[3 * a + b]));
        }
      }
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) K[(a9 + 9 * a) * kKcRow + b9 + 9 * b] = o[3 * a + b];
    } else {
      const int a9 = j - 81;
      double o[3] = {0, 0, 0};
#pragma unroll
      for (int z = 0; z < NP; z++) {
        const double v0 = ry[((c * 2) * 9 + a9) * NP + z], v1 = ry[((c * 2 + 1) * 9 + a9) * NP + z];
#pragma unroll
        for (int a = 0; a < 3; a++) o[a] = fma(v0, f[a][z], fma(v1, d[a][z], o[a]));
      }
#pragma unroll
      for (int a = 0; a < 3; a++) K[(a9 + 9 * a) * kKcRow + 27] = o[a];
    }
  }
}
// Row gather from the cell buffer: the thread of active node p adds row a of
// each incident cell's local matrix into its row of values and sums the rhs column.
// The row's stencil slots are accumulated in registers over its incident
// cells (in the order (iz, iy, ix)) and every slot is stored once, after the
// last cell that touches it (a slot (dx, dy, dz) gets its last contribution
// from the cell on the positive side of each offset that is >= 0), so the
// values are written without being read and without a prior clear.  The local node of the row in cell (ix, iy, iz) and
// the slot of every cell entry are compile-time constants: along an axis
// with extent 2 (even lattice coordinate, a vertex plane) the node is local
// coordinate 2 - 2 i of cell i, along an axis with extent 1 local coordinate 1.
// A wavefront's 64 rows lie in consecutive cells of one x-line of cells (or,
// P < 64, of several lines 3 cells apart in y), so it fetches each incident
// cell's 64 local rows of 224 bytes together, 14 lanes per row, through LDS
// (rows padded to 29 doubles), the next cell's while it adds the current one.
// Bound by HBM: 64^3 Q2 reads the 1.6 GB cell buffer and writes 1.05 GB of
// values in 0.6 ms; a row per lane straight from memory, 14 loads that each
// touch 64 cache lines, took 0.77 - 1.1 ms.
constexpr int kKcPad = kKcRow + 1;
template <int EX, int EY, int EZ>
__device__ __forceinline__ void assemble_row_kc(double (*sh)[64 * kKcPad], bool ok, int px, int py, int pz, int lg, int M,
                                                int n, const double *__restrict__ kc, double *__restrict__ val,
                                                double *__restrict__ rhs) {
  constexpr int NCX = EX == 1 ? 1 : 2, NCY = EY == 1 ? 1 : 2, NCZ = EZ == 1 ? 1 : 2, NC = NCX * NCY * NCZ;
  constexpr int WX = 2 * EX + 1, WY = 2 * EY + 1, WZ = 2 * EZ + 1, NS = WX * WY * WZ;
  constexpr int PIECES = kKcRow / 2;
  const int lane = threadIdx.x;
  const int P = 1 << lg;
  // row r of the wavefront: local row a(cell) of the cell c0 + (r & (P-1)) + 3 n (r >> lg)
  const int x0 = __builtin_amdgcn_readfirstlane(px), y0 = __builtin_amdgcn_readfirstlane(py),
            z0 = __builtin_amdgcn_readfirstlane(pz);
  const int64_t last = (int64_t)n * n * n - 1;
  double2 part[PIECES];
  auto fetch = [&](int i) {
    const int ix = i % NCX, iy = (i / NCX) % NCY, iz = i / (NCX * NCY);
    const int ax = EX == 1 ? 1 : 2 - 2 * ix, ay = EY == 1 ? 1 : 2 - 2 * iy, az = EZ == 1 ? 1 : 2 - 2 * iz;
    const int a = ax + 3 * (ay + 3 * az);
    const int64_t c0 = ((x0 - 1) / 2 + ix) + (int64_t)n * (((y0 - 1) / 2 + iy) + (int64_t)n * ((z0 - 1) / 2 + iz));
#pragma unroll
    for (int e = 0; e < PIECES; e++) {
      const int id = lane + 64 * e, r = id / PIECES, q = id % PIECES;
      int64_t cell = c0 + (lg >= 6 ? r : (r & (P - 1)) + 3 * n * (r >> lg));
      cell = cell < last ? cell : last;  // rows past the lattice (not stored)
      part[e] = reinterpret_cast<const double2 *>(kc + (cell * 27 + a) * kKcRow)[q];
    }
  };
  const GroupOrder<2> go(y0, z0);
  double *v = val + line_values<2>(P, py, pz);
  const int m = (px - 1) >> 1;
  double frhs = 0;
  double acc[NS];
#pragma unroll
  for (int q = 0; q < NS; q++) acc[q] = 0.0;
  fetch(0);
#pragma unroll
  for (int i = 0; i < NC; i++) {
    double *buf = sh[i & 1];
#pragma unroll
    for (int e = 0; e < PIECES; e++) {
      const int id = lane + 64 * e, r = id / PIECES, q = id % PIECES;
      buf[r * kKcPad + 2 * q] = part[e].x;
      buf[r * kKcPad + 2 * q + 1] = part[e].y;
    }
    if (i + 1 < NC) fetch(i + 1);
    __syncthreads();  // one wavefront
    const int ix = i % NCX, iy = (i / NCX) % NCY, iz = i / (NCX * NCY);
    const int ax = EX == 1 ? 1 : 2 - 2 * ix, ay = EY == 1 ? 1 : 2 - 2 * iy, az = EZ == 1 ? 1 : 2 - 2 * iz;
    const double *row = buf + lane * kKcPad;
#pragma unroll
    for (int b = 0; b < 27; b++) {
      const int dx = b % 3 - ax, dy = (b / 3) % 3 - ay, dz = b / 9 - az;
      acc[(dx + EX) + WX * ((dy + EY) + WY * (dz + EZ))] += row[b];
    }
    frhs += row[27];
#pragma unroll
    for (int q = 0; q < NS; q++) {
      const int dx = q % WX - EX, dy = (q / WX) % WY - EY, dz = q / (WX * WY) - EZ;
      const int lx = (NCX == 2 && dx >= 0) ? 1 : 0, ly = (NCY == 2 && dy >= 0) ? 1 : 0,
                lz = (NCZ == 2 && dz >= 0) ? 1 : 0;
      if (lx == ix && ly == iy && lz == iz && ok)
        v[go.position(dy, dz) * (Lines<2>::VL * P) + Slots<double, 2>::at(P, m, EX == 1 ? dx + 1 : dx + 5)] = acc[q];
    }
  }
  if (ok) rhs[px + M * (py + M * pz)] = frhs;
}
__global__ __launch_bounds__(kRowsPerBlock) void k_assemble_kc(LineSet set, int lg, int M, int n,
                                                               const double *__restrict__ kc,
                                                               double *__restrict__ val, double *__restrict__ rhs) {
  static_assert(kRowsPerBlock == 64, "one wavefront");
  __shared__ double sh[2][64 * kKcPad];
  int px, py, pz;
  const RowBlock rb = row_block<2>(set, M, lg);
  const bool ok = unit_row<2>(rb, M, lg, threadIdx.x, &px, &py, &pz);
  const int code = unit_shape<2>(rb);
#define PMX_KROW(EX, EY, EZ) assemble_row_kc<EX, EY, EZ>(sh, ok, px, py, pz, lg, M, n, kc, val, rhs)
  switch (code) {
    case 111: PMX_KROW(1, 1, 1); break;
    case 211: PMX_KROW(2, 1, 1); break;
    case 121: PMX_KROW(1, 2, 1); break;
    case 221: PMX_KROW(2, 2, 1); break;
    case 112: PMX_KROW(1, 1, 2); break;
    case 212: PMX_KROW(2, 1, 2); break;
    case 122: PMX_KROW(1, 2, 2); break;
    default: PMX_KROW(2, 2, 2); break;
  }
#undef PMX_KROW
}

void assemble(const DevLayout &D, const double *prm_dev, int example, int form, const double *qref, int nq,
              const double *tab, double *qpbuf, double *kc, double *val, double *val2, double *rhs, hipStream_t st,
              bool qp_given, double *ftab, const uint8_t *corner) {
  const int64_t ncells = (int64_t)D.n * D.n * D.n;
  const int64_t ncq = ncells * nq;
  int units;
  const LineSet set = all_lines(D, &units);
  const dim3 gr(row_blocks(D, units));
  // with the per-cell frame codes (CELL_MEASURE 4) the coefficients go
  // through the qp records, which carry the cell's first-point size
  const bool inl = !qp_given && coeffs_inline(example) && !corner;
  if (!inl && !qp_given) {
    // (grid y = n^2 lines of cells: up to 255 cells per direction)
    const bool grf = example == PMX_EX_LOGNORMAL && !corner;
    if ((example == PMX_EX_CURL_FOURIER || grf) && ftab && (int64_t)D.n * D.n <= 65535) {
      const int nl = nq == 8 ? 4 : (nq == 27 ? 9 : 16);  // x-lines of points per cell
      if (nq != 8 && nq != 27 && nq != 64) throw std::logic_error("assemble: rule without phase tables");
      // complex entries
      const int64_t nt = (int64_t)(grf ? kGrfModes : kFourierModes) * 3 * D.n * rule_points_1d(nq);
      const dim3 gt((unsigned)((nt + kBlock - 1) / kBlock));
      const int per = grf ? rule_points_1d(nq) : nl;  // threads per cell
      const dim3 g((unsigned)((D.n * per + kBlock - 1) / kBlock), (unsigned)(D.n * D.n));
      if (grf) {
        hipLaunchKernelGGL(k_phase_tables<true>, gt, dim3(kBlock), 0, st, prm_dev, qref, nq, D.n, ftab);
        auto *k = nq == 8 ? k_qp_data_grf<8> : nq == 27 ? k_qp_data_grf<27> : k_qp_data_grf<64>;
        hipLaunchKernelGGL(k, g, dim3(kBlock), 0, st, prm_dev, qref, D.n, ftab, qpbuf);
      } else {
        hipLaunchKernelGGL(k_phase_tables<false>, gt, dim3(kBlock), 0, st, prm_dev, qref, nq, D.n, ftab);
        auto *k = nq == 8 ? k_qp_data_fourier<8> : nq == 27 ? k_qp_data_fourier<27> : k_qp_data_fourier<64>;
        hipLaunchKernelGGL(k, g, dim3(kBlock), 0, st, prm_dev, qref, D.n, ftab, qpbuf, corner);
      }
    } else {
      hipLaunchKernelGGL(k_qp_data, dim3((unsigned)((ncq + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, prm_dev,
                         qref, nq, D.n, qpbuf, corner);
    }
  }
  // the per-row evaluation with inline coefficients reads the stabilisation
  // parameters from a per-point buffer (the start of qpbuf), filled once
  const double *qsrc = qpbuf;
  if (inl) {
    qsrc = nullptr;
    if (form_has_delta(form) && !(kc && D.order == 2 && !val2 && form != PMX_FORM_RHS_SUPG)) {
      if ((int64_t)D.n * nq > 65535) throw std::invalid_argument("assemble: level too large for k_qp_delta");
      hipLaunchKernelGGL(k_qp_delta, dim3((unsigned)((D.n * D.n + kBlock - 1) / kBlock), (unsigned)(D.n * nq)),
                         dim3(kBlock), 0, st, prm_dev, qref, D.n, qpbuf);
      qsrc = qpbuf;
    }
  }
  if (form == PMX_FORM_RHS || form == PMX_FORM_RHS_SUPG) {
    // right-hand-side forms (no local matrices): the matrices are left as they are
#define PMX_RHS(O, IN)                                                                                     \
  hipLaunchKernelGGL((k_assemble<O, IN, true>), gr, dim3(kRowsPerBlock), 0, st, set, D.lg, D.M, D.n, nq, prm_dev, qref, qsrc, tab, nullptr, nullptr, rhs)
    if (D.order == 1) {
      if (inl) PMX_RHS(1, true);
      else PMX_RHS(1, false);
    } else {
      if (inl) PMX_RHS(2, true);
      else PMX_RHS(2, false);
    }
#undef PMX_RHS
    hipLaunchKernelGGL(k_boundary_rhs, dim3((D.nboundary + kBlock - 1) / kBlock), dim3(kBlock), 0, st, D.boundary,
                       D.nboundary, D.M, prm_dev, rhs);
    return;
  }
  if (kc && D.order == 2 && !val2) {
    // local matrices, then the row gather from the cell buffer
#define PMX_CELL(NP, IN)                                                                                               \
  hipLaunchKernelGGL((k_cell_sum<NP, IN>), dim3((unsigned)((ncells + kCells - 1) / kCells)), dim3(kCellThreads), 0, st, \
                     D.n, form, prm_dev, qref, qpbuf, kc)
    if (nq == 27) {
      if (inl) PMX_CELL(3, true);
      else PMX_CELL(3, false);
    } else if (nq == 64) {
      if (inl) PMX_CELL(4, true);
      else PMX_CELL(4, false);
    } else throw std::logic_error("assemble: no Q2 kernel for the rule");
#undef PMX_CELL
    hipLaunchKernelGGL(k_assemble_kc, gr, dim3(kRowsPerBlock), 0, st, set, D.lg, D.M, D.n, kc, val, rhs);
    hipLaunchKernelGGL(k_boundary_rhs, dim3((D.nboundary + kBlock - 1) / kBlock), dim3(kBlock), 0, st, D.boundary,
                       D.nboundary, D.M, prm_dev, rhs);
    return;
  }
  if (D.order == 1) {
    // (every slot is stored; those of boundary nodes are never written and keep
    // the zeros of the allocation)
#define PMX_ASM3(NP, TW, SRC)                                                                                      \
  hipLaunchKernelGGL((k_assemble_q1<NP, TW, SRC>), gr, dim3(8 * kRowsPerBlock), 0, st, set, D.lg, D.M, D.n, prm_dev, \
                     qref, qsrc, val, val2, rhs)
#define PMX_ASM(NP, TW)                                                                                            \
  do {                                                                                                             \
    if (!inl) PMX_ASM3(NP, TW, kRecords);                                                                          \
    else if (example == PMX_EX_ROTATING) PMX_ASM3(NP, TW, kRotating);                                              \
    else PMX_ASM3(NP, TW, kInline);                                                                                \
  } while (0)
    if (nq != 8 && nq != 27) throw std::logic_error("assemble: no Q1 kernel for the rule");
    if (nq == 8 && val2) PMX_ASM(2, true);
    else if (nq == 8) PMX_ASM(2, false);
    else if (val2) PMX_ASM(3, true);
    else PMX_ASM(3, false);
#undef PMX_ASM
#undef PMX_ASM3
  } else {
    // Q2, two matrices: a row per thread adds every cell's contribution into the
    // cleared values
    if (!val2) throw std::logic_error("assemble: Q2 without a cell buffer");
    check(hipMemsetAsync(val, 0, sizeof(double) * D.nvals, st), "memset val");
    check(hipMemsetAsync(val2, 0, sizeof(double) * D.nvals, st), "memset val2");
#define PMX_ASM(IN)                                                                                             \
  hipLaunchKernelGGL((k_assemble<2, IN, false>), gr, dim3(kRowsPerBlock), 0, st, set, D.lg, D.M, D.n, nq, prm_dev, \
                     qref, qsrc, tab, val, val2, rhs)
    if (inl) PMX_ASM(true);
    else PMX_ASM(false);
#undef PMX_ASM
  }
  hipLaunchKernelGGL(k_boundary_rhs, dim3((D.nboundary + kBlock - 1) / kBlock), dim3(kBlock), 0, st, D.boundary,
                     D.nboundary, D.M, prm_dev, rhs);
}

// ============================================================ error norms
// ||u - u_h||_L2 and |u - u_h|_H1 of a lattice FE function against the
// example's exact solution (TFEFunction3D::GetErrors with L2H1Errors,
// FEFunction3D.C:83-300, MainUtilities.C:1649): one thread per cell gathers
// its (order + 1)^3 nodal values, evaluates u_h and grad u_h at the rule's
// points from the reference tables (brick of side h: d/dx = (2/h) d/dxi,
// |detJ| = h^3/8) and adds w |detJ| (u - u_h)^2 and the gradient term;
// fixed-order block partials, then k_reduce_errors.
template <int ORDER>
__global__ __launch_bounds__(kBlock) void k_errors(const double *__restrict__ prm, int n, int M,
                                                   const double *__restrict__ qref, const double *__restrict__ tab,
                                                   int nq, const double *__restrict__ u,
                                                   double *__restrict__ part) {
  constexpr int K = ORDER + 1, NB = K * K * K;
  const int64_t ncells = (int64_t)n * n * n;
  const double h = 1.0 / n, adet = h * h * h / 8.0, g = 2.0 / h;
  double e0 = 0, e1 = 0;
  for (int64_t c = blockIdx.x * (int64_t)kBlock + threadIdx.x; c < ncells; c += (int64_t)gridDim.x * kBlock) {
    const int ci = (int)(c % n), cj = (int)((c / n) % n), ck = (int)(c / ((int64_t)n * n));
    double uc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int a = b % K, bb = (b / K) % K, cc = b / (K * K);
      uc[b] = u[(ORDER * ci + a) + (int64_t)M * ((ORDER * cj + bb) + (int64_t)M * (ORDER * ck + cc))];
    }
    for (int q = 0; q < nq; q++) {
      const double *r = qref + 4 * q;
      double uh[4] = {0, 0, 0, 0};
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const double *t = tab + ((int64_t)q * NB + b) * 4;
        uh[0] += uc[b] * t[0];
        uh[1] += uc[b] * t[1];
        uh[2] += uc[b] * t[2];
        uh[3] += uc[b] * t[3];
      }
      double ex[4];
      example_exact_grad(prm, (ci + 0.5 * (r[0] + 1.0)) * h, (cj + 0.5 * (r[1] + 1.0)) * h,
                         (ck + 0.5 * (r[2] + 1.0)) * h, ex);
      const double w = r[3] * adet;
      const double d0 = uh[0] - ex[0], d1 = g * uh[1] - ex[1], d2 = g * uh[2] - ex[2], d3 = g * uh[3] - ex[3];
      e0 += w * d0 * d0;
      e1 += w * (d1 * d1 + d2 * d2 + d3 * d3);
    }
  }
  e0 = block_sum<double>(e0);
  e1 = block_sum<double>(e1);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = e0;
    part[kRedBlocks + blockIdx.x] = e1;
  }
}
__global__ __launch_bounds__(kBlock) void k_reduce_errors(const double *__restrict__ part, int np,
                                                          double *__restrict__ out) {
  double s = 0, t = 0;
  for (int i = threadIdx.x; i < np; i += kBlock) {
    s += part[i];
    t += part[kRedBlocks + i];
  }
  s = block_sum<double>(s);
  t = block_sum<double>(t);
  if (threadIdx.x == 0) {
    out[0] = sqrt(s);
    out[1] = sqrt(t);
  }
}
void fe_errors(const DevLayout &D, const double *prm_dev, const double *qref, const double *tab, int nq,
               const double *u, double *part, double *out, hipStream_t st) {
  const int64_t ncells = (int64_t)D.n * D.n * D.n;
  const int g = (int)std::max<int64_t>(1, std::min<int64_t>((ncells + kBlock - 1) / kBlock, kRedBlocks));
  if (D.order == 2)
    hipLaunchKernelGGL(k_errors<2>, dim3(g), dim3(kBlock), 0, st, prm_dev, D.n, D.M, qref, tab, nq, u, part);
  else
    hipLaunchKernelGGL(k_errors<1>, dim3(g), dim3(kBlock), 0, st, prm_dev, D.n, D.M, qref, tab, nq, u, part);
  hipLaunchKernelGGL(k_reduce_errors, dim3(1), dim3(kBlock), 0, st, part, g, out);
}

// ============================================================ time stepping
// nodal interpolation of the example's exact (initial) function on the lattice
// (TFEFunction3D::Interpolate for Lagrange nodes)
__global__ void k_interpolate(const double *__restrict__ prm, int M, double *__restrict__ x) {
  const int64_t N = (int64_t)M * M * M;
  const double h = 1.0 / (M - 1);
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
    const int a = (int)(i % M), b = (int)((i / M) % M), c = (int)(i / ((int64_t)M * M));
    x[i] = example_exact(prm, a * h, b * h, c * h);
  }
}
// right-hand side of TSystemTCD3D::AssembleSystMat (SystemTCD3D.C:255-283):
// active rows B = t3 oldrhs + t4 rhs + (M (+ K) - t2 A) oldsol, Dirichlet rows
// B = rhs (k_old = K oldsol of the SUPG form, SystemTCD2D.C:294-297, or nullptr)
__global__ void k_tcd_rhs(int M, const double *__restrict__ oldrhs, const double *__restrict__ rhs,
                          const double *__restrict__ m_old, const double *__restrict__ a_old,
                          const double *__restrict__ k_old, double t3, double t4, double t2,
                          double *__restrict__ B) {
  const int64_t N = (int64_t)M * M * M;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
    const int a = (int)(i % M), b = (int)((i / M) % M), c = (int)(i / ((int64_t)M * M));
    const bool interior = a > 0 && b > 0 && c > 0 && a < M - 1 && b < M - 1 && c < M - 1;
    const double mk = k_old ? m_old[i] + k_old[i] : m_old[i];
    B[i] = interior ? (t3 * oldrhs[i] + t4 * rhs[i]) + (mk - t2 * a_old[i]) : rhs[i];
  }
}
void interpolate(const DevLayout &D, const double *prm_dev, double *x, hipStream_t st) {
  hipLaunchKernelGGL(k_interpolate, dim3(grid_for(D.N)), dim3(kBlock), 0, st, prm_dev, D.M, x);
}
void tcd_rhs(const DevLayout &D, const double *oldrhs, const double *rhs, const double *m_old, const double *a_old,
             const double *k_old, double t3, double t4, double t2, double *B, hipStream_t st) {
  hipLaunchKernelGGL(k_tcd_rhs, dim3(grid_for(D.N)), dim3(kBlock), 0, st, D.M, oldrhs, rhs, m_old, a_old, k_old,
                     t3, t4, t2, B);
}

void givens(double *H, double *cs, double *sn, double *s, int i, int ld, double *res, hipStream_t st) {
  hipLaunchKernelGGL(k_givens, dim3(1), dim3(64), 0, st, H, cs, sn, s, i, ld, res);
}
void backsolve(const double *H, const double *s, double *y, int k, int ld, hipStream_t st) {
  hipLaunchKernelGGL(k_backsolve, dim3(1), dim3(64), 0, st, H, s, y, k, ld);
}
template <typename T, typename X>
void multi_axpy(X *x, const T *z, const double *y, int k1, int64_t n, int64_t stride, hipStream_t st) {
  hipLaunchKernelGGL((k_multi_axpy<T, X>), dim3(grid_for(n)), dim3(kBlock), 0, st, x, z, y, k1, n, stride);
}
void set_scalar(double *dst, const double *src, double scale, hipStream_t st) {
  hipLaunchKernelGGL(k_set_scalar, dim3(1), dim3(64), 0, st, dst, src, scale);
}

// explicit instantiations
#define PMX_INST(T)                                                                                         \
  template void fill<T>(T *, T, int64_t, hipStream_t);                                                      \
  template void copy<T>(T *, const T *, int64_t, hipStream_t);                                              \
  template void copy_surface<T>(const DevLayout &, T *, const T *, T *, hipStream_t);                       \
  template void axpy<T>(T *, const T *, const double *, double, double, int64_t, hipStream_t);              \
  template void scale_inv<T>(T *, const T *, const double *, int64_t, hipStream_t);                         \
  template void dot<T>(const T *, const T *, int64_t, double *, double *, int, hipStream_t);                \
  template void mgs_arnoldi<T>(T *, const T *, int64_t, int, double *, T *, double *, hipStream_t);         \
  template void axpy_diff<T>(T *, const T *, const T *, int64_t, hipStream_t);                              \
  template void step_length_update<T>(T *, const T *, const double *, double, int64_t, hipStream_t);        \
  template void boundary<T>(const DevLayout &, int, T *, const T *, const T *, hipStream_t);                \
  template void prolongate<T>(const DevLayout &, const DevLayout &, const T *, T *, hipStream_t);           \
  template void prolongate_add<T>(const DevLayout &, const DevLayout &, const T *, T *, double, hipStream_t); \
  template void restrict_<T>(const DevLayout &, const DevLayout &, T *, const T *, hipStream_t, T *);       \
  template void start_zero<T>(T *, T *, const T *, int *, int64_t, hipStream_t);                            \
  template void start_boundary<T>(const DevLayout &, T *, const T *, int *, hipStream_t);                    \
  template void gemv_coarse<T>(int, int, const double *, const int *, const T *, T *, hipStream_t);         \
  template void csr_spmv<T>(int, const int *, const int *, const T *, const T *, T *, hipStream_t);         \
  template void csr_defect<T>(int, const int *, const int *, const T *, const T *, const T *, T *, hipStream_t); \
  template void values_to_csr<T>(const DevLayout &, const int *, const int *, const int *, int64_t, const T *, \
                              double *, hipStream_t);
PMX_INST(double)
PMX_INST(float)
template void values_to_csr<_Float16>(const DevLayout &, const int *, const int *, const int *, int64_t,
                                   const _Float16 *, double *, hipStream_t);
template void fill<uint16_t>(uint16_t *, uint16_t, int64_t, hipStream_t);
template void fill<int>(int *, int, int64_t, hipStream_t);
template void convert<float, double>(float *, const double *, int64_t, hipStream_t);
template void add_convert<double, float>(double *, const float *, int64_t, hipStream_t);
template void gather<double, double>(double *, const double *, const int *, int64_t, hipStream_t);
template void gather<float, double>(float *, const double *, const int *, int64_t, hipStream_t);
template void gather<double, float>(double *, const float *, const int *, int64_t, hipStream_t);
template void multi_axpy<double, double>(double *, const double *, const double *, int, int64_t, int64_t, hipStream_t);
template void multi_axpy<float, float>(float *, const float *, const double *, int, int64_t, int64_t, hipStream_t);

}  // namespace pmx
