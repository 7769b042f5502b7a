// pmx_ops.hpp -- stream-ordered launchers of the libpmx kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "pmx_internal.hpp"

namespace pmx {

// device mirror of a Layout
struct DevLayout {
  int order = 1, n = 0, M = 0;
  int lg = 0;  // log2 of the row pairs per line, (M - 1) / 2
  int64_t N = 0, nvals = 0, nactive = 0;
  int nboundary = 0;
  int *boundary = nullptr;
  int64_t max_colour_rows = 0;    // rows of the largest colour
  // the row pairs of each line group (M <= 33; k_pair_table)
  const int2 *pairs = nullptr;
  int pair_tiles = 0;
  int ncolours = 0;
};

void check(hipError_t e, const char *what);

// the numbering of build_numbering on the device (pmx_setup.hip): lat2dof,
// dof2lat (N each), GlobalNumbers (cells x local DOFs, optional) and the
// per-cell frame codes (n^3), all device arrays; synchronises the stream
void device_numbering(const Layout &L, int *lat2dof, int *dof2lat, int *gn, uint8_t *corner, hipStream_t st);
// the CSR structure of build_csr on the device (pmx_setup.hip): rowptr
// (N + 1) and kcol (csr_nnz(L)) from the device numbering; synchronises st
void device_csr(const Layout &L, const int *lat2dof, const int *dof2lat, int *rowptr, int *kcol, hipStream_t st);
int64_t csr_nnz(const Layout &L);

// event pairs of timed dispatches (see set_dispatch_timer)
struct DispatchTimer {
  std::vector<hipEvent_t> ev;
  int used = 0;
  double total_ms() const;  // sum of the dispatch durations (synchronise first)
  DispatchTimer() = default;
  DispatchTimer(const DispatchTimer &) = delete;
  DispatchTimer &operator=(const DispatchTimer &) = delete;
  ~DispatchTimer();
};
// while installed (non-null), the launched row kernels record each dispatch
// between two events of the timer; nullptr uninstalls
void set_dispatch_timer(DispatchTimer *t);

// calibration of the dispatch measurements (both honour the dispatch timer):
// a dispatch that does nothing with the workgroups of a line group's launch,
// and a plain streaming read of `bytes` bytes at p (16-byte aligned; sink: one
// float, written never in practice)
void empty_dispatch(const DevLayout &D, int group, hipStream_t st);
void stream_read(const void *p, int64_t bytes, float *sink, hipStream_t st);

template <typename T> void fill(T *x, T v, int64_t n, hipStream_t st);
template <typename T> void copy(T *y, const T *x, int64_t n, hipStream_t st);
// z = x, and y = x on the Dirichlet nodes
template <typename T> void copy_surface(const DevLayout &D, T *z, const T *x, T *y, hipStream_t st);
template <typename T>
void axpy(T *y, const T *x, const double *alpha_dev, double sgn, double ac, int64_t n, hipStream_t st);
template <typename T, typename U> void convert(T *y, const U *x, int64_t n, hipStream_t st);
template <typename T, typename U> void add_convert(T *y, const U *x, int64_t n, hipStream_t st);
template <typename T> void scale_inv(T *y, const T *x, const double *nrm, int64_t n, hipStream_t st);
template <typename T>
void dot(const T *x, const T *y, int64_t n, double *part, double *out, int do_sqrt, hipStream_t st);
// the Dirichlet rows r = f - x of a defect whose other rows are in r, and
// out = ||r||, with one partial sum per kDotChunk elements in part
// (ceil(N / kDotChunk) doubles), summed in a fixed order
constexpr int kDotChunk = 2048;
void defect_norm(const DevLayout &D, double *r, const double *x, const double *f, double *part, double *out,
                 hipStream_t st);
// e = u - uold
template <typename T> void axpy_diff(T *e, const T *u, const T *uold, int64_t n, hipStream_t st);
// TMGLevel3D::StepLengthControl's update: omega = num_nom[0] / num_nom[1]
// (param0 when num_nom[1] <= 0 or |omega| < 0.1), u = uold + omega (u - uold)
template <typename T>
void step_length_update(T *u, const T *uold, const double *num_nom, double param0, int64_t n, hipStream_t st);
// modified Gram-Schmidt of w against the k1 vectors V[0..k1) (stride n) and
// normalisation: h[k] = (w, v_k) with w -= h[k] v_k in turn, h[k1] = ||w||,
// vnext = w / ||w||, in k1 + 2 launches (each step reduces the previous
// step's partial sums itself; the values are those of dot + axpy in the same
// order).  part: 2 kRedBlocks doubles.
template <typename T>
void mgs_arnoldi(T *w, const T *V, int64_t n, int k1, double *h, T *vnext, double *part, hipStream_t st);

// mode 0 product, 1 defect, 2 Jacobi (x = old iterate, y = new) over the
// interior rows (Dirichlet rows: boundary); psum (modes 0, 1): the upper sums
// that sor_sweeps left for this x, which halves the values read
template <typename T>
void rows_apply(const DevLayout &D, int mode, const T *val, const T *x, const T *f, T *y, double omega,
                hipStream_t st, const T *psum = nullptr);
// n SOR (forward) or SSOR sweeps in colour order, one launch per line group;
// the Dirichlet entries of x are left as they are.  psum (SSOR): N entries of
// scratch that hold the upper sums of the result's rows afterwards.  zero: the
// interior of x is zero (its contribution is not read); bnd_set (optional,
// with zero): a device flag that is not 0 if the boundary of x is not zero;
// planes: a launch per plane colour instead of one per line group where
// plane_sweeps_used (the same result bit for bit).
bool plane_sweeps_fit(const DevLayout &D);   // M <= 17
bool plane_sweeps_used(const DevLayout &D);  // and Q2 levels with M = 33
template <typename T>
void sor_sweeps(const DevLayout &D, const T *val, T *x, const T *f, T *psum, double omega, bool ssor, int n, bool zero,
                const int *bnd_set, bool planes, hipStream_t st);
// the same on the row-scaled FP16 values and the FP32 1/diag of scaled_values
// (psum: sums of the scaled values)
void sor_sweeps_scaled(const DevLayout &D, const _Float16 *val16, const float *dinv, float *x, const float *f,
                       float *psum, double omega, bool ssor, int n, bool zero, const int *bnd_set, hipStream_t st);
// the lines of a launch over all interior lines / over a line group, and its
// number of units
LineSet all_lines(const DevLayout &D, int *units);
LineSet group_lines(const DevLayout &D, int g, int *units);
// out = {||u - u_h||_L2, |u - u_h|_H1} of the lattice function u (FP64) against
// the example's exact solution with the rule of qref/tab (part: 2 kRedBlocks)
void fe_errors(const DevLayout &D, const double *prm_dev, const double *qref, const double *tab, int nq,
               const double *u, double *part, double *out, hipStream_t st);
// a == b bit for bit (n doubles; flag: one device int of scratch; synchronises st)
bool bits_equal(const double *a, const double *b, int64_t n, int *flag, hipStream_t st);
// x of the level fits the LDS of the one-workgroup kernel
inline bool sweep_wg_fits(const DevLayout &D, size_t s) { return (int64_t)D.N * (int64_t)s <= kSweepLdsBytes; }
// pair table of a small level: pair_tiles(L) tiles of kPairTile entries per
// line group
constexpr int kPairTile = 256;
int pair_tiles(const Layout &L);
size_t pair_table_size(const DevLayout &D);
void pair_table(const DevLayout &D, int2 *pairs, hipStream_t st);
// the row-scaled FP16 copy of the FP32 stencil values (a_ij / a_ii,
// saturated to the finite FP16 range) and dinv = 1 / a_ii on the active rows
void scaled_values(const DevLayout &D, const float *val, _Float16 *val16, float *dinv, hipStream_t st);
// the coarse-level smoothing loop of TMultiGrid3D (MultiGrid3D.C:225-337) in
// one workgroup (levels with sweep_wg_fits): sweeps of kind 1 Jacobi, 2 SOR,
// 3 SSOR while ||f - A x|| > red ||f - A x_0|| and fewer than maxit were
// made; xj: scratch of D.N entries
template <typename T>
void coarse_wg(const DevLayout &D, const T *val, T *x, const T *f, double omega, int kind, int maxit, double red,
               T *xj, hipStream_t st);
// Dirichlet rows: mode 0 y=x, 1 y=f-x, 2 y=f, 3 y=0
template <typename T> void boundary(const DevLayout &D, int mode, T *y, const T *x, const T *f, hipStream_t st);
template <typename T>
void prolongate(const DevLayout &C, const DevLayout &F, const T *xc, T *xf, hipStream_t st);
// xf += damp * (P xc with the fine Dirichlet nodes set to 0): prolongation,
// CorrectNodes and the damped update of TMultiGrid3D::Cycle in one launch
// (the Dirichlet nodes of a layout are its lattice surface)
template <typename T>
void prolongate_add(const DevLayout &C, const DevLayout &F, const T *xc, T *xf, double damp, hipStream_t st);
// xc: the cycle's restriction, which also sets the coarse Dirichlet entries
// to 0 (CorrectDefect) and the coarse iterate xc to 0 (Reset)
template <typename T>
void restrict_(const DevLayout &C, const DevLayout &F, T *rc, const T *rf, hipStream_t st, T *xc = nullptr);
// the start of a cycle from zero: f = v, x = 0, *bnd_set = 0; then
// start_boundary: x = f on the Dirichlet nodes, *bnd_set = 1 if any is not 0
template <typename T> void start_zero(T *f, T *x, const T *v, int *bnd_set, int64_t n, hipStream_t st);
template <typename T> void start_boundary(const DevLayout &D, T *x, const T *f, int *bnd_set, hipStream_t st);
// coarsest-level solve: y_I = W x with W = A_II^-1 [I, -A_IB] (n_I x N, lattice
// columns; iidx: interior row -> lattice node); y_B = x_B is set separately
template <typename T>
void gemv_coarse(int nI, int N, const double *W, const int *iidx, const T *x, T *y, hipStream_t st);
// W of the level by Gauss-Jordan with partial pivoting (cidx: lattice node ->
// interior row or -1; aug: workspace of coarse_inverse_scratch doubles; piv: n_I
// ints)
int64_t coarse_inverse_scratch(int nI, int N);
void coarse_inverse_dense(const DevLayout &D, const double *val, const int *iidx, const int *cidx, int nI, double *aug,
                          int *piv, double *W, hipStream_t st);
template <typename T, typename U> void gather(T *out, const U *in, const int *map, int64_t n, hipStream_t st);
template <typename T>
void csr_spmv(int n, const int *rp, const int *kc, const T *val, const T *x, T *y, hipStream_t st);
// r = b - A x on a CSR matrix
template <typename T>
void csr_defect(int n, const int *rp, const int *kc, const T *val, const T *x, const T *b, T *r, hipStream_t st);
// CSR entries with the level's pattern (reference numbering) into the line
// layout's values of the active rows (the inverse of values_to_csr there)
void csr_to_values(const DevLayout &D, const int *rowptr, const int *kcol, const int *dof2lat, int64_t active,
                const double *in, double *val, hipStream_t st);
template <typename T>
void values_to_csr(const DevLayout &D, const int *rowptr, const int *kcol, const int *dof2lat, int64_t active,
                const T *val, double *out, hipStream_t st);
// example: prm[PMX_PRM_EXAMPLE] (selects evaluating the coefficients inline or
// through the quadrature-point buffer); form: prm[PMX_PRM_FORM]; kc: cell
// buffer of n^3 x 27 x 28 doubles for the Q2 one-matrix forms; qp_given: qpbuf already holds the
// quadrature-point records (coefficients from host callbacks)
// ftab (optional): room for phase_tab_len(n, nq) doubles; with it the
// curl-Fourier example's coefficients come from per-level phase tables.
// corner (required for CELL_MEASURE 4, else unused): the per-cell frame codes
// of Numbering::corner on the device.
void assemble(const DevLayout &D, const double *prm_dev, int example, int form, const double *qref, int nq,
              const double *tab, double *qpbuf, double *kc, double *val, double *val2, double *rhs, hipStream_t st,
              bool qp_given = false, double *ftab = nullptr, const uint8_t *corner = nullptr);
// doubles of the phase tables of a level with n cells per direction and an
// nq-point tensor rule: complex factors per mode, axis, cell index and 1D point
// of the 3 x 8 modes of PMX_PRM_FOURIER or the 64 of PMX_PRM_GRF
constexpr int kFourierModes = 24, kGrfModes = 64;
inline int64_t phase_tab_len(int n, int nq) {
  const int np = nq <= 8 ? 2 : (nq <= 27 ? 3 : 4);
  return 2 * (int64_t)kGrfModes * 3 * n * np;
}
// y[idx[i]] = v[i]
void scatter(double *y, const int *idx, const double *v, int n, hipStream_t st);
constexpr int64_t kCellMatrixDoubles = 27 * 28;  // cell buffer entries per Q2 cell
// time stepping (TSystemTCD3D): nodal interpolation of the example's initial
// function, the system matrix val = mass (+ k) + c a, and the Crank-Nicolson
// / theta right-hand side (k, k_old: the SUPG time-derivative matrix K and
// K oldsol, nullptr for the Galerkin forms)
void interpolate(const DevLayout &D, const double *prm_dev, double *x, hipStream_t st);
// val = mass (+ k) + c a; val32 (if not null) receives its FP32 rounding
void system_matrix(const DevLayout &D, double *val, float *val32, const double *mass, const double *k, const double *a,
                   double c, hipStream_t st);
// the FP32 copy of the level's values
void values32(const DevLayout &D, const double *val, float *val32, hipStream_t st);
void tcd_rhs(const DevLayout &D, const double *oldrhs, const double *rhs, const double *m_old, const double *a_old,
             const double *k_old, double t3, double t4, double t2, double *B, hipStream_t st);
void givens(double *H, double *cs, double *sn, double *s, int i, int ld, double *res, hipStream_t st);
void backsolve(const double *H, const double *s, double *y, int k, int ld, hipStream_t st);
template <typename T, typename X>
void multi_axpy(X *x, const T *z, const double *y, int k1, int64_t n, int64_t stride, hipStream_t st);
void set_scalar(double *dst, const double *src, double scale, hipStream_t st);

}  // namespace pmx
