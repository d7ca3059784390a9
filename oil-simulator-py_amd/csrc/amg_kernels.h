// Launchers of the Ruge-Stueben setup kernels (amg_setup.hip) and of the dense
// coarsest-level factor/solve (coarse.hip).
#pragma once

#include "common.h"

namespace impes {

class Readback;  // prims.h

constexpr signed char kC = 0;  // coarse point marker (reference: cf_marker 0 = C)
constexpr signed char kF = 1;  // fine point marker

// diag[i] = a_ii (0 if absent); inv_relax = min(1/max(|a_ii|, 0.3*sum_j|a_ij|, 1e-30), 1e2)
void launch_diag_relax(int n, const int* rp, const int* ci, const double* v, double* diag, double* inv_relax64,
                       float* inv_relax32, hipStream_t s);
// launch_diag_relax (diag not written) and the padded FP32 values v4 of the same
// rows (as launch_csr4_values) in one pass
void launch_diag_relax_pad4(int n, const int* rp, const int* ci, const double* v, const int* rp4, float* v4,
                            double* ir64, float* ir32, hipStream_t s);
// number of rows with |a_ii| < thr (lower-median test of the equilibration switch)
void launch_count_small_diag(int n, const double* diag, double thr, int* flags, hipStream_t s);
// dh[i] = 1/sqrt(max(|diag_i|, 1e-30))
void launch_dhalf_inv(int n, const double* diag, double* dh, hipStream_t s);
// vo[e] = v[e]*dh[row]*dh[col]
void launch_sym_scale(int n, const int* rp, const int* ci, const double* v, const double* dh, double* vo,
                      hipStream_t s);

void launch_strength(int n, long long nnz, const int* rp, const int* ci, const double* v, double theta,
                     unsigned char* strong,
                     hipStream_t s);
// tpos[e] = position of (col,row) in row col, -1 if absent
void launch_transpose_pos(int n, long long nnz, const int* rp, const int* ci, int* tpos, hipStream_t s);
// C/F split: symmetrised strong graph, strict local maxima of (deg, hash, index), lift of F points with no C neighbour
void launch_cf_split(int n, long long nnz, const int* rp, const int* ci, const unsigned char* strong,
                     const int* tpos, int* deg, signed char* is_max, signed char* cf, hipStream_t s);
// iterated independent-set split on the symmetrised strong graph with the same
// (deg, hash, index) order: rounds of local-max selection among undecided points,
// whose undecided neighbours become F, until every point is decided (no lift needed)
// first (may be null): values fetched with the first test of the rounds
void launch_cf_split_iterated(int n, long long nnz, const int* rp, const int* ci, const unsigned char* strong,
                              const int* tpos, int* deg, signed char* newc, int* undecided, signed char* cf,
                              Readback* first, hipStream_t s);
// cf[i] = C where |a_ii| > ratio * sum_j!=i |a_ij| (Dirichlet-like rows)
void launch_force_dominant(int n, const int* rp, const int* ci, const double* v, double ratio, signed char* cf,
                           hipStream_t s);
// promote F points with no strong C neighbour
void launch_orphans(int n, const int* rp, const int* ci, const unsigned char* strong, const signed char* cf_in,
                    signed char* cf_out, int* is_c, hipStream_t s);

// interpolation
void launch_interp_pass_a(int n, const int* rp, const int* ci, const double* v, const unsigned char* strong,
                          const signed char* cf, double* sum_strong, int* cnt_c, hipStream_t s);
void launch_interp_count(int n, const int* rp, const int* ci, const unsigned char* strong, const signed char* cf,
                         const double* sum_strong, const int* cnt_c, int* cand, hipStream_t s);
void launch_interp_expand(int n, long long nnz, const int* rp, const int* ci, const double* v,
                          const unsigned char* strong, const signed char* cf, const double* sum_strong,
                          const int* cnt_c, const int* f2c, const long long* cand_ptr, unsigned long long* keys,
                          double* vals, hipStream_t s);
// final F-row weights; trunc > 0 / pmax > 0 truncate each F row afterwards: weights below
// trunc * row max are dropped, then all but the pmax largest (ties: lower coarse column
// first), and the kept weights are rescaled to the row's previous sum
void launch_interp_reduce(int n, const int* rp, const int* ci, const signed char* cf, const int* f2c,
                          const long long* cand_ptr, const unsigned long long* keys, const double* vals,
                          double trunc, int pmax, int* out_cols, double* out_vals, int* pcnt, hipStream_t s);
void launch_interp_gather(int n, const long long* cand_ptr, const int* cols_tmp, const double* vals_tmp,
                          const int* prp, int* pci, double* pv, hipStream_t s);

// transpose (R = P^T): counts per column, fill, key build, gather after sort
void launch_col_count(int nnz, const int* ci, int* cnt, hipStream_t s);
void launch_transpose_fill(int n_rows, const int* rp, const int* ci, const int* rrp, int* cursor,
                           unsigned long long* keys, hipStream_t s);
// after the per-column sort: rci[p] = source row, rv[p] = source value
void launch_transpose_finish(int nnz, const unsigned long long* keys, const double* src_v, int* rci, double* rv,
                             hipStream_t s);

// SpGEMM C = L*M, symbolic through expanded products sorted per row
void launch_spgemm_count(int n, const int* lrp, const int* lci, const int* mrp, int* cnt, hipStream_t s);
// keys[t] = (column, local index); ex_e/ex_f[t] = (left entry, right entry) in expansion order
void launch_spgemm_expand(int n, long long left_nnz, long long products, const int* lrp, const int* lci, const int* mrp, const int* mci,
                          const long long* prod_ptr, unsigned long long* keys, int* ex_e, int* ex_f, hipStream_t s);
void launch_spgemm_unique_count(int n, const long long* prod_ptr, const unsigned long long* keys, int* cnt,
                                hipStream_t s);
// writes C column indices, product segment pointers (int64, nnzC+1) and the sorted
// operand index pairs (left entry, right entry) of every product
void launch_spgemm_finalize(int n, const long long* prod_ptr, const unsigned long long* keys, const int* crp,
                            const int* ex_e, const int* ex_f, int* cci, long long* seg, int* pe, int* pf,
                            long long total_products, int nnz_c, hipStream_t s);
// C.v[o] = sum_{t in seg(o)} Lv[pe[t]] * Mv[pf[t]]
void launch_spgemm_numeric(int nnz_c, const long long* seg, const int* pe, const int* pf, const double* lv,
                           const double* mv, double* cv, hipStream_t s);

// coarsest level (coarse.hip). pin is a device flag written by launch_pin_decide and
// read by the kernels below, so the decision never leaves the device.
// pin = (mode == reference) || (mode == auto && every row has |row sum| <= 1e-8 |a_ii|)
// *bad (the failure flag of the inverse) is cleared
void launch_pin_decide(int n, const int* rp, const int* ci, const double* v, int mode, int* pin, int* bad,
                       hipStream_t s);
// Inverse of the (optionally DOF-0-pinned) level matrix in M (dense_pad(n)^2 doubles,
// and its transpose behind it, n <= kDenseMfmaMax): blocked Gauss-Jordan without pivoting on the matrix cores
// (dense_mfma.hip), with W (dense_pad(n)^2) and P (kDenseWorkP) as work; sets *bad
// when the operator is not SPD: a pivot that is not positive, and up to
// kDenseStrictMax rows also an asymmetry or a pivot of rounding size. Then
// launch_gauss_jordan_inverse with partial pivoting (n <= kDensePivotMax, aug n x 2n)
// replaces M when *bad. Applied by launch_dense_mv_* (with pin: b[0] treated as 0).
constexpr int kDenseMfmaMax = 4096;
constexpr int kDenseStrictMax = 160;
constexpr int kDensePivotMax = 512;
constexpr int kDenseWorkP = 2 * 64 * 64 + 192;  // two pivot inverses, the diagonal (strict sizes)
int dense_pad(int n);
void launch_dense_inverse_mfma(int n, const int* rp, const int* ci, const double* v, const int* pin, double* M,
                               double* W, double* P, int* bad, hipStream_t s);
void launch_dense_mv_f64(int n, const int* pin, const double* M, const double* b, double* x, hipStream_t s);
void launch_dense_mv_f32(int n, const int* pin, const double* M, const float* b, float* x, hipStream_t s);
void launch_gauss_jordan_inverse(int n, const int* rp, const int* ci, const double* v, const int* pin, const int* bad,
                                 double* aug, double* M, hipStream_t s);
// b[0] = 0 when *pin (Jacobi coarsest path)
void launch_pin_rhs_f64(const int* pin, double* b, hipStream_t s);
void launch_pin_rhs_f32(const int* pin, float* b, hipStream_t s);


// The coarse end of the cycle as one matrix (tail.hip): levels of at most kTailMax
// rows and kTailNnz entries above a coarsest level of at most kTailCoarsest rows,
// whose vectors fit kTailLds bytes of LDS for one workgroup's columns.
constexpr int kTailMax = 2048;
constexpr int kTailNnz = 40000;
constexpr int kTailCoarsest = 400;
constexpr int kTailLevels = 8;  // the coarsest one included
constexpr size_t kTailLds = 157 * 1024;
struct TailLevel {
  int n = 0;
  int so = 0;                // first of its slice offsets (in 64-entry lines) in TailArgs::so
  const void* ell = nullptr; // sliced operator
  const double* ir = nullptr;
  const int *prp = nullptr, *pci = nullptr, *rrp = nullptr, *rci = nullptr;
  const double *pv = nullptr, *rv = nullptr;
  int x = 0, y = 0, b = 0;   // LDS offsets of its vectors
};
struct TailArgs {
  int levels = 0;  // non-coarsest levels; lv[levels] is the coarsest
  TailLevel lv[kTailLevels];
  const int* so = nullptr;        // slice offsets of all levels
  int so_len = 0;
  const double* inv_t = nullptr;  // transposed inverse of the coarsest operator
  int inv_ld = 0;
  const int* pin = nullptr;
  int pre = 0, post = 0;
  double omega = 0.0;
  int part = 0, splits = 0;  // LDS offset and count of the coarsest solve's partial sums
  int ld = 0;         // row stride of B (tail_ld)
  void* B = nullptr;  // float (precision 32) or double; formed in FP64
};
int tail_slices(int n);
void launch_tail_slices(int n, const int* rp, int* so, hipStream_t s);  // tail_slices(n) + 1 offsets
size_t tail_ell_bytes(long long lines);
void launch_tail_pack(int n, const int* rp, const int* ci, const double* v, const int* so, void* ell, hipStream_t s);
bool tail_fits(const TailArgs& A);  // from the levels' sizes
constexpr int tail_ld(int n) { return (n + 12) / 8 * 8; }  // row stride of B: n and the last workgroup's padding
void launch_tail_form(int precision, TailArgs A, hipStream_t s);
void launch_tail_mv_f32(int n, int ld, const float* B, const float* b, float* x, hipStream_t s);
void launch_tail_mv_f64(int n, int ld, const double* B, const double* b, double* x, hipStream_t s);

}  // namespace impes
