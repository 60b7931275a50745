// kernels.hpp -- host launchers of the gfx950 kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

#include "../../include/dpg_capi.h"
#include "device_common.hpp"

namespace dpg {

struct DeviceError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// C(i,j) = alpha * sum_k X(k,i) Y(k,j) + beta * C(i,j) for every cell of a batch
struct GemmArgs {
  const double* X;
  int64_t ldx, sx;  // X(k,i) = X[k*ldx + i], per-cell stride sx (0: shared)
  const double* Y;
  int64_t ldy, sy;
  double* C;
  int64_t ldc, sc;  // C(i,j) = C[i + j*ldc]
  int32_t m, n, k, lower;
  double alpha, beta;
  int32_t tiles_m, ntiles, ncells;
  // optional: scale C(i,j) by srow[i] * scol[j] (per-cell vectors, stride ss)
  const double* srow;
  const double* scol;
  int64_t ss;
  // optional (mixed-precision GEMMs): scale X(k,i) by px[i] and Y(k,j) by py[j]
  // before the conversion to the low-precision operand format
  const double* px;
  const double* py;
  // optional (FP64 GEMMs): k runs over segments of kseg rows (kseg a multiple of
  // the 16-row k-chunk); bit s of kmask[tile] clear means segment s is zero for
  // this tile's rows or columns and is skipped (adds exact zeros otherwise)
  const uint64_t* kmask;
  int64_t kseg;
  // optional (with kmask): kw[tile*nseg + s] scales the staged X rows of segment s
  // (a segment standing for several equal terms counts once per term)
  const double* kw;
  int32_t nseg;
  // optional (the trailing update, lower): its results also as outputs per cell, the
  // symmetric matrix of the first nout rows row by row and row nout; drop: C itself
  // is not written
  double* sym;
  double* row;
  int32_t nout, drop;
};

// the point weights of all of a cell's points; nside_points: nsides * Qs, or 0 without side variables
void launch_point(int dim, const DevProgram* prog, const DevTables& tab, int QG, int Q, int Qs, int nside_points,
                  int ncells, const double* nodes, const int8_t* par, const double* coefs, int ncoef, int nsides,
                  const dpg_load_desc& load, double* Wip, double* Wvol, double* Wrhs, double* Wside, hipStream_t st);
void launch_operand(int dim, const double* W, int ng, int nvar, const double* R, const int32_t* vod, int N, int npts,
                    int ncells, double* out, int64_t sc, int64_t sb, int64_t sp, hipStream_t st);
// Gram operand: out[c][lt*QGp + q][j] = weighted value of IP term lt at point q
// for test dof j (G = out^T out); s[c][j] = 1/sqrt(G_jj). reach (optional): the term
// masks of G's lower 64-tiles; terms that reach none of 64 dofs are not written there
void launch_ip_operand(int dim, const double* Wip, int n_lt, int nvar, const double* R, const int32_t* vod, int N,
                       int QG, int QGp, int ncells, double* out, int64_t sc, int64_t ld, double* s, int64_t ss,
                       const uint64_t* reach, hipStream_t st);
enum { kGemmGram = 0, kGemmBmat = 1, kGemmUpdate = 2 };
// points whose weights one operand workgroup stages in LDS, and the LDS bytes
// of the weight-staging kernels (at most kMaxLds per workgroup)
constexpr int kOperandPoints = 8;
constexpr size_t kMaxLds = 64 * 1024;
inline size_t operand_lds_bytes(int ng, int nvar, int dim) {
  return sizeof(double) * kOperandPoints * (size_t)ng * nvar * (dim + 1);
}
inline size_t ip_operand_lds_bytes(int n_lt, int nvar, int dim) { return sizeof(double) * (size_t)n_lt * nvar * (dim + 1); }
inline size_t ip_digits_lds_bytes(int n_lt, int nvar, int dim) {
  return sizeof(double) * 32 * (size_t)n_lt * nvar * (dim + 1);
}
void launch_gemm(GemmArgs g, int role, hipStream_t st, int tile = 64);
void launch_fill_i32(int32_t* p, int n, int32_t v, hipStream_t st);
// copies info (n) to out (optional) and writes the count of non-zero entries to *count
void launch_info_count(const int32_t* info, int n, int32_t* out, int32_t* count, hipStream_t st);
// sum-factorised Gram matrix, lower triangle of A's first N rows/columns: unscaled, or S G S
// with the DPOEQU factors s; diag_only: G's diagonal alone (what s is computed from)
void launch_gram_sf(int dim, const SfBlockPair* bps, int nbp, const SfPair* pairs, const double* F, int nF, int q,
                    const double* Wip, int n_lt, int na, int QG, double* A, int64_t lda, int64_t sA, int ncells,
                    size_t lds_bytes, hipStream_t st, const double* s = nullptr, int64_t ss = 0,
                    bool diag_only = false);
// s[i] = 1 / sqrt(A[r0 + i][r0 + i]), i < n (the DPOEQU factors alone)
void launch_scale_factors(const double* A, int64_t lda, int64_t sA, int r0, int n, double* s, int64_t ss, int ncells,
                          hipStream_t st);
// the volume part of B, sum-factorised: block pairs (trial field block, test
// block) and their pairs, 1D tables of 4 families on the stiffness points
// (q per direction), point weights Wvol (na per point), stores scaled by s
// (the DPOEQU factors of the test columns; none when s is NULL)
void launch_bmat_sf(int dim, const SfBlockPair* bps, int nbp, const SfPair* pairs, const double* F, int nF, int q,
                    const double* Wvol, int na, int Q, double* A, int64_t lda, int64_t sA, const double* s,
                    int64_t ss, int ncells, size_t lds_bytes, hipStream_t st);
// the side part of B, sum-factorised per side: side A a trace or flux block on
// one side (rows N + its offset), side B a test block restricted to the side;
// nfam 1D families per block pair from F + foff (tangential directions on the
// side's points, the normal one at the side's coordinate), point weights Wside
// (npts side points per cell, na per point, the pair's side from woff)
void launch_bmat_side_sf(int dim, const SfBlockPair* bps, int nbp, const SfPair* pairs, const double* F, int nF,
                         int nfam, int q, const double* Wside, int npts, int na, double* A, int64_t lda, int64_t sA,
                         const double* s, int64_t ss, int ncells, size_t lds_bytes, hipStream_t st);
// the same contraction with FP64 operands converted on load to FP32 (precision
// DPG_PREC_FP32) or to hi+lo BF16/FP16 pairs (DPG_PREC_BF16X3/FP16X3, products
// hi*hi + hi*lo + lo*hi), FP32 MFMA accumulation, FP64 epilogue
void launch_gemm_mixed(GemmArgs g, int precision, int role, hipStream_t st);
// Int8 digit split of the Gram product (precision DPG_PREC_INT8SPLIT).
// The equilibrated operand x(k,j) = s_j out(k,j), with s_j = 1/||out(:,j)|| so
// that |x| <= 1, is written as kI8Digits signed digits of 7 bits:
//   x = sum_p d_p 2^(1-7p) + r,   d_p in [-64, 64],   |r| <= 2^(-7 kI8Digits).
// Digit planes, bytes per cell: kI8Digits * (KG/32) * NR * 32, plane p, k-chunk c
// (32 consecutive k), row j at ((p*(KG/32) + c)*NR + j)*32 + k%32; NR = N rounded
// up to 64, rows N..NR-1 zero. s[c][j] as launch_ip_operand.
constexpr int kI8Digits = 8;
void launch_ip_digits(int dim, const double* Wip, int n_lt, int nvar, const double* R, const int32_t* vod, int N,
                      int QG, int QGp, int NR, int ncells, int8_t* dig, int64_t sd, double* s, int64_t ss,
                      hipStream_t st);
// G(i,j) (lower, i >= j, rows and columns < N) = sum_k x(k,i) x(k,j) from the
// digit planes: the digit products d_p(i) d_q(j) with p + q <= kI8Digits + 1
// on v_mfma_i32_32x32x32_i8, exact int32 sums per level p + q, the levels
// scaled by 2^(2-7(p+q)) and added in FP64 from the smallest. kmask/kseg as
// GemmArgs, kseg in k (a multiple of 32).
struct I8GramArgs {
  const int8_t* dig;
  int64_t sd;  // bytes per cell
  int32_t N, NR, nch, ncells;
  double* C;
  int64_t ldc, sc;
  const uint64_t* kmask;
  int64_t kseg;
  int32_t tiles_m, ntiles;
};
void launch_gram_i8(I8GramArgs a, hipStream_t st);
constexpr int kPanelMax = 128;  // columns of a factorisation panel
// A panel [k0, k0 + kb) of the cells' augmented matrices of D rows, columns
// [kbeg, k0) being factored (k0 - kbeg a multiple of 64).
struct PanelArgs {
  double* A;
  int64_t lda, sA;
  int32_t D, k0, kb, kbeg;
  // the diagonal factor as potrf_block leaves it, kPanelMax doubles a column:
  // Lt[j * kPanelMax + m] = L[m][j] below the diagonal, 1 / L[j][j] on it, zeros above
  // it and past the panel (its width rounded up to 32 columns)
  double* Lt;
  int64_t sLt;
  const int32_t* z;  // optional: the first column of each row of A that can be non-zero
  // optional: factors of rows and columns [kbeg, kbeg + ns), applied as the panel's
  // columns are read
  const double* s;
  int64_t ss;
  int32_t ns;
  int32_t ntiles;
};
// The diagonal block: its update by columns [kbeg, k0), POTRF. Ld: per-cell (rows, 64)
// store of the factored 64-column diagonal blocks (row k0 + r, column r'); rows below
// one within a wider panel go to A. info: first failing column (1-based) if none is set.
void launch_potrf(const PanelArgs& g, double* Ld, int64_t sLd, int ncells, int32_t* info, hipStream_t st);
// the rows below it: A[k0 + kb:, panel] -= A[.., kbeg:k0] A[panel, kbeg:k0]^T, then X L^-T
void launch_update_solve(PanelArgs g, int ncells, hipStream_t st);
// The rows of B and the load vector in FP64 from the point weights (contract.hip).
// A task is up to bmat_rows(dim) rows of one trial block, a phase the tasks of up
// to kBmatPhaseRows consecutive rows of the augmented matrix, a chunk up to 64
// test dofs of one variable.
constexpr int bmat_rows(int dim) { return dim == 2 ? 16 : 32; }
constexpr int kBmatPhaseRows = 64;
enum { kBmatVolume = 0, kBmatSide = 1, kBmatLoad = 2 };
enum { kBmatField = 0, kBmatTrace = 1, kBmatFlux = 2 };
struct BmatTask {
  int32_t kind, table;
  int32_t row, nf;           // first row within the phase, rows
  int32_t f0, card;          // first basis function of the block, functions per point of its table
  int32_t w0, wstride;       // first point weight of the cell, weights per point
  int32_t point0, npts;      // first row of the kind's reference prims, points
  uint32_t vars;             // test variables some term couples the block with
};
struct BmatPhase {
  int32_t row0, nrows, task0, ntasks;
};
struct BmatChunk {
  int32_t i0, n, var;
};
struct BmatArgs {
  const BmatPhase* phases;
  const BmatChunk* chunks;
  const BmatTask* tasks;
  const double *Wvol, *Wside, *Wrhs;  // point weights, per-cell strides below
  int64_t nWvol, nWside, nWrhs;
  const double *R_vol, *R_side, *field, *trace, *flux;
  double* A;  // rows N .. N+M+1 written (the residual row as zeros)
  int64_t lda, sA;
  int32_t N;
  const double* s;  // optional: column scales, per-cell stride ss
  int64_t ss;
  int32_t nphases;
  // optional: the DPOEQU factors too, from the IP terms' point weights
  double* s_out;  // per-cell stride ss
  const double *Wip, *R_ip;
  int64_t nWip;
  int32_t QG, n_lt, nvar;
};
void launch_bmat(int dim, const BmatArgs& g, int nchunks, int ncells, hipStream_t st);
// the load vector's row (and the residual's zeros) alone; phases: the one that holds it
void launch_load(int dim, const BmatArgs& g, int nchunks, int ncells, hipStream_t st);
// The dense Gram matrix of small cells in FP64, unscaled, into A's lower triangle
// (contract.hip): up to kGramMaxN test dofs, 4 waves with at most kGramTiles of the
// lower triangle's 16 x 16 tiles each.
constexpr int kGramMaxN = 80, kGramTiles = 4;
constexpr int kGramEntries = 8;  // operand entries a thread forms per step
constexpr int gram_pitch(int N) { return (N + 15) / 16 * 16 + 4; }
inline size_t gram_lds_bytes(int N, int kc, int weights) {
  return sizeof(double) * ((size_t)2 * kc * gram_pitch(N) + (size_t)kc * weights);
}
struct GramArgs {
  const uint32_t* active;    // per IP term and wave (4): the wave's tiles the term reaches
  const uint32_t* twice;     // ... of them those it enters twice
  const int32_t* var_of_dof;
  const double* R;           // (QG, npr, N)
  const double* Wip;         // (QG, n_lt, nvar, npr) per cell, stride nWip
  int64_t nWip;
  int32_t N, QG, n_lt, nvar;
  int32_t kc;                // points per step, a multiple of 4
  double* A;
  int64_t lda, sA;
  double* G;                 // optional: (N, N) per cell
};
void launch_gram(int dim, const GramArgs& g, int ncells, hipStream_t st);
// Small cells (D = N + M + 2 <= kCellMaxD: the lower triangle of the augmented
// matrix fits one compute unit's LDS): everything after the contractions in one
// launch (cellfactor.hip). A holds the columns [G; B; l; r] scaled to [SGS; SB; Sl;
// Sr], or with s the columns [G; B; l] to be scaled as they are read; every output
// but info is optional; info[c] is the LAPACK INFO of the cell.
constexpr int kCellMaxD = 192;
struct CellFactorArgs {
  const double* A;
  int64_t lda, sA;
  int32_t N, M, F;
  double *K, *rhs, *schur, *schur_rhs, *eta2;
  double* factor;  // (N+M+1, N) row-major, per-cell stride sF
  int64_t sF;
  const double* s;         // optional: DPOEQU factors, per-cell stride ss, A unscaled
  int64_t ss;
  const double* u;         // with s: trial coefficients (M per cell) of the residual r = l - B u (NULL: r = 0)
  double* factor_scale;    // with s: its copy (N per cell)
  double* z;  // Lt^-1 S (l - B u) (N per cell): the residual row's factored columns
  int32_t* info;
};
void launch_cell_factor(CellFactorArgs g, int ncells, hipStream_t st);
// u_F = K_FF^-1 (rhs_F - K_FT u_T) of cells of F + 1 <= kCellMaxD; info as CellFactorArgs'
void launch_cell_recover(const double* K, const double* rhs, int M, int F, double* u, int ncells, int32_t* info,
                         hipStream_t st);
void launch_scaling(double* A, int64_t lda, int64_t sA, int r0, int D, int n, int ncol, double* s, int64_t ss,
                    int ncells, hipStream_t st);
void launch_residual_row(double* A, int64_t lda, int64_t sA, int N, int M, int r0, int row_l, int row_r,
                         const double* u, int ncells, hipStream_t st);
// per cell of n doubles: out[2c] = |a_c - b_c|^2, out[2c+1] = |b_c|^2
void launch_cell_diff_norms(const double* a, const double* b, int64_t n, int ncells, double* out, hipStream_t st);
void launch_extract_sym(const double* A, int64_t lda, int64_t sA, int r0, int n, double sign, double* out, int ncells,
                        hipStream_t st);
// field recovery after a condensed solve: S K_FF S and the row s (rhs_F - K_FT u_T) into A
void launch_recover_setup(const double* K, const double* rhs, const double* u, int M, int F, double* A, int64_t lda,
                          int64_t sA, double* s, int64_t ss, int ncells, hipStream_t st);
// e = S Lt^-T y (y = residual row of A): the Riesz representation and the field back solve
void launch_backsolve(const double* A, int64_t lda, int64_t sA, int N, int row_r, const double* Ld, int64_t sLd,
                      const double* s, int64_t ss, double* e, int64_t se, int ncells, hipStream_t st);
// the factored first N columns of the augmented matrices as row-major (N+M+1, N)
// blocks (Lt, (Lt^-1 S B)^T, (Lt^-1 S l)^T), per-cell stride sF
void launch_extract_factor(const double* A, int64_t lda, int64_t sA, int N, int M, const double* Ld, int64_t sLd,
                           double* F, int64_t sF, int ncells, hipStream_t st);
// z = Lt^-1 S (l - B u) and eta2 = z^T z from stored factors (z, eta2 optional)
void launch_factored_residual(const double* F, int64_t sF, int N, int M, const double* u, double* z, int64_t sz,
                              double* eta2, int ncells, hipStream_t st);
// X (N x ncol per cell) = S Lt^-T [Y (nT columns) | y_l (with_y) | z (z != NULL)]
void launch_factor_backsolve(const double* F, int64_t sF, int N, int M, const double* s, int64_t ss, int nT,
                             int with_y, const double* z, int64_t sz, double* X, int64_t sX, int ncol, int ncells,
                             hipStream_t st);
size_t adjoint_lds_bytes(int nvar, int dim, int ncol);
// grad (C, ncoef) of <Kbar, K> + <rbar, rhs> + eta2(u) from X = [G^-1 B | G^-1 l | G^-1 r]
void launch_adjoint(int dim, const DevProgram* prog, const DevTables& tab, int N, int M, int QG, int Q, int Qs,
                    int nsides, int nvar, const double* nodes, const int8_t* par, const double* coefs,
                    const double* X, int64_t sX, int ncol, int nT, int cy, int ce, const double* Kbar,
                    const double* rbar, const double* u, double* grad, int ncells, hipStream_t st);
// grad (C, ncoef) of eta2(u) alone from a stored factor and z = Lt^-1 S (l - B u);
// false (nothing launched) where a cell's points do not fit LDS: launch_adjoint then
bool launch_adjoint_eta(int dim, const DevProgram* prog, const DevTables& tab, int N, int M, int QG, int Q, int Qs,
                        int nsides, int nvar, const double* nodes, const int8_t* par, const double* coefs,
                        const double* F, int64_t sF, const double* s, int64_t ss, const double* z, int64_t sz,
                        const double* u, double* grad, int ncells, hipStream_t st);
void launch_extract_row(const double* A, int64_t lda, int64_t sA, int row, int r0, int n, double sign, double* out,
                        int ncells, hipStream_t st);

}  // namespace dpg
