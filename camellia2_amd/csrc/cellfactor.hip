// cellfactor.hip -- the factorisation of small cells in LDS.
//
// cell_factor_kernel takes the augmented matrices of cells whose whole lower
// triangle fits a compute unit's LDS (D = N + M + 2 <= kCellMaxD) from their
// contractions to every output in one launch: partial Cholesky over the N test
// columns, K, rhs, eta2 and the kept factor, then the partial Cholesky of K
// over the F field columns and the Schur complement. What the panel kernels do
// in two launches per 128 columns and a product, each reading the matrix from HBM.
//
// What bounds it is the chain of pivots: N + F of them, each a square root, a
// divide and a broadcast after the one before (42 us for the 92 of the 2D
// Poisson cells of N = 65, M = 55 at 16 cells, 44 us at 256, 425 us at 4,096, 2 cells
// of 8 waves per compute unit; the 14 launches it replaced took 172 us at 16 cells and
// 870 us at 4,096). 16-column panels keep a panel's rows in registers and
// leave the rest to rank-16 MFMA updates.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <utility>

#include "../../include/dpg_capi.h"
#include "device_common.hpp"
#include "kernels.hpp"

namespace dpg {

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

// The lower triangle in LDS: 16-column panels, panel p holding rows 16p and
// below column by column with one double of padding per column (rows and
// columns of a panel are then both read without bank conflicts).
struct CellLds {
  int np;  // panels: D rounded up to 16, over 16
  __device__ int pitch(int p) const { return 16 * (np - p) + 1; }
  __device__ int base(int p) const { return 256 * (p * np - p * (p - 1) / 2) + 16 * p; }
  __device__ int at(int row, int col) const {
    const int p = col >> 4;
    return base(p) + (col & 15) * pitch(p) + row - 16 * p;
  }
};

// sqrt(d) and its reciprocal by Goldschmidt's iteration from the hardware's estimate,
// each with a last correction from its exact residual: sqrt's and a division's results
// in all of 1.7e7 random d, the reciprocal one unit off for a root of all ones (the
// known exception), for d far from the ends of the exponent range, which the pivots of
// matrices with ones on the diagonal are. 13 dependent operations; the scaled square
// root and the division after it have 2.5 times that, and the next pivot waits for them.
__device__ inline void sqrt_and_reciprocal(double d, double& sd, double& rs) {
  const double y = __builtin_amdgcn_rsq(d);
  double g = d * y, h = 0.5 * y;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
  }
  sd = fma(fma(-g, g, d), h, g);
  h *= 2.0;
  rs = fma(fma(-sd, h, 1.0), h, h);
}

// column J of a panel: the pivot, L's column, and the columns after it
template <bool IEEE, int J, int... K>
__device__ inline void panel_column(double (&a)[16], double (&y)[16], int r, int c0, int& fail,
                                    std::integer_sequence<int, K...>) {
  double d = row_lane<J>(a[J]);
  const bool bad = !(d > 0.0);
  fail = bad && fail < 0 ? c0 + J : fail;
  d = bad ? __builtin_nan("") : d;
  double sd, rs;
  if constexpr (IEEE) {
    sd = sqrt(d);
    rs = 1.0 / sd;
  } else {
    sqrt_and_reciprocal(d, sd, rs);
  }
  a[J] *= rs;
  y[J] = r == J ? sd : y[J] * rs;
  auto update = [&](auto k) {
    constexpr int KK = decltype(k)::value;
    if constexpr (KK > J) {
      const double l = row_lane<KK>(a[J]);
      a[KK] = fma(-a[J], l, a[KK]);
      y[KK] = fma(-y[J], l, y[KK]);
      // updated here and now: left to itself the compiler moves the updates to
      // the entries' next use and keeps every broadcast value live meanwhile
      asm volatile("" : "+v"(a[KK]), "+v"(y[KK]));
    }
  };
  (update(std::integral_constant<int, K>()), ...);
}
template <bool FULL, bool IEEE, int... J>
__device__ inline void panel_columns(double (&a)[16], double (&y)[16], int r, int c0, int lo, int hi, int& fail,
                                     std::integer_sequence<int, J...>) {
  auto column = [&](auto j) {
    constexpr int JJ = decltype(j)::value;
    if (FULL || (JJ >= lo && JJ < hi))  // uniform
      panel_column<IEEE, JJ>(a, y, r, c0, fail, std::make_integer_sequence<int, 16>());
  };
  (column(std::integral_constant<int, J>()), ...);
}

// Columns [lo, hi) of panel p: factored in registers by every wave that owns
// rows of it (a lane holds one row's 16 columns, y; every wave also holds the
// 16 rows of the diagonal block, a, in each group of 16 lanes, so the pivots
// and columns of L come from its own lanes and no wave waits for another). The
// panel's later columns are updated along with it if LATER. Entries above the diagonal
// take part with values nothing reads. FULL: lo = 0, hi = 16 without branches, so
// that the next pivot's square root and divide run under this one's updates. IEEE: the
// pivots' root and reciprocal by sqrt and a division (cells without panels before their
// block keep the bits of the panel kernels' column-by-column factor).
template <bool FULL, bool IEEE, bool LATER>
__device__ inline void factor_panel(double* A, const CellLds& L, int p, int lo, int hi, int w, int lane, int& fail) {
  const int h = 16 * (L.np - p), ld = L.pitch(p), r = 64 * w + lane;
  const bool owner = 64 * w < h;
  double* P = A + L.base(p);
  const int rr = min(r, h - 1), dr = lane & 15;
  double a[16], y[16];
  if (owner) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      a[k] = P[k * ld + dr];
      y[k] = P[k * ld + rr];
    }
  }
  __syncthreads();  // the diagonal block is rewritten below by the wave that owns it
  if (!owner) return;
  panel_columns<FULL, IEEE>(a, y, r, 16 * p, lo, hi, fail, std::make_integer_sequence<int, 16>());
  int rs;  // the row once more: one copy shared with the pivots would keep sixteen lane masks live
  asm volatile("v_mov_b32 %0, %1" : "=v"(rs) : "v"(r));
  if (rs < h) {
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if ((FULL || (k >= lo && (LATER || k < hi))) && rs >= k) P[k * ld + rs] = y[k];
  }
}

// C -= X Y^T over the 16 x 16 tiles of the panels after p, X and Y the columns
// [lo, hi) of panel p (the others as zeros), on MFMA; tiles dealt to the waves
__device__ inline void update_trailing(double* A, const CellLds& L, int p, int lo, int hi, int w, int nw, int lane) {
  const int n = L.np - p - 1, nt = n * (n + 1) / 2, ld = L.pitch(p);
  const double* P = A + L.base(p);
  const int kq = lane >> 4, rl = lane & 15;
  int tj = 0, ti = w;  // tile (row ti, column tj) of the lower triangle, column by column
  for (int t = w; t < nt; t += nw) {
    while (ti >= n) {
      ++tj;
      ti = ti - n + tj;
    }
    const int q = p + 1 + tj, ldc = L.pitch(q);
    double* C = A + L.base(q) + kq * ldc + 16 * (ti - tj) + rl;
    const double* X = P + 16 * (ti + 1) + rl;
    const double* Y = P + 16 * (tj + 1) + rl;
    d4 acc;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = C[4 * v * ldc];
#pragma unroll
    for (int k4 = 0; k4 < 16; k4 += 4) {
      if (k4 + 4 <= lo || k4 >= hi) continue;  // uniform
      const int k = k4 + kq;
      const bool in = k >= lo && k < hi;
      const double x = X[k * ld], y = Y[k * ld];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? -y : 0.0, in ? x : 0.0, acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) C[4 * v * ldc] = acc[v];
    ti += nw;
  }
}

__device__ inline void factor_range(double* A, const CellLds& L, int c0, int c1, int w, int nw, int lane, int& fail) {
  for (int c = c0; c < c1;) {
    const int p = c >> 4, lo = c & 15, hi = min(16, c1 - 16 * p);
    if (lo == 0 && hi == 16) factor_panel<true, true, true>(A, L, p, lo, hi, w, lane, fail);
    else factor_panel<false, true, true>(A, L, p, lo, hi, w, lane, fail);
    __syncthreads();
    update_trailing(A, L, p, lo, hi, w, nw, lane);
    __syncthreads();
    c = 16 * p + hi;
  }
}

// A[:, j0:j1] -= A[:, k0:k1] A[j0:j1, k0:k1]^T on and below the diagonal (k1 <= j0), on
// MFMA: the products summed from zero and taken off once; tiles dealt to the waves
__device__ inline void take_off(double* A, const CellLds& L, int k0, int k1, int j0, int j1, int w, int nw, int lane) {
  const int q1 = (j1 + 15) >> 4, kq = lane >> 4, rl = lane & 15;
  int q = j0 >> 4, i = q + w;  // tile of rows 16 i and panel q, column by column
  while (true) {
    while (i >= L.np) {
      ++q;
      i = i - L.np + q;
      if (q >= q1) return;
    }
    if (q >= q1) return;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int p = k0 >> 4; 16 * p < k1; ++p) {
      const int ld = L.pitch(p);
      const double* X = A + L.base(p) + 16 * (i - p) + rl;
      const double* Y = A + L.base(p) + 16 * (q - p) + rl;
#pragma unroll
      for (int k4 = 0; k4 < 16; k4 += 4) {
        if (16 * p + k4 + 4 <= k0 || 16 * p + k4 >= k1) continue;  // uniform
        const int k = 16 * p + k4 + kq;
        const bool in = k >= k0 && k < k1;
        const double x = X[(k4 + kq) * ld], y = Y[(k4 + kq) * ld];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? y : 0.0, in ? x : 0.0, acc, 0, 0, 0);
      }
    }
    const int ldc = L.pitch(q);
    double* C = A + L.base(q) + kq * ldc + 16 * (i - q) + rl;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = 16 * q + kq + 4 * v;
      if (j >= j0 && j < j1) C[4 * v * ldc] -= acc[v];
    }
    i += nw;
  }
}

// Columns [c0, c1) factored in place, in blocks of up to 64 that first take the columns
// before them, summed from zero: taken off the entries panel by panel instead, every 16
// columns would cost each entry a rounding at its full size (the Schur complement of 2D
// Poisson cells, F = 27: 2.2e-16 of |K| from that of its K, and 4.1e-17 so). The columns
// from c1 on are left as they are.
template <bool IEEE>
__device__ inline void factor_in_place(double* A, const CellLds& L, int c0, int c1, int w, int nw, int lane,
                                       int& fail) {
  for (int b0 = c0; b0 < c1;) {
    const int b1 = min(c1, (b0 & ~15) + 64);
    if (b0 > c0) {
      take_off(A, L, c0, b0, b0, b1, w, nw, lane);
      __syncthreads();
    }
    for (int c = b0; c < b1;) {
      const int p = c >> 4, lo = c & 15, hi = min(16, b1 - 16 * p);
      if (lo == 0 && hi == 16) factor_panel<true, IEEE, false>(A, L, p, lo, hi, w, lane, fail);
      else factor_panel<false, IEEE, false>(A, L, p, lo, hi, w, lane, fail);
      __syncthreads();
      const int k0 = 16 * p + lo;
      c = 16 * p + hi;
      if (c < b1) {
        take_off(A, L, k0, c, c, b1, w, nw, lane);
        __syncthreads();
      }
    }
    b0 = b1;
  }
}

}  // namespace

constexpr int kCellThreads = 512;

__global__ __launch_bounds__(kCellThreads) void cell_factor_kernel(CellFactorArgs g) {
  constexpr int NT = kCellThreads;
  extern __shared__ double A[];
  const int c = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  constexpr int NW = NT / 64;
  const int N = g.N, M = g.M, F = g.F, T = M - F, D = N + M + 2;
  const CellLds L{(D + 15) / 16};
  const double* Ac = g.A + (size_t)c * g.sA;
  // sums start from zero in the columns past the first 64, and in the trailing
  // block (entries above the diagonal and rows past D are never read)
  for (int e = L.base(min(4, N >> 4)) + t; e < 128 * L.np * (L.np + 1) + 16 * L.np; e += NT) A[e] = 0.0;
  constexpr int RC = (kCellMaxD + 63) / 64, CU = 4;  // row chunks of a column; columns on their way at a time
  double sr[RC];
#pragma unroll
  for (int k = 0; k < RC; ++k) {
    const int r = 64 * k + lane;
    sr[k] = g.s && r < N ? g.s[(size_t)c * g.ss + r] : 1.0;
  }
  int fail = -1;
  // 64 columns at a time: the updates by earlier columns have by then been
  // summed from zero, and the contractions' columns are added to that sum
  // (the panel kernels' order of the same operations, so their bits)
  for (int k0 = 0; k0 < N; k0 += 64) {
    const int k1 = min(k0 + 64, N), rows = g.s ? D - 1 : D;  // with s the residual row is formed below
    __syncthreads();
    for (int j0 = k0 + CU * w; j0 < k1; j0 += CU * NW) {  // a wave per column, rows contiguous
      double v[CU][RC], sj[CU];
#pragma unroll
      for (int q = 0; q < CU; ++q) {
        const int j = min(j0 + q, k1 - 1);
        sj[q] = g.s ? g.s[(size_t)c * g.ss + j] : 1.0;
#pragma unroll
        for (int k = 0; k < RC; ++k) {
          const int r = min(64 * k + lane, rows - 1);
          v[q][k] = Ac[(size_t)max(r, j) + (size_t)j * g.lda];
        }
      }
#pragma unroll
      for (int q = 0; q < CU; ++q) {
        const int j = j0 + q;
        if (j >= k1) break;
        double* col = A + L.at(16 * (j >> 4), j) - 16 * (j >> 4);
#pragma unroll
        for (int k = 0; k < RC; ++k) {
          const int r = 64 * k + lane;
          const double x = v[q][k] * sr[k] * sj[q];  // (g s_i) s_j; B and l by s_j alone
          if (r >= j && r < rows) col[r] = k0 > 0 ? col[r] + x : x;
        }
        if (!g.s) continue;
        double res = 0.0;  // the residual row
        if (g.u) {
          const double* uc = g.u + (size_t)c * M;
          const double* a = Ac + (size_t)j * g.lda + N;
          double acc = 0.0;
          for (int m = lane; m < M; m += 64) acc = fma(uc[m], a[m] * sj[q], acc);
          for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
          res = a[M] * sj[q] - acc;
        }
        if (lane == 0) col[D - 1] = k0 > 0 ? col[D - 1] + res : res;
      }
    }
    __syncthreads();
    factor_range(A, L, k0, k1, w, NW, lane, fail);
  }
  // -[B l r]^T G^-1 [B l r] now stands in the trailing block
  if (g.factor) {
    double* Fc = g.factor + (size_t)c * g.sF;
    for (int i = w; i < N + M + 1; i += NW)
      for (int j = lane; j < N; j += 64) Fc[(size_t)i * N + j] = i >= j ? A[L.at(i, j)] : 0.0;
  }
  if (g.factor_scale)
    for (int j = t; j < N; j += NT) g.factor_scale[(size_t)c * N + j] = g.s[(size_t)c * g.ss + j];
  if (g.z)
    for (int j = t; j < N; j += NT) g.z[(size_t)c * N + j] = A[L.at(D - 1, j)];
  if (g.eta2 && t == 0) g.eta2[c] = -A[L.at(D - 1, D - 1)];
  if (g.K) {
    double* Kc = g.K + (size_t)c * M * M;
    for (int a = w; a < M; a += NW)
      for (int b = lane; b < M; b += 64) Kc[(size_t)a * M + b] = -A[L.at(N + max(a, b), N + min(a, b))];
  }
  if (g.rhs)
    for (int a = t; a < M; a += NT) g.rhs[(size_t)c * M + a] = -A[L.at(N + M, N + a)];
  if (g.schur || g.schur_rhs) {
    __syncthreads();
    // K itself, whose field columns are then eliminated. (Not equilibrated: a diagonal
    // scaling changes Cholesky's rounding only through over- and underflow, and the
    // products stay below K's own diagonal entries.)
    for (int j = N + w; j < D; j += NW)
      for (int r = j + lane; r < D; r += 64) A[L.at(r, j)] = -A[L.at(r, j)];
    __syncthreads();
    factor_in_place<true>(A, L, N, N + F, w, NW, lane, fail);
    take_off(A, L, N, N + F, N + F, D, w, NW, lane);
    __syncthreads();
    if (g.schur) {
      double* Sc = g.schur + (size_t)c * T * T;
      for (int a = w; a < T; a += NW)
        for (int b = lane; b < T; b += 64) Sc[(size_t)a * T + b] = A[L.at(N + F + max(a, b), N + F + min(a, b))];
    }
    if (g.schur_rhs)
      for (int a = t; a < T; a += NT) g.schur_rhs[(size_t)c * T + a] = A[L.at(N + M, N + F + a)];
  }
  // wave 0 owns rows of every panel
  if (t == 0) g.info[c] = fail + 1;
}

// A panel's diagonal block of larger cells: its update by the columns before it (k of
// them, on MFMA, summed from zero and then taken off), its Cholesky factor as above,
// and the factor in the forms its readers want: the 64-column diagonal blocks in Ld,
// what is below them in A, all of it with the reciprocal diagonal in Lt. One workgroup
// per cell, of 4 waves up to 64 columns, of 8 above.
// Columns from 64 on take the first 64's products into the same sums: taken off the
// entries 16 columns at a time, |L L^T - G| was 1.2 to 2 times as large.
// Bound by its chain of pivots, as cell_factor_kernel, and with many cells by the
// columns before the panel, staged through LDS (283 us for the chain of 128 columns of
// 1,612 cells, 585 us with 512 columns before them; with each wave reading its tiles'
// rows from memory the last took 1,190 us). One wave with a 64-column block in its registers took
// 38 to 55 us a panel of 60 cells, 115 us at 4,096, and its update another launch.
// NW waves, U of the block's tiles a wave
template <int NW, int U>
__global__ __launch_bounds__(64 * NW) void potrf_block(PanelArgs g, double* __restrict__ Ld, int64_t sLd,
                                                       int32_t* __restrict__ info) {
  extern __shared__ double B[];
  const int kb = g.kb, k0 = g.k0;
  const int64_t lda = g.lda;
  const int c = blockIdx.x, t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const CellLds L{(kb + 15) / 16};
  double* Ac = g.A + (size_t)c * g.sA;
  const double* sc = g.s + (size_t)c * g.ss + (k0 - g.kbeg);  // with g.s
  const int nt = L.np * (L.np + 1) / 2, kq = lane >> 4, rl = lane & 15;
  d4 acc[U];
  int ti[U], tj[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    acc[u] = d4{0.0, 0.0, 0.0, 0.0};
    int n = nt - 1 - min(w + NW * u, nt - 1), col = 0;  // the last columns' tiles first
    while (n >= L.np - col) n -= L.np - col++;
    ti[u] = __builtin_amdgcn_readfirstlane(col + n);
    tj[u] = __builtin_amdgcn_readfirstlane(col);
  }
  const int k = k0 - g.kbeg;  // whole panels: a multiple of 64
  if (k > 0) {
    // the panel's rows of KC columns at a time, two buffers in B's place
    constexpr int TR = 16 * NW, KC = 16, PT = KC / 4, LS = TR + 4;
    const int r = t % TR, kr = t / TR;
    const double* X = Ac + k0 + min(r, kb - 1) + (size_t)(g.kbeg + kr) * lda;  // rows past the block repeat its last one
    double p[PT];
    auto fetch = [&](int kc) {
#pragma unroll
      for (int i = 0; i < PT; ++i) p[i] = X[(size_t)(kc + 4 * i) * lda];
    };
    fetch(0);
    for (int kc = 0, buf = 0; kc < k; kc += KC, buf ^= 1) {
      double* S = B + buf * KC * LS;
#pragma unroll
      for (int i = 0; i < PT; ++i) S[(kr + 4 * i) * LS + r] = p[i];
      fetch(min(kc + KC, k - KC));
      __syncthreads();
#pragma unroll
      for (int k4 = 0; k4 < KC; k4 += 4) {
        const double* Sk = S + (k4 + kq) * LS + rl;
        double x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          x[u] = Sk[16 * ti[u]];
          y[u] = Sk[16 * tj[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[u], x[u], acc[u], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // the block less its sum, tile u
  auto put = [&](int u) {
    const int i = 16 * ti[u] + rl, ld = L.pitch(tj[u]);
    double* C = B + L.base(tj[u]) + 16 * (ti[u] - tj[u]) + rl;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = 16 * tj[u] + kq + 4 * v;
      double a = i >= j && i < kb ? Ac[(size_t)(k0 + i) + (size_t)(k0 + j) * lda] : 0.0;
      if (g.s) a = a * sc[min(i, kb - 1)] * sc[min(j, kb - 1)];
      C[(kq + 4 * v) * ld] = a - acc[u][v];
    }
  };
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (w + NW * u < nt && tj[u] < 4) put(u);
  __syncthreads();
  int fail = -1;
  factor_in_place<false>(B, L, 0, min(kb, 64), w, NW, lane, fail);
  if constexpr (NW > 4) {
    // columns from 64 on (at most 10 tiles: the first two of a wave): the first 64 go on
    // into the same sums
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (w + NW * u >= nt || tj[u] < 4) continue;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const double* X = B + L.base(p) + 16 * (ti[u] - p) + rl + kq * L.pitch(p);
        const double* Y = B + L.base(p) + 16 * (tj[u] - p) + rl + kq * L.pitch(p);
#pragma unroll
        for (int k4 = 0; k4 < 16; k4 += 4)
          acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(Y[k4 * L.pitch(p)], X[k4 * L.pitch(p)], acc[u], 0, 0, 0);
      }
      put(u);
    }
    __syncthreads();
    factor_in_place<false>(B, L, 64, kb, w, NW, lane, fail);
  }
  double* Lc = Ld + (size_t)c * sLd + (size_t)k0 * 64;
  double* Ltc = g.Lt + (size_t)c * g.sLt;
  const int kr = (int)((kb + 31) / 32) * 32;
  for (int j = w; j < kr; j += NW)
    for (int i = lane; i < kr; i += 64) {
      const bool in = i < kb && j < kb;
      const double v = in && i >= j ? B[L.at(i, j)] : 0.0;
      Ltc[(size_t)j * kPanelMax + i] = in && i == j ? 1.0 / v : v;
      if (!in) continue;
      if ((i ^ j) < 64) Lc[(size_t)j * 64 + (i & 63)] = v;
      else if (i > j) Ac[(size_t)(k0 + i) + (size_t)(k0 + j) * lda] = v;
    }
  if (t == 0 && fail >= 0 && info) atomicCAS(&info[c], 0, k0 + fail + 1);
}

// Field recovery after a condensed solve, u_F = K_FF^-1 (rhs_F - K_FT u_T), one
// workgroup per cell: S K_FF S (s_j = 1/sqrt(K_jj)) and s_j b_j as a row below it go to
// LDS, are factored as above, and one wave substitutes back. K is symmetric: row j
// from column j on holds both column j of K_FF and row j of K_FT.
// Bound by the two chains of F pivots: 155 us for 990 cells of F = 108, M = 258
// (two of 58 KB a compute unit); the panel kernels took 300 us in five launches.
__global__ __launch_bounds__(kCellThreads) void cell_recover_kernel(const double* __restrict__ K,
                                                                    const double* __restrict__ rhs, int M, int F,
                                                                    double* __restrict__ u, int32_t* __restrict__ info) {
  constexpr int NW = kCellThreads / 64, RC = kCellMaxD / 64;
  extern __shared__ double A[];
  __shared__ double sl[kCellMaxD];
  const int c = blockIdx.x, t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const CellLds L{F / 16 + 1};
  const double* __restrict__ Kc = K + (size_t)c * M * M;
  double* uc = u + (size_t)c * M;
  for (int j = t; j < F; j += kCellThreads) sl[j] = 1.0 / sqrt(Kc[(size_t)j * (M + 1)]);
  __syncthreads();
  for (int j = w; j < F; j += NW) {
    const double* row = Kc + (size_t)j * M;
    const double sj = sl[j];
    double k[RC], dot = 0.0;
#pragma unroll
    for (int r = 0; r < RC; ++r) k[r] = row[min(64 * r + lane, F - 1)];
    for (int q = F + lane; q < M; q += 64) dot = fma(row[q], uc[q], dot);
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const int i = 64 * r + lane;
      if (i >= j && i < F) A[L.at(i, j)] = sl[i] * sj * k[r];
    }
    for (int m = 32; m > 0; m >>= 1) dot += __shfl_xor(dot, m);
    if (lane == 0) A[L.at(F, j)] = sj * (rhs[(size_t)c * M + j] - dot);
  }
  __syncthreads();
  int fail = -1;
  factor_in_place<false>(A, L, 0, F, w, NW, lane, fail);
  if (w > 0) return;
  // L^T x = y over the rows of L from the last one, a lane an entry (one of each 64)
  double z[RC], row[RC];
  int at[RC];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    at[r] = L.at(0, min(64 * r + lane, F - 1));
    z[r] = A[at[r] + F];
    row[r] = A[at[r] + F - 1];
  }
#pragma unroll
  for (int b = RC - 1; b >= 0; --b) {
    for (int j = min(F - 1, 64 * b + 63); j >= 64 * b; --j) {
      const double zj = wave_read(z[b], j & 63) / wave_read(row[b], j & 63);
      double v[RC];
#pragma unroll
      for (int r = 0; r <= b; ++r) {
        v[r] = row[r];
        row[r] = A[at[r] + max(j - 1, 0)];
      }
#pragma unroll
      for (int r = 0; r <= b; ++r) {
        const int i = 64 * r + lane;
        z[r] = i < j ? fma(-v[r], zj, z[r]) : i == j ? zj : z[r];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RC; ++r)
    if (64 * r + lane < F) uc[64 * r + lane] = sl[64 * r + lane] * z[r];
  if (lane == 0) info[c] = fail + 1;
}

size_t cell_factor_lds_bytes(int D) {
  const size_t np = (D + 15) / 16;
  return sizeof(double) * (128 * np * (np + 1) + 16 * np);
}

// Lets a kernel have up to `most` bytes of LDS beyond the 64 KB that every kernel may have.
// The limit is an attribute of the function on the current device, for all host threads:
// always the kernel's largest size, so that no thread's small launch lowers it between
// another's setting it and launching.
static void allow_lds(const void* kernel, size_t most, const char* what) {
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
  if (e != hipSuccess) throw DeviceError(std::string(what) + ": LDS size: " + hipGetErrorString(e));
}

void launch_cell_factor(CellFactorArgs g, int ncells, hipStream_t st) {
  if (ncells <= 0) return;
  const int D = g.N + g.M + 2;
  if (D > kCellMaxD) throw DeviceError("cell_factor: the cell does not fit in LDS");
  const size_t lds = cell_factor_lds_bytes(D);
  if (lds > kMaxLds) allow_lds((const void*)cell_factor_kernel, cell_factor_lds_bytes(kCellMaxD), "cell_factor_kernel");
  cell_factor_kernel<<<ncells, kCellThreads, lds, st>>>(g);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw DeviceError(std::string("cell_factor_kernel: ") + hipGetErrorString(e));
}

void launch_cell_recover(const double* K, const double* rhs, int M, int F, double* u, int ncells, int32_t* info,
                         hipStream_t st) {
  if (ncells <= 0 || F <= 0) return;
  if (F + 1 > kCellMaxD) throw DeviceError("cell_recover: the field block does not fit in LDS");
  const size_t lds = cell_factor_lds_bytes(F + 1);
  if (lds + sizeof(double) * kCellMaxD > kMaxLds)
    allow_lds((const void*)cell_recover_kernel, cell_factor_lds_bytes(kCellMaxD), "cell_recover_kernel");
  cell_recover_kernel<<<ncells, kCellThreads, lds, st>>>(K, rhs, M, F, u, info);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw DeviceError(std::string("cell_recover_kernel: ") + hipGetErrorString(e));
}

void launch_potrf(const PanelArgs& g, double* Ld, int64_t sLd, int ncells, int32_t* info, hipStream_t st) {
  if (g.kb <= 0 || g.kb > kPanelMax || (g.k0 - g.kbeg) % 64 != 0)
    throw DeviceError("potrf_block: panel width must be 1..128");
  if (ncells <= 0) return;
  auto run = [&](auto kernel, int nw) {
    // the block, and before it two buffers of 16 of the panel's columns
    const size_t lds = std::max(cell_factor_lds_bytes(g.kb), sizeof(double) * 2 * 16 * (16 * nw + 4));
    if (lds > kMaxLds) allow_lds((const void*)kernel, cell_factor_lds_bytes(kPanelMax), "potrf_block");
    kernel<<<ncells, 64 * nw, lds, st>>>(g, Ld, sLd, info);
  };
  if (g.kb <= 64) run(potrf_block<4, 3>, 4);
  else run(potrf_block<8, 5>, 8);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw DeviceError(std::string("potrf_block: ") + hipGetErrorString(e));
}

}  // namespace dpg
