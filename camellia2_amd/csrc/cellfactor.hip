// cellfactor.hip -- the factorisation of small cells in LDS.
//
// cell_factor_kernel takes the augmented matrices of cells whose whole lower
// triangle fits a compute unit's LDS (D = N + M + 2 <= kCellMaxD) from their
// contractions to every output in one launch: partial Cholesky over the N test
// columns, K, rhs, eta2 and the kept factor, then the partial Cholesky of K
// over the F field columns and the Schur complement. What the panel kernels do
// in 4 launches per 64 columns, each re-reading the matrix from HBM.
//
// What bounds it is the chain of pivots: D of them, each a square root, a
// divide and a broadcast after the one before (58 us for the 92 of the 2D
// Poisson cells of N = 65, M = 55, at 16 and at 256 cells; the 14 launches it
// replaces took 172 us there, and at 4,096 cells 870 us against 610 us, 2 cells
// per compute unit). 16-column panels keep a panel's rows in registers and
// leave the rest to rank-16 MFMA updates.
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/dpg_capi.h"
#include "kernels.hpp"

namespace dpg {

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

__device__ inline double lane_read(double v, int k) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), k);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

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

// Columns [lo, hi) of panel p: factored in registers by every wave that owns
// rows of it (a lane holds one row's 16 columns, y; every wave also holds the
// 16 rows of the diagonal block, a, in each group of 16 lanes, so the pivots
// and columns of L come from its own lanes and no wave waits for another). The
// panel's later columns are updated along with it. Entries above the diagonal
// take part with values nothing reads.
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
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    if (j < lo || j >= hi) continue;  // uniform
    double d = lane_read(a[j], j);
    const bool bad = !(d > 0.0);
    if (bad && fail < 0) fail = 16 * p + j;
    d = bad ? __builtin_nan("") : d;
    const double sd = sqrt(d), rs = 1.0 / sd;
    a[j] *= rs;
    y[j] = r == j ? sd : y[j] * rs;
#pragma unroll
    for (int k = j + 1; k < 16; ++k) {
      const double lk = lane_read(a[j], k);
      a[k] = fma(-a[j], lk, a[k]);
      y[k] = fma(-y[j], lk, y[k]);
    }
  }
  if (r < h) {
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k >= lo && r >= k) P[k * ld + r] = y[k];
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
    factor_panel(A, L, p, lo, hi, w, lane, fail);
    __syncthreads();
    update_trailing(A, L, p, lo, hi, w, nw, lane);
    __syncthreads();
    c = 16 * p + hi;
  }
}

}  // namespace

template <int NT>
__global__ __launch_bounds__(NT) void cell_factor_kernel(CellFactorArgs g) {
  extern __shared__ double A[];
  const int c = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  constexpr int NW = NT / 64;
  const int N = g.N, M = g.M, F = g.F, T = M - F, D = N + M + 2;
  const CellLds L{(D + 15) / 16};
  const double* Ac = g.A + (size_t)c * g.sA;
  for (int e = t; e < 128 * L.np * (L.np + 1) + 16 * L.np; e += NT) A[e] = 0.0;
  int fail = -1;
  // 64 columns at a time: the updates by earlier columns have by then been
  // summed from zero, and the contractions' columns are added to that sum
  // (the panel kernels' order of the same operations, so their bits)
  for (int k0 = 0; k0 < N; k0 += 64) {
    const int k1 = min(k0 + 64, N);
    __syncthreads();
    for (int j = k0 + w; j < k1; j += NW) {  // a wave per column, rows contiguous
      double* col = A + L.at(16 * (j >> 4), j) - 16 * (j >> 4);
      const double* a = Ac + (size_t)j * g.lda;
      if (!g.s) {
        for (int r = j + lane; r < D; r += 64) col[r] += a[r];
        continue;
      }
      const double* sc = g.s + (size_t)c * g.ss;
      const double sj = sc[j];
      for (int r = j + lane; r < D - 1; r += 64) col[r] += r < N ? a[r] * sc[r] * sj : a[r] * sj;
      if (g.u) {  // the residual row
        const double* uc = g.u + (size_t)c * M;
        double acc = 0.0;
        for (int m = lane; m < M; m += 64) acc = fma(uc[m], a[N + m] * sj, acc);
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
        if (lane == 0) col[D - 1] += a[N + M] * sj - acc;
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
    // K itself, whose field columns are then eliminated. (Not equilibrated:
    // Cholesky's rounding error does not depend on a diagonal scaling.)
    for (int j = N + w; j < D; j += NW)
      for (int r = j + lane; r < D; r += 64) A[L.at(r, j)] = -A[L.at(r, j)];
    __syncthreads();
    factor_range(A, L, N, N + F, w, NW, lane, fail);
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

size_t cell_factor_lds_bytes(int D) {
  const size_t np = (D + 15) / 16;
  return sizeof(double) * (128 * np * (np + 1) + 16 * np);
}

void launch_cell_factor(CellFactorArgs g, int ncells, hipStream_t st) {
  if (ncells <= 0) return;
  const int D = g.N + g.M + 2;
  if (D > kCellMaxD) throw DeviceError("cell_factor: the cell does not fit in LDS");
  const size_t lds = cell_factor_lds_bytes(D);
  // up to 80 KB (D <= 128) two workgroups share a compute unit and hide each
  // other's pivot chains; above, one workgroup of twice the waves
  auto run = [&](auto kernel, int nt) {
    // more than the 64 KB every kernel may have (an attribute of the function on the current device)
    if (lds > kMaxLds && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds) != hipSuccess)
      throw DeviceError("cell_factor: LDS size");
    kernel<<<ncells, nt, lds, st>>>(g);
  };
  if (lds <= 80 * 1024) run(cell_factor_kernel<256>, 256);
  else run(cell_factor_kernel<512>, 512);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw DeviceError(std::string("cell_factor_kernel: ") + hipGetErrorString(e));
}

}  // namespace dpg
