// contract.hip -- contractions of whole cells with their operands formed in place.
//
// bmat_kernel: the rows of B and the load vector of the augmented matrix, straight
// from the point weights. B[t, i] = sum_q phi_t(q) T(q, i) with the operand
// T(q, i) = sum_r W[q][g][var i][r] R[q][r][i]; a lane owns one test dof i, keeps
// up to NF trial rows t of one block in registers and runs over the points, so T
// lives in a register instead of a round trip through HBM and a block of any
// number of rows wastes no matrix-core tile. A wave's dofs belong to one test
// variable: weights and basis values are then the same for all lanes (scalar
// loads), and a block no term couples with the variable is skipped.
//
// Bound by HBM writes on many cells (4,096 Stokes cells, N = 228, M = 184: 1.4 GB
// of B in 0.83 ms, 0.36 ms of it the stores, the rest the latency of short
// tasks; the operand kernels and one GEMM per block took 2.7 ms), by latency on few (16 cells
// of 2D Poisson: 10 us against 73 us, 504 hexes of N = 365: 0.32 against 0.76 ms).
// Not taken where B is sum-factorised: the 4,096 hexes of N = 666 take 13.7 ms
// here and 7.0 ms there.
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/dpg_capi.h"
#include "kernels.hpp"

namespace dpg {

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

// rows row .. row + nf - 1 of the phase for this wave's 64 test dofs, nf <= NF
template <int NPR, int NF>
__device__ inline void bmat_rows(const BmatArgs& g, const BmatTask& k, int c, int i, int var, double* out, int pitch,
                                 int lane) {
  const bool side = k.kind == kBmatSide;
  const double* __restrict__ W = (side ? g.Wside + (size_t)c * g.nWside : g.Wvol + (size_t)c * g.nWvol) + k.w0 +
                                 var * NPR;
  const double* __restrict__ R = (side ? g.R_side : g.R_vol) + (size_t)k.point0 * NPR * g.N + i;
  const double* __restrict__ phi = (k.table == kBmatField ? g.field : k.table == kBmatTrace ? g.trace : g.flux) + k.f0;
  const int npts = k.npts, wstride = k.wstride, card = k.card, nf = k.nf, row = k.row;
  double acc[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) acc[f] = 0.0;
  // U points' basis values at a time, the next U on their way meanwhile (they
  // come from L2, several hundred cycles a load)
  constexpr int U = NPR == 3 ? 4 : 2;
  double rc[U][NPR], rn[U][NPR];
  auto fetch = [&](double (&x)[U][NPR], int q) {
#pragma unroll
    for (int v = 0; v < U; ++v) {
      const size_t o = (size_t)min(q + v, npts - 1) * NPR;
#pragma unroll
      for (int r = 0; r < NPR; ++r) x[v][r] = R[(o + r) * g.N];
    }
  };
  fetch(rn, 0);
  for (int q0 = 0; q0 < npts; q0 += 64) {
    // the weights of 64 points, one per lane, read back lane by lane below:
    // fetched point by point each would wait for memory on its own
    double wq[NPR];
    const int ql = min(q0 + lane, npts - 1), qe = min(q0 + 64, npts);
#pragma unroll
    for (int r = 0; r < NPR; ++r) wq[r] = q0 + lane < npts ? W[(size_t)ql * wstride + r] : 0.0;
    for (int q = q0; q < qe; q += U) {  // whole groups: past the last point T is zero
#pragma unroll
      for (int v = 0; v < U; ++v)
#pragma unroll
        for (int r = 0; r < NPR; ++r) rc[v][r] = rn[v][r];
      fetch(rn, q + U);
#pragma unroll
      for (int v = 0; v < U; ++v) {
        double t = 0.0;
#pragma unroll
        for (int r = 0; r < NPR; ++r) t = fma(wave_read(wq[r], q + v - q0), rc[v][r], t);
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f] = fma(phi[(q + v) * card + f], t, acc[f]);  // past nf: not used
      }
    }
  }
#pragma unroll
  for (int f = 0; f < NF; ++f)
    if (f < nf) out[lane * pitch + row + f] = acc[f];
}

// the load vector's entry of test dof i
template <int NPR>
__device__ inline double load_entry(const BmatArgs& g, const BmatTask& k, int c, int i, int var, int lane) {
  const double* __restrict__ W = g.Wrhs + (size_t)c * g.nWrhs + var * NPR;
  const int npts = k.npts, wstride = k.wstride;
  double acc = 0.0;
  for (int q0 = 0; q0 < npts; q0 += 64) {
    double wq[NPR];
    const int ql = min(q0 + lane, npts - 1), qe = min(q0 + 64, npts);
#pragma unroll
    for (int r = 0; r < NPR; ++r) wq[r] = W[(size_t)ql * wstride + r];
#pragma unroll 8
    for (int q = q0; q < qe; ++q)
#pragma unroll
      for (int r = 0; r < NPR; ++r)
        acc = fma(wave_read(wq[r], q - q0), g.R_vol[(size_t)(q * NPR + r) * g.N + i], acc);
  }
  return acc;
}

}  // namespace

// The load vector and the residual row's zeros alone, a wave per chunk of dofs
// (the paths that contract B elsewhere).
template <int NPR>
__global__ __launch_bounds__(256) void load_kernel(BmatArgs g, int nchunks) {
  const int n = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= nchunks) return;
  const BmatChunk ch = g.chunks[n];
  const BmatTask& k = g.tasks[g.phases[0].task0];
  const int c = blockIdx.y, i = ch.i0 + min(lane, ch.n - 1);
  double v = load_entry<NPR>(g, k, c, i, ch.var, lane);
  if (lane >= ch.n) return;
  if (g.s) v *= g.s[(size_t)c * g.ss + i];
  double* __restrict__ Ac = g.A + (size_t)c * g.sA + g.N + g.phases[0].row0 + (size_t)i * g.lda;
  Ac[0] = v;
  Ac[1] = 0.0;
}

// The DPOEQU factors s_i = 1 / sqrt(G_ii) of a chunk's dofs, G_ii the sum over the
// points, and over each point's IP terms, of the squared operand values: the waves
// form the values of some points at a time in LDS, the first adds them up in order.
template <int NPR>
__device__ inline void gram_factors(const BmatArgs& g, const BmatChunk& ch, int c, int w, int lane, double* V) {
  constexpr int TPG = 64 / NPR;  // terms whose weights a wave's lanes hold
  const int per = g.nvar * NPR, slice = g.n_lt * per, i = ch.i0 + min(lane, ch.n - 1);
  const double* __restrict__ W = g.Wip + (size_t)c * g.nWip + ch.var * NPR;
  const int pb = kBmatPhaseRows / g.n_lt;
  double diag = 0.0;
  for (int q0 = 0; q0 < g.QG; q0 += pb) {
    const int np = min(pb, g.QG - q0);
    for (int p = w; p < np; p += 4) {
      double r[NPR];
#pragma unroll
      for (int k = 0; k < NPR; ++k) r[k] = g.R_ip[(size_t)((q0 + p) * NPR + k) * g.N + i];
      for (int l0 = 0; l0 < g.n_lt; l0 += TPG) {
        const int m = min(TPG, g.n_lt - l0);
        const double wl = W[(size_t)(q0 + p) * slice + (l0 + min(lane / NPR, m - 1)) * per + lane % NPR];
#pragma unroll 4
        for (int l = 0; l < m; ++l) {
          double v = 0.0;
#pragma unroll
          for (int k = 0; k < NPR; ++k) v = fma(wave_read(wl, l * NPR + k), r[k], v);
          V[(p * g.n_lt + l0 + l) * 64 + lane] = v;
        }
      }
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll 8
      for (int m = 0; m < np * g.n_lt; ++m) {
        const double v = V[m * 64 + lane];
        diag = fma(v, v, diag);
      }
    }
    __syncthreads();
  }
  if (w == 0 && lane < ch.n) g.s_out[(size_t)c * g.ss + i] = 1.0 / sqrt(diag);
}

// One workgroup of 4 waves per (up to 64 dofs of a test variable, phase of up to
// 64 consecutive rows, cell): the waves take the phase's tasks in turn, the rows
// are collected in LDS and written column by column, consecutive rows together.
template <int NPR, int NFMAX>
__global__ __launch_bounds__(256) void bmat_kernel(BmatArgs g) {
  extern __shared__ double out[];
  const BmatChunk ch = g.chunks[blockIdx.x];
  const int c = blockIdx.z, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int)blockIdx.y == g.nphases) {  // one more than the phases: G's factors
    gram_factors<NPR>(g, ch, c, w, lane, out);
    return;
  }
  const BmatPhase ph = g.phases[blockIdx.y];
  const int i = ch.i0 + min(lane, ch.n - 1), var = ch.var;
  const int pitch = ph.nrows | 1;
  for (int n = w; n < ph.ntasks; n += 4) {
    const BmatTask& k = g.tasks[ph.task0 + n];
    if (k.kind == kBmatLoad) {
      // the load vector, and the residual row's zeros (with a solution its values are written later)
      out[lane * pitch + k.row] = load_entry<NPR>(g, k, c, i, var, lane);
      out[lane * pitch + k.row + 1] = 0.0;
    } else if (!((k.vars >> var) & 1u)) {
      // no term couples the block with the variable: the zeros the sums would give
      for (int f = 0; f < k.nf; ++f) out[lane * pitch + k.row + f] = 0.0;
    } else if (k.nf <= 4) {
      bmat_rows<NPR, 4>(g, k, c, i, var, out, pitch, lane);
    } else if (k.nf <= 8) {
      bmat_rows<NPR, 8>(g, k, c, i, var, out, pitch, lane);
    } else if (NFMAX == 16 || k.nf <= 16) {
      bmat_rows<NPR, 16>(g, k, c, i, var, out, pitch, lane);
    } else {
      bmat_rows<NPR, NFMAX>(g, k, c, i, var, out, pitch, lane);
    }
  }
  __syncthreads();
  if (lane >= ph.nrows) return;
  double* __restrict__ Ac = g.A + (size_t)c * g.sA + g.N + ph.row0 + lane;
  for (int j = w; j < ch.n; j += 4) {
    const double v = out[j * pitch + lane];
    Ac[(size_t)(ch.i0 + j) * g.lda] = g.s ? v * g.s[(size_t)c * g.ss + ch.i0 + j] : v;
  }
}

// ------------------------------------------------------------------- Gram matrix
// G = sum over points and IP terms of (operand row)^T (operand row) for a cell, on
// MFMA, the operand rows formed in LDS; one workgroup of 4 waves per cell, a wave
// holding up to kGramTiles of the lower triangle's 16 x 16 tiles from the first point to
// the last. Per step (the KC >= QG points of one IP term) every thread forms its share of
// the operand from basis values it holds in registers and weights staged in LDS,
// then every wave takes its tiles that the term reaches. Terms that are the same
// on a tile's variables enter once with weight 2. Stores the lower triangle
// unscaled (and both triangles if G is an output).
// Bound by the latency of its steps: N = 65, 25 points and 6 terms take 16 us at 16
// cells and 18 us at 256 (the operand kernel and the GEMM it replaces 40 and 51 us),
// 134 us at 4,096 (353 us, most of them writing and reading 580 MB of operand). The
// DPOEQU factors, a chain over points and terms, are left to a workgroup of
// bmat_kernel's launch (formed here they took 12 us more).
template <int NPR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gram_cell_kernel(GramArgs g) {
  constexpr int NT = 256, NW = 4, E = kGramEntries, U = kGramTiles;
  extern __shared__ double lds[];
  const int c = blockIdx.x, t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int N = g.N, nt = (N + 15) / 16, ntiles = nt * (nt + 1) / 2, pitch = gram_pitch(N), KC = g.kc;
  const int per = g.nvar * NPR, slice = g.n_lt * per;
  double* X = lds;                    // two buffers of KC rows
  double* Wl = lds + 2 * KC * pitch;  // KC points' weights
  const double* __restrict__ W = g.Wip + (size_t)c * g.nWip;
  d4 acc[U];
  int ti[U], tj[U];  // this wave's tiles (uniform), column by column of the lower triangle
#pragma unroll
  for (int u = 0; u < U; ++u) {
    acc[u] = d4{0.0, 0.0, 0.0, 0.0};
    int n = min(w + NW * u, ntiles - 1), col = 0;
    while (n >= nt - col) n -= nt - col++;
    ti[u] = __builtin_amdgcn_readfirstlane(col + n);
    tj[u] = __builtin_amdgcn_readfirstlane(col);
  }
  // term lt's words in lane lt: this wave's tiles it reaches, those it enters twice
  const int lw = min(lane, g.n_lt - 1);
  const uint32_t actw = g.active[lw * NW + w], twow = g.twice[lw * NW + w];
  // this thread's entries (point kk, dof j) of a step: LDS place and weights' place.
  // (Threads left over write a padding column of the last row, which nothing reads.)
  int xo[E], wo[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int n = t + NT * e, kk = n / N, j = n - kk * N;
    const bool in = kk < KC;
    xo[e] = in ? kk * pitch + j : KC * pitch - 1;
    wo[e] = (in ? kk : 0) * slice + g.var_of_dof[in ? j : 0] * NPR;
  }
  // columns past the last dof stay zero
  for (int e = t; e < 2 * KC * (pitch - N); e += NT) X[(e / (pitch - N)) * pitch + N + e % (pitch - N)] = 0.0;
  int buf = 0;
  const int rl = lane & 15, kq = lane >> 4;
  double r[E][NPR];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int n = t + NT * e, kk = n / N, j = n - kk * N;
    const bool in = kk < g.QG;
    const double* R = g.R + (size_t)(in ? kk : 0) * NPR * N + (in ? j : 0);
#pragma unroll
    for (int k = 0; k < NPR; ++k) r[e][k] = in ? R[(size_t)k * N] : 0.0;
  }
  for (int e = t; e < KC * slice; e += NT) Wl[e] = e < g.QG * slice ? W[e] : 0.0;
  __syncthreads();
  for (int lt = 0; lt < g.n_lt; ++lt) {
    double* Xb = X + buf * KC * pitch;
    double v[E];  // the weights of variables the term does not reach are zeros
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const double* wp = Wl + wo[e] + lt * per;
      v[e] = 0.0;
#pragma unroll
      for (int k = 0; k < NPR; ++k) v[e] = fma(wp[k], r[e][k], v[e]);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) Xb[xo[e]] = v[e];
    __syncthreads();
    const uint32_t act = __builtin_amdgcn_readlane(actw, lt), two = __builtin_amdgcn_readlane(twow, lt);
    if (act) {
      const double* Xr = Xb + kq * pitch + rl;
      double x[U], y[U];
      auto fetch = [&](int k4) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          x[u] = Xr[k4 * pitch + 16 * ti[u]];
          y[u] = Xr[k4 * pitch + 16 * tj[u]];
        }
      };
      fetch(0);
      for (int k4 = 0; k4 < KC; k4 += 4) {
        double xc[U], yc[U];  // the next rows' entries are fetched while these are multiplied
#pragma unroll
        for (int u = 0; u < U; ++u) {
          xc[u] = (two >> u) & 1u ? 2.0 * x[u] : x[u];
          yc[u] = y[u];
        }
        fetch(min(k4 + 4, KC - 4));
#pragma unroll
        for (int u = 0; u < U; ++u)
          if ((act >> u) & 1u)  // uniform
            acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(yc[u], xc[u], acc[u], 0, 0, 0);
      }
    }
    buf ^= 1;
  }
  double* __restrict__ Ac = g.A + (size_t)c * g.sA;
  double* __restrict__ Gc = g.G ? g.G + (size_t)c * N * N : nullptr;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (w + NW * u >= ntiles) continue;
    const int i = 16 * ti[u] + rl;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = 16 * tj[u] + kq + 4 * v;
      if (i < j || i >= N) continue;
      Ac[(size_t)i + (size_t)j * g.lda] = acc[u][v];
      if (Gc) {
        Gc[(size_t)j * N + i] = acc[u][v];
        Gc[(size_t)i * N + j] = acc[u][v];
      }
    }
  }
}

static void check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw DeviceError(std::string(what) + ": " + hipGetErrorString(e));
}

void launch_bmat(int dim, const BmatArgs& g, int nchunks, int ncells, hipStream_t st) {
  if (ncells <= 0) return;
  const dim3 grid(nchunks, g.nphases + (g.s_out ? 1 : 0), ncells);
  const size_t lds = sizeof(double) * 64 * (kBmatPhaseRows + 1);
  if (dim == 2) bmat_kernel<3, 16><<<grid, 256, lds, st>>>(g);
  else bmat_kernel<4, 32><<<grid, 256, lds, st>>>(g);
  check("bmat_kernel");
}

void launch_load(int dim, const BmatArgs& g, int nchunks, int ncells, hipStream_t st) {
  if (ncells <= 0) return;
  const dim3 grid((nchunks + 3) / 4, ncells);
  if (dim == 2) load_kernel<3><<<grid, 256, 0, st>>>(g, nchunks);
  else load_kernel<4><<<grid, 256, 0, st>>>(g, nchunks);
  check("load_kernel");
}

void launch_gram(int dim, const GramArgs& g, int ncells, hipStream_t st) {
  if (ncells <= 0) return;
  const size_t lds = gram_lds_bytes(g.N, g.kc, g.n_lt * g.nvar * (dim + 1));
  if (g.N > kGramMaxN || g.kc * g.N > 256 * kGramEntries || lds > kMaxLds) throw DeviceError("gram_cell: size");
  if (dim == 2) gram_cell_kernel<3><<<ncells, 256, lds, st>>>(g);
  else gram_cell_kernel<4><<<ncells, 256, lds, st>>>(g);
  check("gram_cell_kernel");
}

}  // namespace dpg
