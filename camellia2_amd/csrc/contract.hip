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

namespace {

__device__ inline double lane_read(double v, int k) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), k);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

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
        for (int r = 0; r < NPR; ++r) t = fma(lane_read(wq[r], q + v - q0), rc[v][r], t);
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
        acc = fma(lane_read(wq[r], q - q0), g.R_vol[(size_t)(q * NPR + r) * g.N + i], acc);
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

// One workgroup of 4 waves per (up to 64 dofs of a test variable, phase of up to
// 64 consecutive rows, cell): the waves take the phase's tasks in turn, the rows
// are collected in LDS and written column by column, consecutive rows together.
template <int NPR, int NFMAX>
__global__ __launch_bounds__(256) void bmat_kernel(BmatArgs g) {
  extern __shared__ double out[];
  const BmatPhase ph = g.phases[blockIdx.y];
  const BmatChunk ch = g.chunks[blockIdx.x];
  const int c = blockIdx.z, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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

static void check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw DeviceError(std::string(what) + ": " + hipGetErrorString(e));
}

void launch_bmat(int dim, const BmatArgs& g, int nchunks, int nphases, int ncells, hipStream_t st) {
  if (ncells <= 0) return;
  const dim3 grid(nchunks, nphases, ncells);
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

}  // namespace dpg
