// gfx950 FP64 IRLS accumulate for the last genes of a fit whose rows are too
// long for the gene kernel: a wavefront owns one gene and one chunk of cells,
// lane = cell.
//
// The tile kernel's wavefronts own 16 genes; with few genes left most of
// their lanes compute nothing, and a round of 10 genes x 500000 cells costs
// what 64 genes do.  Here the counts, X and the offsets are read coalesced in
// the caller's layout, the sums of a chunk stay in registers and end in one
// reduce-scatter.  The four wavefronts of a workgroup take four genes over the
// same cells (X once from L2), and chunks are dealt to the XCDs as in the tile
// kernel (X once from HBM).  Issue-bound at p + 23 + p (p + 1) / 2 + p vector
// instructions per cell and lane where the rows fill the GPU, latency-bound
// below.  40 genes x 500000 cells, p = 8: 39 rounds, 6.9 ms in the tile
// kernel, 1.4 ms here.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/devil_hip.h"
#include "device_common.hpp"
#include "kernels.hpp"
#include "lane_sums.hpp"
#include "tile_common.hpp"

namespace dv {

// r x_a x_b of one cell added to the sums (a <= b; with an intercept the pairs
// (0, b) are the gradient, else it follows them).
template <int P, bool ICPT, typename X>
__device__ __forceinline__ void add_products(double r, X&& x, double* acc) {
  int q = 0;
#pragma unroll
  for (int a = 0; a < P; ++a) {
    const double rx = ICPT && a == 0 ? r : r * x(a);
#pragma unroll
    for (int b = a; b < P; ++b) {
      if (ICPT && b == 0) acc[q] += rx;
      else acc[q] = fma(rx, x(b), acc[q]);
      ++q;
    }
  }
}

constexpr int kCellsWaves = 4;

// One gene, one chunk, a cell per lane; X and off in the caller's layout.
template <int P, bool ICPT, typename CT>
__device__ __forceinline__ void irls_cells(const TileDesign& td, const CT* __restrict__ Y,
                                           int64_t ld, const double* __restrict__ X,
                                           const double* __restrict__ off, int slot, int g,
                                           const double* __restrict__ beta,
                                           const double* __restrict__ kvec, int chunk,
                                           double* __restrict__ part, const double* e2) {
  constexpr int NP = P * (P + 1) / 2;
  constexpr int NV = ICPT ? NP : NP + P;
  constexpr int J0 = ICPT ? 1 : 0;
  const int lane = threadIdx.x & 63;
  double b[P];
#pragma unroll
  for (int j = 0; j < P; ++j) b[j] = uniform_f64(-beta[(int64_t)g * P + j]);
  const double k = uniform_f64(kvec[g]);
  double acc[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) acc[q] = 0.0;
  const int64_t c0 = min((int64_t)chunk * td.chunk_blocks * 16, td.n);
  const int64_t c1 = min((int64_t)(chunk + 1) * td.chunk_blocks * 16, td.n);
  const int len = (int)(c1 - c0);  // a chunk is far below 2^31 cells
  if (len > 0) {
    const CT* y0 = Y + (int64_t)g * ld + c0;
    const double* o0 = off + c0;
    const double* x0[P];
#pragma unroll
    for (int j = 0; j < P; ++j) x0[j] = X + (int64_t)j * td.n + c0;
    struct Ops {
      CT y;
      double off, x[P];
    };
    auto load = [&](int i, Ops& o) {
      const uint32_t at = (uint32_t)min(i, len - 1);
      o.y = y0[at];
      o.off = o0[at];
#pragma unroll
      for (int j = J0; j < P; ++j) o.x[j] = x0[j][at];
    };
    auto body = [&](const Ops& o, bool in) {
      double eta = -o.off;
      if constexpr (ICPT) eta += b[0];
#pragma unroll
      for (int j = J0; j < P; ++j) eta = fma(b[j], o.x[j], eta);
      const double w = exp_tab(eta, e2);
      const double d = fma(k, w, 1.0);
      double r = fma((double)o.y, w, -1.0) * rcp1_f64(d);
      r = in ? r : 0.0;
      add_products<P, ICPT>(r, [&](int j) { return o.x[j]; }, acc);
      if constexpr (!ICPT) {
#pragma unroll
        for (int a = 0; a < P; ++a) acc[NP + a] = fma(r, o.x[a], acc[NP + a]);
      }
    };
    Ops A, B;
    load(lane, A);
    for (int i = 0; i < len; i += 128) {
      load(i + 64 + lane, B);
      body(A, i + lane < len);
      load(i + 128 + lane, A);
      body(B, i + 64 + lane < len);
    }
  }
  scatter_step<NV, 32>(acc, lane);
  double* out = part + (((int64_t)(slot >> 4) * td.nchunk + chunk) * 16 + (slot & 15)) * td.ncp;
#pragma unroll
  for (int i = 0; i < scatter_left(NV); ++i) {
    const int q = scatter_index<NV>(lane, i);
    if (q < 0) continue;
    // equal columns share a place: their first sum is the one stored
    if (q < NP ? (td.own_pair >> q) & 1 : (td.own_lin >> (q - NP)) & 1)
      out[q < NP ? td.kidx_pair[q] : td.kidx_lin[q - NP]] = acc[i];
  }
}

template <int P, bool ICPT>
__global__ __launch_bounds__(64 * kCellsWaves) void k_irls_cells(
    TileDesign td, Counts c, const double* __restrict__ X, const double* __restrict__ off,
    const int32_t* __restrict__ active, const int32_t* __restrict__ nactive,
    const double* __restrict__ beta, const double* __restrict__ kvec,
    double* __restrict__ part) {
  __shared__ double e2[kExpTab];
  exp_tab_fill(e2, threadIdx.x, blockDim.x);
  __syncthreads();
  const int nA = *nactive;
  int chunk, wg;
  tile_coords(td.nchunk, chunk, wg);
  const int slot = wg * kCellsWaves + wave_index();
  if (slot >= nA) return;
  const int g = __builtin_amdgcn_readfirstlane(active[slot]);
  auto run = [&](auto* Y) {
    irls_cells<P, ICPT>(td, Y, c.ld, X, off, slot, g, beta, kvec, chunk, part, e2);
  };
  if (c.dtype == 0) run(static_cast<const int32_t*>(c.ptr));
  else if (c.dtype == 1) run(static_cast<const float*>(c.ptr));
  else run(static_cast<const double*>(c.ptr));
}

#define DV_CELLS_P(P_, KERNEL, ICPT, GRID, S, ...)                                            \
  case P_:                                                                                    \
    if (ICPT)                                                                                 \
      hipLaunchKernelGGL((KERNEL<P_, true>), GRID, dim3(64 * kCellsWaves), 0, S, __VA_ARGS__); \
    else                                                                                      \
      hipLaunchKernelGGL((KERNEL<P_, false>), GRID, dim3(64 * kCellsWaves), 0, S, __VA_ARGS__); \
    return hipGetLastError();
#define DV_CELLS(P_, KERNEL, ICPT, GRID, S, ...)              \
  switch (P_) {                                               \
    DV_CELLS_P(1, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(2, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(3, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(4, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(5, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(6, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(7, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(8, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(9, KERNEL, ICPT, GRID, S, __VA_ARGS__)         \
    DV_CELLS_P(10, KERNEL, ICPT, GRID, S, __VA_ARGS__)        \
    default: return hipErrorInvalidValue;                     \
  }

hipError_t launch_irls_cells(hipStream_t s, const TileDesign& td, Counts c, int p, int intercept,
                             const double* X, const double* off, const int32_t* active,
                             const int32_t* nactive, int nA_bound, const double* beta,
                             const double* kvec, double* part) {
  if (nA_bound <= 0) return hipSuccess;
  const int64_t wgs = (nA_bound + kCellsWaves - 1) / kCellsWaves;
  const dim3 grid((unsigned)(wgs * td.nchunk));
  DV_CELLS(p, k_irls_cells, intercept, grid, s, td, c, X, off, active, nactive, beta, kvec, part)
}

}  // namespace dv
