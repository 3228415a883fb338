// gfx950 FP64 IRLS of one gene per workgroup: every iteration of a gene
// (src/beta.cpp:25-51) runs in one launch.
//
// The round kernels (kernels_tile.hip) take four launches per iteration of
// the whole problem.  Where a round's work is microseconds the launches are
// the time: 2000 genes x 5000 cells, p = 2, ran 123 rounds of 36 us (4.4 ms)
// for 85 us of arithmetic, and runs 0.66 ms here; 64 genes x 2000 cells 71
// rounds, 3.2 ms, and 0.16 ms here.  A workgroup keeps a gene until it stops:
// its threads stride over the cells (lane = cell, so counts and the columns of X are read
// coalesced, in the caller's layout), each lane sums r x_a x_b in registers,
// a reduce-scatter over the lanes and an LDS sum over the wavefronts give the
// p x p system, one wavefront solves it and the next iteration starts.  Genes
// that stop early make room for the next ones; nothing returns to the host.
//
// FP64 issue bounds it (p + 25 + p (p + 1) / 2 + p instructions per cell
// and lane); against the tile kernel it pads no columns to 16 and no features
// to 4.  X and the offsets are read once per gene and iteration, from the
// XCD's L2, which is why the caller takes this path only where they fit there
// (launch_irls_gene's callers hold the rule).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/devil_hip.h"
#include "device_common.hpp"
#include "kernels.hpp"
#include "tile_common.hpp"

namespace dv {

// Lane sums of V values: after reduce_scatter the lane with index parts
// scatter_index holds the wave's sum of value scatter_index + i in v[i],
// i < scatter_left(V).  Each step halves the values a lane holds and pairs
// lanes 32, 16, 8, 4, 2, 1 apart, so the 64-lane sums of V values take about
// V exchanges instead of 6 V.
__host__ __device__ constexpr int scatter_left(int V) {
  for (int i = 0; i < 6; ++i) V = (V + 1) / 2;
  return V;
}

template <int M, int MASK>
__device__ __forceinline__ void scatter_step(double* v, int lane) {
  constexpr int H = (M + 1) / 2;
  const bool up = lane & MASK;
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const double lo = v[i], hi = H + i < M ? v[H + i] : 0.0;
    const double keep = up ? hi : lo, send = up ? lo : hi;
    v[i] = keep + __shfl_xor(send, MASK, 64);
  }
  if constexpr (MASK > 1) scatter_step<H, MASK / 2>(v, lane);
}

// first value index of this lane's sums; *valid[i] false where the lane's
// i-th entry stands for no value
template <int V>
__device__ __forceinline__ int scatter_index(int lane, int i) {
  int m[6], v = V;
  for (int k = 0; k < 6; ++k) {
    m[k] = v;
    v = (v + 1) / 2;
  }
  int pos = i;
  for (int k = 5; k >= 0; --k) {
    const int half = (m[k] + 1) / 2;
    if (lane & (32 >> k)) {
      pos += half;
      if (pos >= m[k]) return -1;
    }
  }
  return pos;
}

template <int P, typename CT>
struct GeneOps {
  CT y;
  double x[P];
  double off;
};

constexpr int kGeneMaxWaves = 8;

// ICPT: column 0 of X is all ones (no loads and products for it, and the
// pairs (0, b) are the gradient).
template <int P, bool ICPT, typename CT>
__device__ __forceinline__ void irls_gene(const GeneDesign& gd, const CT* __restrict__ yrow,
                                          int g, double k, double* __restrict__ beta,
                                          int max_iter, double eps, int32_t* __restrict__ iters,
                                          int32_t* __restrict__ status, const double* e2,
                                          double* part, double* tot, double* bsh, int* flag) {
  constexpr int NP = P * (P + 1) / 2;
  constexpr int NV = ICPT ? NP : NP + P;
  constexpr int J0 = ICPT ? 1 : 0;
  constexpr int NL = scatter_left(NV);
  const int tid = threadIdx.x, T = blockDim.x, lane = tid & 63;
  const int wave = wave_index(), nw = T >> 6;
  const int64_t n = gd.n;
  int where[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) where[i] = scatter_index<NV>(lane, i);
  int it = 0, st = 0;
  for (;;) {
    double b[P];
#pragma unroll
    for (int j = 0; j < P; ++j) b[j] = uniform_f64(bsh[j]);
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] = 0.0;
    typedef GeneOps<P, CT> Ops;
    auto load = [&](int64_t step, Ops& o) {
      const int64_t i = min(step * T + tid, n - 1);
#pragma unroll
      for (int j = J0; j < P; ++j) o.x[j] = gd.X[i + j * n];
      o.off = gd.off[i];
      o.y = yrow[i];
    };
    // the element arithmetic of the tile kernel: w = exp(-x'b - off),
    // r = m w - 1 = (y w - 1) / (1 + k w)
    auto body = [&](const Ops& o, bool in) {
      double eta = -o.off;
      if constexpr (ICPT) eta -= b[0];
#pragma unroll
      for (int j = J0; j < P; ++j) eta = fma(-b[j], o.x[j], eta);
      const double w = exp_tab(eta, e2);
      const double d = fma(k, w, 1.0);
      double r = fma((double)o.y, w, -1.0) * rcp1_f64(d);
      r = in ? r : 0.0;
      int q = 0;
#pragma unroll
      for (int a = 0; a < P; ++a) {
        const double rx = ICPT && a == 0 ? r : r * o.x[a];
#pragma unroll
        for (int bb = a; bb < P; ++bb) {
          if (ICPT && bb == 0) acc[q] += rx;
          else acc[q] = fma(rx, o.x[bb], acc[q]);
          ++q;
        }
      }
      if constexpr (!ICPT) {
#pragma unroll
        for (int a = 0; a < P; ++a) acc[NP + a] = fma(r, o.x[a], acc[NP + a]);
      }
    };
    const int64_t full = n / T, steps = (n + T - 1) / T;
    {
      Ops A, B;
      load(0, A);
      for (int64_t s = 0; s < full; s += 2) {
        load(min(s + 1, steps - 1), B);
        body(A, true);
        if (s + 1 >= full) break;
        load(min(s + 2, steps - 1), A);
        body(B, true);
      }
      if (full < steps) {  // the last cells, one per lane at most
        if (full & 1) body(B, full * T + tid < n);
        else body(A, full * T + tid < n);
      }
    }
    scatter_step<NV, 32>(acc, lane);
#pragma unroll
    for (int i = 0; i < NL; ++i)
      if (where[i] >= 0) part[wave * NV + where[i]] = acc[i];
    __syncthreads();
    if (wave == 0) {
      for (int q = lane; q < NV; q += 64) {
        double s = 0.0;
        for (int u = 0; u < nw; ++u) s += part[u * NV + q];
        tot[q] = s;
      }
      __builtin_amdgcn_wave_barrier();
      // A = k (X'diag(r)X + X'X), g = k X'r (k_irls_update's system)
      double M[P][P], v[P];
#pragma unroll
      for (int a = 0; a < P; ++a) {
        const double ga = tot[ICPT ? a : NP + a];
        v[a] = k * (gd.kidx_lin[a] >= 0 ? ga : 0.0);
#pragma unroll
        for (int bb = a; bb < P; ++bb) {
          const int q = tri<P>(a, bb);
          const int pi = gd.kidx_pair[q];
          const double e = k * (pi >= 0 ? tot[q] + gd.ksum[pi] : 0.0);
          M[a][bb] = e;
          M[bb][a] = e;
        }
      }
      int perm[P];
      if (lu_factor<P>(M, perm)) st |= DEVIL_GENE_SINGULAR;
      lu_solve<P>(M, perm, v);
      double mx = 0.0;
      bool has_nan = false;
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const double d = fabs(v[j]);
        if (isnan(d)) has_nan = true;
        else mx = fmax(mx, d);
      }
      bool conv = !has_nan && mx < eps;
      ++it;
      if (isnan(v[0])) {
        conv = true;
        st |= DEVIL_GENE_NAN;
      }
      if (!conv && it >= max_iter) st |= DEVIL_GENE_MAXITER;
      const bool stop = conv || it >= max_iter;
      if (lane == 0) {
#pragma unroll
        for (int j = 0; j < P; ++j) bsh[j] += v[j];
        *flag = stop;
        if (stop) {
#pragma unroll
          for (int j = 0; j < P; ++j) beta[(int64_t)g * P + j] = bsh[j];
          iters[g] = it;
          status[g] = st;
        }
      }
    }
    __syncthreads();
    if (*flag) return;
  }
}

template <int P, bool ICPT>
__global__ __launch_bounds__(64 * kGeneMaxWaves) void k_irls_gene(
    GeneDesign gd, Counts c, const int32_t* __restrict__ list, double* __restrict__ beta,
    const double* __restrict__ kvec, int max_iter, double eps, int32_t* __restrict__ iters,
    int32_t* __restrict__ status) {
  constexpr int NV = P * (P + 1) / 2 + (ICPT ? 0 : P);
  __shared__ double e2[64];
  __shared__ double part[kGeneMaxWaves * NV];
  __shared__ double tot[NV];
  __shared__ double bsh[P];
  __shared__ int flag;
  const int g = list ? list[blockIdx.x] : (int)blockIdx.x;
  exp_tab_fill(e2, threadIdx.x, blockDim.x);
  if (threadIdx.x < P) bsh[threadIdx.x] = beta[(int64_t)g * P + threadIdx.x];
  __syncthreads();
  const double k = uniform_f64(kvec[g]);
  auto run = [&](auto* Y) {
    irls_gene<P, ICPT>(gd, Y + (int64_t)g * c.ld, g, k, beta, max_iter, eps, iters, status, e2,
                       part, tot, bsh, &flag);
  };
  if (c.dtype == 0) run(static_cast<const int32_t*>(c.ptr));
  else if (c.dtype == 1) run(static_cast<const float*>(c.ptr));
  else run(static_cast<const double*>(c.ptr));
}

template <int P>
hipError_t launch_gene_p(hipStream_t s, const GeneDesign& gd, Counts c, const int32_t* list,
                         int ngenes, double* beta, const double* kvec, int max_iter, double eps,
                         int32_t* iters, int32_t* status) {
  // Four wavefronts fill a CU's SIMDs once and leave room for other genes'
  // workgroups beside them (their solves overlap this one's cells); long rows
  // take eight, which shortens the last genes' iterations.
  const int T = gd.n <= 16384 ? 256 : 512;
  if (gd.intercept)
    hipLaunchKernelGGL((k_irls_gene<P, true>), dim3((unsigned)ngenes), dim3(T), 0, s, gd, c,
                       list, beta, kvec, max_iter, eps, iters, status);
  else
    hipLaunchKernelGGL((k_irls_gene<P, false>), dim3((unsigned)ngenes), dim3(T), 0, s, gd, c,
                       list, beta, kvec, max_iter, eps, iters, status);
  return hipGetLastError();
}

hipError_t launch_irls_gene(hipStream_t s, const GeneDesign& gd, Counts c, int p,
                            const int32_t* list, int ngenes, double* beta, const double* kvec,
                            int max_iter, double eps, int32_t* iters, int32_t* status) {
  if (ngenes <= 0) return hipSuccess;
  if (max_iter <= 0) return hipErrorInvalidValue;
#define DV_GENE_P(P_) \
  case P_: \
    return launch_gene_p<P_>(s, gd, c, list, ngenes, beta, kvec, max_iter, eps, iters, status);
  switch (p) {
    DV_GENE_P(1)
    DV_GENE_P(2)
    DV_GENE_P(3)
    DV_GENE_P(4)
    DV_GENE_P(5)
    DV_GENE_P(6)
    DV_GENE_P(7)
    DV_GENE_P(8)
    DV_GENE_P(9)
    DV_GENE_P(10)
    default: return hipErrorInvalidValue;
  }
#undef DV_GENE_P
}

}  // namespace dv
