// gfx950 FP64 IRLS of one gene per workgroup: every iteration of a gene
// (src/beta.cpp:25-51) runs in one launch.
//
// The round kernels (kernels_tile.hip) take four launches per iteration of
// the whole problem.  Where a round's work is microseconds the launches are
// the time: 2000 genes x 5000 cells, p = 2, ran 123 rounds of 36 us (4.4 ms)
// for 85 us of arithmetic, and runs 0.55 ms here; 64 genes x 2000 cells 71
// rounds, 3.2 ms, and 0.16 ms here.  A workgroup keeps a gene until it stops:
// its threads stride over the cells (lane = cell, so counts and the columns
// of X are read coalesced, in the caller's layout), each lane sums r x_a x_b
// in registers, a reduce-scatter over the lanes and an LDS sum over the
// wavefronts give the p x p system, one wavefront solves it and the next
// iteration starts.  A gene that stops makes room for the next one, taken
// from a counter; nothing returns to the host.
//
// While all workgroups have genes, FP64 issue bounds it: 48 vector instructions
// per cell and lane for p = 4 (SQ_INSTS_VALU), about p + 22 + p (p + 1) / 2 + p
// and the loop around them; at the end the iterations of the genes that stop
// last, one workgroup's pass each.  4000 genes x 20000 cells, p = 4 (103347 gene
// iterations, the longest 148): 2.5 ms of vector issue at 2.4 GHz (3.4 at the
// rate a loop of FP64 multiply-adds reaches) in a 5.4 ms kernel.  The longest
// gene alone takes 1.94 ms (13.1 us an iteration), the 100 genes with more than
// 74 iterations 1.96, the other 3900 3.4; handed out longest first all take
// 3.7, so the rest is long genes that started late.  2000 x 5000, p = 2: 0.55
// ms, the longest gene alone 0.47 (123 iterations of 3.8 us).  Against the tile
// kernel it pads no columns to 16 and no features to 4: 4000 x 20000, p = 4,
// round kernels 7.9 ms, here 5.4; 1500 x 30001, p = 5: 3.2 and 1.9 ms.  X and
// the offsets are read once per iteration of two genes (one above p = 5), from
// the XCD's L2, which is why the caller takes this path only where they fit
// there (launch_irls_gene's callers hold the rule).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../../include/devil_hip.h"
#include "device_common.hpp"
#include "kernels.hpp"
#include "lane_sums.hpp"
#include "tile_common.hpp"
#include "wave_solve.hpp"

namespace dv {

template <int P, int NG, typename CT>
struct GeneOps {
  CT y[NG];
  double x[P];
  double off;
};

constexpr int kGeneMaxWaves = 8;

// LDS of a workgroup.
template <int NV, int NG, int P>
struct GeneLds {
  double e2[kExpTab];
  double part[NG][kGeneMaxWaves * NV];
  double tot[NG][NV + P];  // system entries, then the right-hand side
  double b[NG][P];
  double k[NG];
  int gene[NG];            // -1: the slot is empty
};

// p[i] from a scalar base and a 32-bit byte offset
template <typename T>
__device__ __forceinline__ T at(const T* p, uint32_t i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) +
                                     i * (uint32_t)sizeof(T));
}

// ICPT: column 0 of X is all ones (no loads and products for it, and the
// pairs (0, b) are the gradient).
template <int P, bool ICPT, int NG, typename CT>
__device__ __forceinline__ void irls_genes(
    const GeneDesign& gd, const CT* __restrict__ Y, int64_t ld, const int32_t* __restrict__ list,
    int ngenes, int32_t* __restrict__ next, double* __restrict__ beta,
    const double* __restrict__ kvec, int max_iter, double eps, int32_t* __restrict__ iters,
    int32_t* __restrict__ status,
    GeneLds<P*(P + 1) / 2 + (ICPT ? 0 : P), NG, P>& sh) {
  constexpr int NP = P * (P + 1) / 2;
  constexpr int NV = ICPT ? NP : NP + P;
  constexpr int J0 = ICPT ? 1 : 0;
  constexpr int NL = scatter_left(NV);
  const uint32_t tid = threadIdx.x, T = blockDim.x;
  const int lane = tid & 63, wave = wave_index(), nw = (int)(T >> 6);
  const uint32_t n = (uint32_t)gd.n, full = n / T;
  const double* xcol[P];
#pragma unroll
  for (int j = 0; j < P; ++j) xcol[j] = gd.X + (int64_t)j * gd.n;
  int where[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) where[i] = scatter_index<NV>(lane, i);
  // wave u < NG solves slot u; lane q of it finishes entry q of the system
  constexpr int NQ = (NV + 63) / 64;
  double ks[NQ], kz[NQ];  // column sum and 1, or 0 and 0 for an all-zero column
  if (wave < NG) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int q = lane + 64 * i;
      const int pi = q < NP ? gd.kidx_pair[q] : q < NV ? gd.kidx_lin[q - NP] : -1;
      kz[i] = pi >= 0 ? 1.0 : 0.0;
      ks[i] = pi >= 0 && q < NP ? gd.ksum[pi] : 0.0;
    }
  }
  int it = 0, st = 0;
  auto take = [&](int idx) {  // by wave `slot`, all lanes
    const int slot = wave;
    const int g = idx < ngenes ? (list ? list[idx] : idx) : -1;
    if (lane == 0) {
      sh.gene[slot] = g;
      if (g >= 0) sh.k[slot] = kvec[g];
    }
    if (g >= 0 && lane < P) sh.b[slot][lane] = beta[(int64_t)g * P + lane];
    it = 0;
    st = 0;
  };
  // slot 0 starts with gene blockIdx.x; the others with what no workgroup
  // starts with, from the counter (which starts at the grid size)
  auto fetch = [&]() {
    int idx = 0;
    if (lane == 0) idx = atomicAdd(next, 1);
    return __builtin_amdgcn_readfirstlane(idx);
  };
  if (wave == 0) take(blockIdx.x);
  else if (wave < NG) take(ngenes > (int)gridDim.x ? fetch() : ngenes);
  __syncthreads();
  typedef GeneOps<P, NG, CT> Ops;
  for (;;) {
    int g[NG];
    bool any = false, all = true;
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      g[u] = __builtin_amdgcn_readfirstlane(sh.gene[u]);
      any |= g[u] >= 0;
      all &= g[u] >= 0;
    }
    if (!any) return;
    // The sums of M genes (slots u0 .. u0 + M - 1) over the cells.
    auto pass = [&](auto count, int u0) {
      constexpr int M = decltype(count)::value;
      double b[M][P], k[M];
      const CT* yrow[M];
#pragma unroll
      for (int u = 0; u < M; ++u) {
        k[u] = uniform_f64(sh.k[u0 + u]);
        yrow[u] = Y + (int64_t)__builtin_amdgcn_readfirstlane(sh.gene[u0 + u]) * ld;
#pragma unroll
        for (int j = 0; j < P; ++j) b[u][j] = uniform_f64(sh.b[u0 + u][j]);
      }
      double acc[M][NV];
#pragma unroll
      for (int u = 0; u < M; ++u)
#pragma unroll
        for (int q = 0; q < NV; ++q) acc[u][q] = 0.0;
      // cell min(c, n - 1); scalar column pointers and 32-bit byte offsets (the
      // caller's rule keeps a column far below 4 GB)
      auto load = [&](uint32_t c, Ops& o) {
        const uint32_t i = min(c, n - 1);
#pragma unroll
        for (int j = J0; j < P; ++j) o.x[j] = at(xcol[j], i);
        o.off = at(gd.off, i);
#pragma unroll
        for (int u = 0; u < M; ++u) o.y[u] = at(yrow[u], i);
      };
      // the element arithmetic of the tile kernel: w = exp(-x'b - off),
      // r = m w - 1 = (y w - 1) / (1 + k w)
      auto body = [&](const Ops& o, bool in) {
        double r[M];
#pragma unroll
        for (int u = 0; u < M; ++u) {
          double eta = -o.off;
          if constexpr (ICPT) eta -= b[u][0];
#pragma unroll
          for (int j = J0; j < P; ++j) eta = fma(-b[u][j], o.x[j], eta);
          const double w = exp_tab(eta, sh.e2);
          const double d = fma(k[u], w, 1.0);
          r[u] = fma((double)o.y[u], w, -1.0) * rcp1_f64(d);
          r[u] = in ? r[u] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < M; ++u) {
          int q = 0;
#pragma unroll
          for (int a = 0; a < P; ++a) {
            const double rx = ICPT && a == 0 ? r[u] : r[u] * o.x[a];
#pragma unroll
            for (int bb = a; bb < P; ++bb) {
              if (ICPT && bb == 0) acc[u][q] += rx;
              else acc[u][q] = fma(rx, o.x[bb], acc[u][q]);
              ++q;
            }
          }
          if constexpr (!ICPT) {
#pragma unroll
            for (int a = 0; a < P; ++a) acc[u][NP + a] = fma(r[u], o.x[a], acc[u][NP + a]);
          }
        }
      };
      // two buffers in turn, loaded a step ahead; the last step is partial
      // (or empty) and masks its lanes
      Ops A, B;
      load(tid, A);
      uint32_t c = tid;
      for (uint32_t s = 0; s < full / 2; ++s, c += 2 * T) {
        load(c + T, B);
        body(A, true);
        load(c + 2 * T, A);
        body(B, true);
      }
      if (full & 1) {
        load(c + T, B);
        body(A, true);
        c += T;
        A = B;
      }
      if (full * T < n) body(A, c < n);
#pragma unroll
      for (int u = 0; u < M; ++u) {
        scatter_step<NV, 32>(acc[u], lane);
#pragma unroll
        for (int i = 0; i < NL; ++i)
          if (where[i] >= 0) sh.part[u0 + u][wave * NV + where[i]] = acc[u][i];
      }
    };
    if (NG > 1 && all) {
      pass(std::integral_constant<int, NG>{}, 0);
    } else {
#pragma unroll 1
      for (int u = 0; u < NG; ++u)
        if (__builtin_amdgcn_readfirstlane(sh.gene[u]) >= 0)
          pass(std::integral_constant<int, 1>{}, u);
    }
    __syncthreads();
    int mine = -1;
#pragma unroll
    for (int u = 0; u < NG; ++u)
      if (wave == u) mine = g[u];
    if (mine >= 0) {
      const int slot = wave;
      const double k = uniform_f64(sh.k[slot]);
      // A = k (X'diag(r)X + X'X), g = k X'r (k_irls_update's system)
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int q = lane + 64 * i;
        if (q < NV) {
          double s = 0.0;
          for (int u = 0; u < nw; ++u) s += sh.part[slot][u * NV + q];
          if (q < NP) sh.tot[slot][q] = kz[i] != 0.0 ? k * (s + ks[i]) : 0.0;
          if (ICPT ? q < P : q >= NP)
            sh.tot[slot][NV + (ICPT ? q : q - NP)] = kz[i] != 0.0 ? k * s : 0.0;
        }
      }
      __builtin_amdgcn_wave_barrier();
      double x[P];
      if constexpr (P <= 2) {  // shorter than the searches and exchanges
        double A[P][P];
        int perm[P];
#pragma unroll
        for (int a = 0; a < P; ++a) {
          x[a] = sh.tot[slot][NV + a];
#pragma unroll
          for (int c = a; c < P; ++c) A[a][c] = A[c][a] = sh.tot[slot][tri<P>(a, c)];
        }
        if (lu_factor<P>(A, perm)) st |= DEVIL_GENE_SINGULAR;
        lu_solve<P>(A, perm, x);
      } else {
        const int li = min(lane, P - 1);
        double row[P];
#pragma unroll
        for (int j = 0; j < P; ++j) {
          const int a = min(li, j), c = max(li, j);
          row[j] = sh.tot[slot][a * P - a * (a - 1) / 2 + (c - a)];
        }
        if (wave_lu_solve<P>(row, sh.tot[slot][NV + li], lane, x)) st |= DEVIL_GENE_SINGULAR;
      }
      double mx = 0.0;
      bool has_nan = false;
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const double d = fabs(x[j]);
        if (isnan(d)) has_nan = true;
        else mx = fmax(mx, d);
      }
      bool conv = !has_nan && mx < eps;
      ++it;
      if (isnan(x[0])) {
        conv = true;
        st |= DEVIL_GENE_NAN;
      }
      if (!conv && it >= max_iter) st |= DEVIL_GENE_MAXITER;
      const bool stop = conv || it >= max_iter;
      if (lane == 0) {
#pragma unroll
        for (int j = 0; j < P; ++j) {
          const double bj = sh.b[slot][j] + x[j];
          sh.b[slot][j] = bj;
          if (stop) beta[(int64_t)mine * P + j] = bj;
        }
        if (stop) {
          iters[mine] = it;
          status[mine] = st;
        }
      }
      if (stop) take(fetch());
    }
    __syncthreads();
  }
}

template <int P, bool ICPT>
__global__ __launch_bounds__(64 * kGeneMaxWaves) void k_irls_gene(
    GeneDesign gd, Counts c, const int32_t* __restrict__ list, int ngenes,
    int32_t* __restrict__ next, double* __restrict__ beta, const double* __restrict__ kvec,
    int max_iter, double eps, int32_t* __restrict__ iters, int32_t* __restrict__ status) {
  constexpr int NG = gene_slots(P);
  __shared__ GeneLds<P*(P + 1) / 2 + (ICPT ? 0 : P), NG, P> sh;
  exp_tab_fill(sh.e2, threadIdx.x, blockDim.x);
  auto run = [&](auto* Y) {
    irls_genes<P, ICPT, NG>(gd, Y, c.ld, list, ngenes, next, beta, kvec, max_iter, eps, iters,
                            status, sh);
  };
  if (c.dtype == 0) run(static_cast<const int32_t*>(c.ptr));
  else if (c.dtype == 1) run(static_cast<const float*>(c.ptr));
  else run(static_cast<const double*>(c.ptr));
}

// Workgroups of a launch: enough to fill the GPU; each takes further genes
// from the counter (*next must hold the grid size when the kernel starts).
template <int P>
hipError_t launch_gene_p(hipStream_t s, const GeneDesign& gd, Counts c, const int32_t* list,
                         int ngenes, int32_t* next, double* beta, const double* kvec,
                         int max_iter, double eps, int32_t* iters, int32_t* status) {
  // Four wavefronts fill a CU's SIMDs once and leave room for other genes'
  // workgroups beside them (their solves overlap this one's cells); long rows
  // take eight, which shortens the last genes' iterations.  IRLS ms with 256
  // and 512 threads:
  //   10000 genes x 4000 cells     p = 2 0.93, 0.88;  p = 5 1.62, 2.15;  p = 8 2.88, 4.90
  //   3000 x 16384                 p = 2 1.45, 1.17;  p = 5 2.06, 1.80;  p = 8 3.60, 4.05
  //   10000 x 16384                p = 2 2.84, 2.48;  p = 5 4.54, 4.57;  p = 8 9.52, 10.6
  //   3000 x 30000                 p = 2 2.24, 1.80;  p = 5 3.64, 3.13
  // (p = 2 would take 512 from 4000 cells on, p = 8 256 throughout; the line is
  // p = 5's.)
  const int T = gd.n <= 16384 ? 256 : 512;
  const int grid = std::min(ngenes, T == 256 ? 1024 : 512);
  const hipError_t e = launch_fill_i32(s, next, 1, grid);
  if (e != hipSuccess) return e;
  if (gd.intercept)
    hipLaunchKernelGGL((k_irls_gene<P, true>), dim3((unsigned)grid), dim3(T), 0, s, gd, c,
                       list, ngenes, next, beta, kvec, max_iter, eps, iters, status);
  else
    hipLaunchKernelGGL((k_irls_gene<P, false>), dim3((unsigned)grid), dim3(T), 0, s, gd, c,
                       list, ngenes, next, beta, kvec, max_iter, eps, iters, status);
  return hipGetLastError();
}

hipError_t launch_irls_gene(hipStream_t s, const GeneDesign& gd, Counts c, int p,
                            const int32_t* list, int ngenes, int32_t* next, double* beta,
                            const double* kvec, int max_iter, double eps, int32_t* iters,
                            int32_t* status) {
  if (ngenes <= 0) return hipSuccess;
  if (max_iter <= 0) return hipErrorInvalidValue;
#define DV_GENE_P(P_) \
  case P_: \
    return launch_gene_p<P_>(s, gd, c, list, ngenes, next, beta, kvec, max_iter, eps, iters,     \
                             status);
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
