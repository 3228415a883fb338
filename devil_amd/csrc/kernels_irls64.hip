// gfx950 FP64 IRLS accumulate of one round, 16-gene tiles (irls_tile.hpp; the
// scheme is described in kernels_tile.hip).  FP64 issue bounds it: per block
// of 16 cells ~145 vector instructions and, at 64 cycles each on the same
// units, ceil(p / 4) + 4 per 16-column tile matrix instructions, which is why
// a last tile of one or two columns is summed by vector instructions
// (vcols_of).
#include <hip/hip_runtime.h>

#include "irls_tile.hpp"

namespace dv {

template <int P, int VC>
__global__ __launch_bounds__(256) void k_irls_accum(TileDesign td, Counts c,
                                                    const int32_t* __restrict__ active,
                                                    const int32_t* __restrict__ nactive,
                                                    const double* __restrict__ beta,
                                                    const double* __restrict__ kvec,
                                                    double* __restrict__ part) {
  __shared__ double e2[kExpTab];
  exp_tab_fill(e2, threadIdx.x, blockDim.x);
  __syncthreads();
  irls_accum_body<P, VC>(td, c, active, nactive, beta, kvec, part, e2, blockIdx.x, gridDim.x);
}

template <int P>
hipError_t launch_irls_accum_p(hipStream_t s, dim3 grid, const TileDesign& td, Counts c,
                               const int32_t* active, const int32_t* nactive,
                               const double* beta, const double* kvec, double* part) {
  switch (vcols_of(td.ncol)) {
    case 0:
      hipLaunchKernelGGL((k_irls_accum<P, 0>), grid, dim3(256), 0, s, td, c, active, nactive,
                         beta, kvec, part);
      break;
    case 1:
      hipLaunchKernelGGL((k_irls_accum<P, 1>), grid, dim3(256), 0, s, td, c, active, nactive,
                         beta, kvec, part);
      break;
    default:
      hipLaunchKernelGGL((k_irls_accum<P, 2>), grid, dim3(256), 0, s, td, c, active, nactive,
                         beta, kvec, part);
  }
  return hipGetLastError();
}

hipError_t launch_irls_accum(hipStream_t s, const TileDesign& td, Counts c, int p,
                             const int32_t* active, const int32_t* nactive, int nA_bound,
                             const double* beta, const double* kvec, double* part) {
  if (nA_bound <= 0) return hipSuccess;
  const int ntile = (nA_bound + 15) / 16;
  const int groups = (ntile + 3) / 4;
  const dim3 grid((unsigned)((int64_t)groups * td.nchunk));
#define DV_ACCUM_P(P_) \
  case P_: return launch_irls_accum_p<P_>(s, grid, td, c, active, nactive, beta, kvec, part);
  switch (p) {
    DV_ACCUM_P(1)
    DV_ACCUM_P(2)
    DV_ACCUM_P(3)
    DV_ACCUM_P(4)
    DV_ACCUM_P(5)
    DV_ACCUM_P(6)
    DV_ACCUM_P(7)
    DV_ACCUM_P(8)
    DV_ACCUM_P(9)
    DV_ACCUM_P(10)
    default: return hipErrorInvalidValue;
  }
#undef DV_ACCUM_P
}

}  // namespace dv
