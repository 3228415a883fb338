// The FP64 IRLS accumulate of one 16-gene tile and cell chunk (see
// kernels_tile.hip), shared by the round kernel (kernels_irls64.hip) and the
// joint rounds (kernels_tile.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "kernels.hpp"
#include "tile_common.hpp"

namespace dv {

// lane l of a wave: gene slot s = l % 16, cell group h = l / 16; its cells in
// block b are 16 b + 4 h + r.
template <int P, int VC, typename CT, bool VEC>
__device__ __forceinline__ void irls_tile_chunk(const TileDesign& td, const CT* __restrict__ Y,
                                                int64_t ld, const int32_t* __restrict__ active,
                                                int nA, const double* __restrict__ beta,
                                                const double* __restrict__ kvec, int tile,
                                                int chunk, double* __restrict__ part,
                                                const double* __restrict__ e2) {
  constexpr int NJ = (P + 3) / 4;
  constexpr int NTMAX = mfma_tiles<P, VC>();
  const int lane = threadIdx.x & 63;
  const int s = lane & 15, h = lane >> 4;
  const int slot = tile * 16 + s;
  const bool live = slot < nA;
  const int g = live ? active[slot] : active[tile * 16];
  const int NT = VC > 0 ? td.ncol / 16 : td.nt;
  // B operand of the eta product: -beta[g][4 j + h]
  double bneg[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int f = 4 * j + h;
    bneg[j] = (live && f < P) ? -beta[(int64_t)g * P + f] : 0.0;
  }
  const double k = live ? kvec[g] : 0.0;
  const CT* yrow = Y + (int64_t)g * ld;
  const CT* yh = yrow + 4 * h;
  d4 acc[NTMAX > 0 ? NTMAX : 1];
#pragma unroll
  for (int t = 0; t < NTMAX; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
  double accv[VC > 0 ? VC : 1];
#pragma unroll
  for (int v = 0; v < VC; ++v) accv[v] = 0.0;
  const int64_t b0 = (int64_t)chunk * td.chunk_blocks;
  const int64_t b1 = min((int64_t)(chunk + 1) * td.chunk_blocks, td.nblk);
  typedef TileBlock<NJ, NTMAX, CT> Blk;
  auto body = [&](const Blk& cur, const VCols<VC>& kv, int64_t) {
    d4 eta = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < NJ; ++j) eta = mfma16x16x4(cur.xa[j], bneg[j], eta);
    // m w - 1 = (y w - 1) / (1 + k w), summed without the n-term
    // cancellation of sum (m w) - sum 1
    double q[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double w = exp_tab(eta[r] - cur.off[r], e2);
      const double d = fma(k, w, 1.0);
      q[r] = fma((double)cur.y[r], w, -1.0) * rcp1_f64(d);
    }
#pragma unroll
    for (int t = 0; t < NTMAX; ++t) {
      if (t < NT) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t] = mfma16x16x4(q[r], cur.kb[t][r], acc[t]);
      }
    }
    add_vcols<VC>(q, kv.k, accv);
  };
  auto load_own = [&](int64_t b, VCols<VC>& o) { load_vcols<VC>(td, b, h, NT, o.k); };
  auto load = [&](int64_t b, Blk& o) {
    load_tile_block<NJ, NTMAX, CT, VEC>(td, yh, b, lane, h, NT, td.offp, o);
  };
  auto load_tail = [&](int64_t b, Blk& o) {
    load_tile_block_tail<NJ, NTMAX, CT>(td, yrow, b, lane, h, NT, td.offp, o);
  };
  // trailing chunks may be empty
  pipeline_own<Blk, VCols<VC>>(b0, min(b1, td.n / 16), b1, load, load_tail, load_own, body);
  // partial sums: register r holds gene slot h + 4 r, column 16 t + s
  double* out = part + ((int64_t)tile * td.nchunk + chunk) * 16 * td.ncp;
#pragma unroll
  for (int t = 0; t < NTMAX; ++t) {
    if (t < NT) {
#pragma unroll
      for (int r = 0; r < 4; ++r) out[(h + 4 * r) * td.ncp + 16 * t + s] = acc[t][r];
    }
  }
  store_vcols<VC>(td, h, NT, accv, out + s * td.ncp + 16 * NT);
}

// FP64 accumulate of workgroup wb of nwb (4 tiles, one per wave); e2: the
// exponential table, filled by the caller
template <int P, int VC>
__device__ __forceinline__ void irls_accum_body(const TileDesign& td, const Counts& c,
                                                const int32_t* __restrict__ active,
                                                const int32_t* __restrict__ nactive,
                                                const double* __restrict__ beta,
                                                const double* __restrict__ kvec,
                                                double* __restrict__ part, const double* e2,
                                                int wb, int nwb) {
  const int nA = *nactive;
  const int ntile = (nA + 15) / 16;
  const int wave = wave_index();
  int chunk, group;
  tile_coords_at(wb, nwb, td.nchunk, chunk, group);
  const int tile = group * 4 + wave;
  if (tile >= ntile) return;
  with_counts(c, [&](auto Y, auto vec) {
    typedef std::remove_cv_t<std::remove_pointer_t<decltype(Y)>> CT;
    irls_tile_chunk<P, VC, CT, decltype(vec)::value>(td, Y, c.ld, active, nA, beta, kvec, tile,
                                                 chunk, part, e2);
  });
}

}  // namespace dv
