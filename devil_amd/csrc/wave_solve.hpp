// The p x p solve of an IRLS step on one wavefront, a row per lane.
#pragma once
#include <hip/hip_runtime.h>

namespace dv {

// DPP moves within 16 lanes (all lanes active): xor 1, xor 2, then mirrors,
// which pair the quads and the halves of a row once their lanes agree.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}

template <int CTRL>
__device__ __forceinline__ void pivot_step(double& key, int& pos) {
  const double ok = __hiloint2double(dpp_i<CTRL>(__double2hiint(key)),
                                     dpp_i<CTRL>(__double2loint(key)));
  const int op = dpp_i<CTRL>(pos);
  const bool take = ok > key || (ok == key && op < pos);
  key = take ? ok : key;
  pos = take ? op : pos;
}

__device__ __forceinline__ double lane_f64(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Solves the P x P system whose row i lane i < P holds, by the LU with partial
// pivoting of lu_factor / lu_solve, one lane per row: a pivot search over 16
// lanes, the pivot row in scalar registers, every row eliminated at once.  The
// rows keep their lanes; pos is a row's place in the permuted matrix.  x is
// the same in every lane.  Returns 1 where a pivot column is exactly zero.
template <int P>
__device__ __forceinline__ int wave_lu_solve(double (&row)[P], double rhs, int lane,
                                             double (&x)[P]) {
  int pos = lane, sing = 0;
  bool open = lane < P;
  int piv[P];
#pragma unroll
  for (int k = 0; k < P; ++k) {
    // the first row of largest magnitude; a NaN is chosen only where it
    // stands first, as the comparisons of lu_factor have it
    const double m = fabs(row[k]);
    double key = -2.0;
    if (open) key = isnan(m) ? (pos == k ? __builtin_inf() : -1.0) : m;
    int best = open ? pos : 64;
    pivot_step<0xB1>(key, best);
    pivot_step<0x4E>(key, best);
    pivot_step<0x141>(key, best);
    pivot_step<0x140>(key, best);
    best = __builtin_amdgcn_readfirstlane(best);
    const bool mine = open && pos == best;
    const int r = __builtin_ctzll(__ballot(mine));
    piv[k] = r;
    if (open && pos == k) pos = best;
    if (mine) {
      pos = k;
      open = false;
    }
    const double pk = lane_f64(row[k], r), prhs = lane_f64(rhs, r);
    if (pk == 0.0) sing = 1;
    const double l = pk == 0.0 ? row[k] : row[k] / pk;
#pragma unroll
    for (int j = k + 1; j < P; ++j) {
      const double pj = lane_f64(row[j], r);
      if (open) row[j] = fma(-l, pj, row[j]);
    }
    if (open) rhs = fma(-l, prhs, rhs);
  }
#pragma unroll
  for (int i = P - 1; i >= 0; --i) {
    x[i] = lane_f64(rhs / row[i], piv[i]);
    if (pos < i) rhs = fma(-row[i], x[i], rhs);
  }
  return sing;
}

}  // namespace dv
