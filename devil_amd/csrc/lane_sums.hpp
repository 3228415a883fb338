// Sums over a wavefront's lanes of many values at once, for the kernels whose
// lanes own cells.
#pragma once
#include <hip/hip_runtime.h>

namespace dv {

// Lane sums of V values: after scatter_step<V, 32> a lane's v[i] holds the
// wave's sum of value scatter_index<V>(lane, i), i < scatter_left(V).  Each
// step halves the values a lane holds and pairs lanes 32, 16, 8, 4, 2, 1 apart,
// so the 64-lane sums of V values take about V exchanges instead of 6 V.
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

// the value whose sum this lane's i-th entry holds, -1 for none
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

}  // namespace dv
