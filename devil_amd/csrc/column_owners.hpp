// Which of an IRLS pass's sums stands for a column of K.
#pragma once
#include <stdint.h>

namespace dv {

// The sums of a pass are the p (p + 1) / 2 products x_a x_b, then the p design
// columns; equal columns share one column of K (kidx_pair, kidx_lin; -1: the
// column is zero).  A kernel whose lanes own sums stores a column once: the
// first sum with it owns it.  Sums of equal columns need not have equal bits
// (with x_3 = x_1 x_2 the sums r x_0 x_3 and r x_1 x_2 are rounded differently),
// so which of them is kept must not be left to the order of the writes.
// pair: bit q for product q; lin: bit a for design column a.
inline void column_owners(const int* kidx_pair, const int* kidx_lin, int p, uint64_t& pair,
                          uint32_t& lin) {
  const int np = p * (p + 1) / 2;
  pair = 0;
  lin = 0;
  for (int q = 0; q < np + p; ++q) {
    const int col = q < np ? kidx_pair[q] : kidx_lin[q - np];
    bool first = col >= 0;
    for (int e = 0; e < q && first; ++e)
      first = (e < np ? kidx_pair[e] : kidx_lin[e - np]) != col;
    if (!first) continue;
    if (q < np) pair |= uint64_t(1) << q;
    else lin |= uint32_t(1) << (q - np);
  }
}

}  // namespace dv
