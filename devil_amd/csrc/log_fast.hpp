// log(1 + x) of the init pass's ordinary counts.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dv {

// log(1 + x) for 0 <= x < 2^52: log_tab's scheme without its special cases, on
// the bits of u = 1 + x.  Rounding u's mantissa to 7 bits (with the carry into
// the exponent) gives e and j with m = u 2^-e within 2^-8 of F = 1 + j/128;
// r = m / F - 1 by one fused multiply-add with the rounded 1/F, whose own
// error is in the table's logarithm (-log(inv), correctly rounded, computed to
// 60 digits); x = 0 gives 0 exactly.  Largest errors against log1pl, in units
// of 2^-53: 2.33 over (0, 2^50) and 2.19 over counts divided by size factors;
// log_tab's scheme with a correctly rounded table has 3.17 and 2.23.  About 26
// instructions against log_tab's 42; the init pass of 4000 genes x 500000
// cells, p = 8, takes 3.2 ms against 3.9 (FP64 issue bounds it: this logarithm
// and 4 matrix instructions of 64 cycles per block of 16 cells).
struct LogFast {
  double inv, ln;
};
constexpr int kLogFast = 128;
static __device__ constexpr double kLogFastLn[kLogFast] = {
    0.0, 0x1.fe02a6b106799p-8, 0x1.fc0a8b0fc03c4p-7, 0x1.7b91b07d5b126p-6, 0x1.f829b0e7832f8p-6,
    0x1.39e87b9febd68p-5, 0x1.77458f632dcffp-5, 0x1.b42dd711971b9p-5, 0x1.f0a30c01162a8p-5,
    0x1.16536eea37ae3p-4, 0x1.341d7961bd1d0p-4, 0x1.51b073f06183cp-4, 0x1.6f0d28ae56b4ep-4,
    0x1.8c345d6319b23p-4, 0x1.a926d3a4ad562p-4, 0x1.c5e548f5bc743p-4, 0x1.e27076e2af2eap-4,
    0x1.fec9131dbeabcp-4, 0x1.0d77e7cd08e5bp-3, 0x1.1b72ad52f67a2p-3, 0x1.29552f81ff521p-3,
    0x1.371fc201e8f75p-3, 0x1.44d2b6ccb7d1cp-3, 0x1.526e5e3a1b438p-3, 0x1.5ff3070a793d6p-3,
    0x1.6d60fe719d21bp-3, 0x1.7ab890210d907p-3, 0x1.87fa06520c911p-3, 0x1.9525a9cf456b6p-3,
    0x1.a23bc1fe2b561p-3, 0x1.af3c94e80bff3p-3, 0x1.bc286742d8cd4p-3, 0x1.c8ff7c79a9a20p-3,
    0x1.d5c216b4fbb94p-3, 0x1.e27076e2af2e8p-3, 0x1.ef0adcbdc5935p-3, 0x1.fb9186d5e3e29p-3,
    0x1.0402594b4d041p-2, 0x1.0a324e27390e2p-2, 0x1.1058bf9ae4ad4p-2, 0x1.1675cababa60fp-2,
    0x1.1c898c16999fbp-2, 0x1.22941fbcf7966p-2, 0x1.2895a13de86a4p-2, 0x1.2e8e2bae11d31p-2,
    0x1.347dd9a987d56p-2, 0x1.3a64c556945eap-2, 0x1.404308686a7e4p-2, 0x1.4618bc21c5ec2p-2,
    0x1.4be5f957778a1p-2, 0x1.51aad872df82ep-2, 0x1.5767717455a6cp-2, 0x1.5d1bdbf5809cap-2,
    0x1.62c82f2b9c796p-2, 0x1.686c81e9b14adp-2, 0x1.6e08eaa2ba1e4p-2, 0x1.739d7f6bbd007p-2,
    0x1.792a55fdd47a1p-2, 0x1.7eaf83b82afc2p-2, 0x1.842d1da1e8b18p-2, 0x1.89a3386c1425bp-2,
    0x1.8f11e873662c8p-2, 0x1.947941c2116fbp-2, 0x1.99d958117e08ap-2, 0x1.9f323ecbf984dp-2,
    0x1.a484090e5bb09p-2, 0x1.a9cec9a9a084ap-2, 0x1.af1293247786bp-2, 0x1.b44f77bcc8f64p-2,
    0x1.b9858969310fdp-2, 0x1.beb4d9da71b7ap-2, 0x1.c3dd7a7cdad4dp-2, 0x1.c8ff7c79a9a21p-2,
    0x1.ce1af0b85f3ecp-2, 0x1.d32fe7e00ebd5p-2, 0x1.d83e7258a2f3ep-2, 0x1.dd46a04c1c4a1p-2,
    0x1.e24881a7c6c26p-2, 0x1.e744261d68789p-2, 0x1.ec399d2468cc1p-2, 0x1.f128f5faf06ecp-2,
    0x1.f6123fa7028adp-2, 0x1.faf588f78f31dp-2, 0x1.ffd2e0857f497p-2, 0x1.02552a5a5d0ffp-1,
    0x1.04bdf9da926d2p-1, 0x1.0723e5c1cdf41p-1, 0x1.0986f4f573521p-1, 0x1.0be72e4252a83p-1,
    0x1.0e44985d1cc8cp-1, 0x1.109f39e2d4c96p-1, 0x1.12f719593efbdp-1, 0x1.154c3d2f4d5eap-1,
    0x1.179eabbd899a0p-1, 0x1.19ee6b467c96fp-1, 0x1.1c3b81f713c25p-1, 0x1.1e85f5e7040d1p-1,
    0x1.20cdcd192ab6ep-1, 0x1.23130d7bebf43p-1, 0x1.2555bce98f7cap-1, 0x1.2795e1289b11bp-1,
    0x1.29d37fec2b08bp-1, 0x1.2c0e9ed448e8cp-1, 0x1.2e47436e40268p-1, 0x1.307d7334f10bep-1,
    0x1.32b1339121d71p-1, 0x1.34e289d9ce1d2p-1, 0x1.37117b54747b6p-1, 0x1.393e0d3562a1ap-1,
    0x1.3b68449fffc23p-1, 0x1.3d9026a7156fbp-1, 0x1.3fb5b84d16f43p-1, 0x1.41d8fe84672afp-1,
    0x1.43f9fe2f9ce67p-1, 0x1.4618bc21c5ec2p-1, 0x1.48353d1ea88dfp-1, 0x1.4a4f85db03ebbp-1,
    0x1.4c679afccee39p-1, 0x1.4e7d811b75bb0p-1, 0x1.50913cc01686bp-1, 0x1.52a2d265bc5abp-1,
    0x1.54b2467999498p-1, 0x1.56bf9d5b3f399p-1, 0x1.58cadb5cd7989p-1, 0x1.5ad404c359f2dp-1,
    0x1.5cdb1dc6c1765p-1, 0x1.5ee02a9241676p-1, 0x1.60e32f44788d9p-1,
};

// threads [0, nthreads) of the workgroup fill tab; the caller synchronises
__device__ __forceinline__ void log_fast_fill(LogFast* tab, int tid, int nthreads) {
  for (int j = tid; j < kLogFast; j += nthreads) {
    tab[j].inv = 1.0 / (1.0 + (double)j * (1.0 / kLogFast));
    tab[j].ln = kLogFastLn[j];
  }
}

// (also compiled for the host, where its error is checked)
__host__ __device__ __forceinline__ double log1p_fast(double x, const LogFast* tab) {
  const double u = 1.0 + x;
  const double c = x - (u - 1.0);  // the rounding error of u
  const uint64_t bits = __builtin_bit_cast(uint64_t, u);
  const int hi = (int)(bits >> 32);
  const int t = hi + 0x1000;
  const int e20 = (t & 0x7ff00000) - 0x3ff00000;  // 2^20 e
  const LogFast en = tab[(t >> 13) & (kLogFast - 1)];
  const double m = __builtin_bit_cast(
      double, (uint64_t)(uint32_t)(hi - e20) << 32 | (uint32_t)bits);
  const double scale =
      __builtin_bit_cast(double, (uint64_t)(uint32_t)(0x3ff00000 - e20) << 32);  // 2^-e
  const double r = fma(c * scale, en.inv, fma(m, en.inv, -1.0));
  double q = 1.0 / 7;
  q = fma(q, r, -1.0 / 6);
  q = fma(q, r, 1.0 / 5);
  q = fma(q, r, -1.0 / 4);
  q = fma(q, r, 1.0 / 3);
  q = fma(q, r, -0.5);
  const double lp = fma(r * r, q, r);
  const double ed = (double)e20;
  return fma(ed, 6.93147180369123816490e-01 / 1048576, en.ln) +
         fma(ed, 1.90821492927058770002e-10 / 1048576, lp);
}

}  // namespace dv
