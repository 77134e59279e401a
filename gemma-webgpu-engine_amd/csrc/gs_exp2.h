// The binary64 table exponential of the chunk scan's rescales and of the
// finish kernel's normaliser recomputation: 2^(y/256) = 2^(j/256) * 2^k * e^r
// with y = 256 k + j + s, |s| <= 1/2, r = s ln2 / 256, a correctly rounded
// 256-entry table and the quadratic 1 + r + r^2/2: relative error below
// 4.2e-10 per evaluation (tests/test_scan_exp2.py pins it). exp2_256_tight
// takes the quartic instead, for the deep draw's masses: relative error
// below 1e-15 per evaluation. exp_neg is e^d within an ulp, for
// log-probabilities and the typical-p rows.
#pragma once

#include <hip/hip_runtime.h>

#include "gs_exp2_table.h"
#include "gs_math.h"

namespace gs {

// 2^(j/256), j = 0..255 (each translation unit holds its own copy)
static __constant__ double c_exp2_256[256] = {GS_EXP2_TABLE_256};

// Terms with (l - lmax)/T < -60 are not summed: each is below e^-60 of the
// maximum's term, so together they move the normaliser by less than
// V * e^-60 < 3e-21 relative. In units of y = 256 log2(e) (l - lmax)/T:
constexpr double kSkipY = -22160.0;

// tab: the table above, or a copy of it in LDS
__device__ __forceinline__ double exp2_256(double y, const double* tab) {
  const double n = __builtin_rint(y);
  const double s = y - n;  // |s| <= 1/2
  const double p = __builtin_fma(s, __builtin_fma(s, GS_EXP2_256_C2, GS_EXP2_256_C1), 1.0);
  const int ni = (int)n;
  return __builtin_ldexp(tab[ni & 255] * p, ni >> 8);
}

__device__ __forceinline__ double exp2_256_tight(double y, const double* tab) {
  const double n = __builtin_rint(y);
  const double s = y - n;  // |s| <= 1/2
  double p = __builtin_fma(s, GS_EXP2_256_C4, GS_EXP2_256_C3);
  p = __builtin_fma(s, p, GS_EXP2_256_C2);
  p = __builtin_fma(s, p, GS_EXP2_256_C1);
  p = __builtin_fma(s, p, 1.0);
  const int ni = (int)n;
  return __builtin_ldexp(tab[ni & 255] * p, ni >> 8);
}

// exp_neg's factors 2^(j/32), one LDS bank pair each: random j never conflict
constexpr int kExpTableBits = 5;
constexpr int kExpTable = 1 << kExpTableBits;

// e^d for d <= 0, within an ulp. Below -700 it is e^-700: a sum here is at
// least 1, so no such term ever changes it.
__device__ __forceinline__ double exp_neg(double d, const double* tab) {
  constexpr double kInv = kExpTable * 1.44269504088896338700e+00;
  constexpr double kHi = 6.93147180369123816490e-01 / kExpTable;  // 33 bits: k kHi is exact
  constexpr double kLo = 1.90821492927058770002e-10 / kExpTable;
  constexpr double kShift = 6755399441055744.0;  // 1.5 2^52: the sum's low word is the nearest integer
  d = __builtin_fmax(d, -700.0);
  const double z = __builtin_fma(d, kInv, kShift);
  const double k = z - kShift;
  const int i = (int)(uint32_t)gsm::bits_of(z);
  const double r = __builtin_fma(-k, kLo, __builtin_fma(-k, kHi, d));
  double p = __builtin_fma(r, 1.0 / 720.0, 1.0 / 120.0);
  p = __builtin_fma(r, p, 1.0 / 24.0);
  p = __builtin_fma(r, p, 1.0 / 6.0);
  p = __builtin_fma(r, p, 0.5);
  p = __builtin_fma(r, p, 1.0);
  const double t = tab[i & (kExpTable - 1)];
  // the exponent stays normal: i / kExpTable >= -1011
  return gsm::double_of(gsm::bits_of(__builtin_fma(t * r, p, t)) + ((uint64_t)(uint32_t)(i >> kExpTableBits) << 52));
}

// (the whole workgroup calls it)
__device__ __forceinline__ void load_exp_table(double* tab) {
  if (threadIdx.x < kExpTable) tab[threadIdx.x] = c_exp2_256[threadIdx.x * (256 / kExpTable)];
  __syncthreads();
}

}  // namespace gs
