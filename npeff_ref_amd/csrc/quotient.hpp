// The quotients of the multiplicative updates.
#pragma once
#include "split_bf16.hpp"

namespace dn {

// n / den from the reciprocal and one correction step: 5 vector instructions where the IEEE division
// sequence takes 11.  For positive den: the quotient as the division rounds it but for about one in four
// million (then an ulp off; emulated with every reciprocal an ulp off), within 2 ulp where n is too small
// for the correction's residue (below 2^-100).
// Outside 2^-126 <= den < 2^126, and where the quotient is 2^126 or more, the result means nothing:
// the reciprocal of such a den is no normal number, and the correction turns an infinity into NaN.
__device__ __forceinline__ float quotient_in_range(float n, float den) {
  const float rc = __builtin_amdgcn_rcpf(den), q0 = n * rc;
  return __builtin_fmaf(__builtin_fmaf(-den, q0, n), rc, q0);
}

// Four quotients n / den, any operands: as quotient_in_range where that holds for all four, else by
// division.  One unsigned maximum over the bits of the dens and the results (four instructions) shows
// everything that does not hold: a large, infinite, negative or NaN den, and by its result (an infinity
// or NaN) a zero or subnormal one.  (Negative results take the division, too.)
__device__ __forceinline__ f32x4 mu_quotients(const f32x4& n, const f32x4& den) {
  f32x4 q;
  unsigned top = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    q[i] = quotient_in_range(n[i], den[i]);
    const unsigned a = __float_as_uint(q[i]), b = __float_as_uint(den[i]);
    top = top > a ? top : a;
    top = top > b ? top : b;
  }
  if (__builtin_expect(top >= 0x7e800000u, 0)) {  // (2^126)
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = n[i] / den[i];
  }
  return q;
}

}  // namespace dn
