// Several quotients by one divisor.  quot_recip(v) is 1/v to about half an ulp: the
// hardware estimate (relative error 4.7e-8 in FP64, an ulp in FP32), then two
// Newton steps (FP32: one).  quot(a, v, r) multiplies and corrects with the
// remainder a - v q from a fused multiply-add (Markstein, IBM J. Res. Dev. 34,
// 1990), and the result is a/v correctly rounded.  In FP64 that is how the
// compiler's own division ends.  In FP32 the quotient before the correction is
// within 1.5 ulp, the reciprocal within 2^-24 and the remainder within 2^-25, so
// before its rounding the corrected value is within 4.5 x 2^-25 ulp of a/v: only
// quotients that near to a midpoint could round wrongly.  A divisor of 24 bits has
// at most a few such numerators; all were tried, none does.  div_fixup restores the
// special cases (zeros, infinities, NaN).  v, 1/v and a/v must be in the normal
// range, as the sweeps' pivots are.  The first quotient costs about what `/` does,
// each further one four instructions instead of twelve.
#pragma once

namespace c3d {

__device__ __forceinline__ double quot_recip(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
}
__device__ __forceinline__ double quot(double a, double v, double r) {
  const double q = a * r;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-v, q, a), r, q), v, a);
}
__device__ __forceinline__ float quot_recip(float v) {
  const float r = __builtin_amdgcn_rcpf(v);
  return __builtin_fmaf(__builtin_fmaf(-v, r, 1.0f), r, r);
}
__device__ __forceinline__ float quot(float a, float v, float r) {
  const float q = a * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-v, q, a), r, q), v, a);
}

// quot by a divisor whose reciprocal is tabulated: r is 1/v rounded (FP64), or
// that rounded to FP32 and refined for the FP32 divisor.
__device__ __forceinline__ double tab_recip(double, double r) { return r; }
__device__ __forceinline__ float tab_recip(float v, double r) {
  const float q = (float)r;
  return __builtin_fmaf(__builtin_fmaf(-v, q, 1.0f), q, q);
}

}  // namespace c3d
