/* fx_near.hpp -- square root and reciprocal of a float, correctly rounded,
 * for arguments in the middle of the range.
 *
 * The compiler's IEEE sqrtf and division carry scaling, special cases and
 * fix-ups for every float: 16 and 11 instructions on gfx950, 27 of about 62
 * of a pair term.  In [2^-79, 2^49) one residual step on the hardware's
 * approximation is enough (Newton's iteration with an exact residual by
 * fmaf, as Markstein describes it): 5 and 3 instructions.  Every float of
 * that range gives the bits of sqrtf and of 1.0f / b (tests/test_gpu_near.py
 * goes through all of them); outside it some do not (75 of them between
 * 2^-111 and 2^113), so a caller checks with near_bits and takes sqrtf and
 * the division where an argument lies elsewhere.
 *
 * near_bits(x) < FX_NEAR_SPAN for x in the range; zero, negative, infinite
 * and NaN arguments are outside.  Several are checked by one comparison of
 * their OR (FX_NEAR_SPAN is a power of two).
 */
#ifndef FX_NEAR_HPP
#define FX_NEAR_HPP

#define FX_NEAR_SPAN 0x40000000u

__device__ __forceinline__ unsigned near_bits(float x) { return __float_as_uint(x) - 0x18000000u; }

__device__ __forceinline__ float near_sqrt(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float s = x * y, h = 0.5f * y;
  return fmaf(fmaf(-s, s, x), h, s);
}

__device__ __forceinline__ float near_rcp(float b) {
  const float r = __builtin_amdgcn_rcpf(b);
  return fmaf(fmaf(-b, r, 1.0f), r, r);
}

#endif
