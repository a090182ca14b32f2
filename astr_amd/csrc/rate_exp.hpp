// e^x for the rate constants: x = n ln 2 + r with the nearest n (Cody and
// Waite's two-part ln 2: n times the high part, 42 bits, is exact), e^r =
// 1 + r (1 + r P(r)) with P of degree 10, its constant 1/2, through the Chebyshev
// nodes of |r| <= ln 2 / 2 (its error 1e-18), scaled by 2^n.  The last two
// steps are fused, so what they add is rounded once: with 1 + (r + r^2 P) and
// degree 9, as many instructions, the result was off by 1.14 ulp and 0.321 RMS.
// Against 64 bits: at most 0.861 ulp, 0.3011 RMS; the library's exp on this GPU
// 0.868 and 0.3015.
// Host and device compile this text alike (a host program measures it).
#pragma once

namespace astr {

struct RateExpConstants {
  double l2e = 0x1.71547652b82fep+0, rnd = 0x1.8p52, hi = 0x1.62e42fefa3800p-1, lo = 0x1.ef35793c76730p-45;
  double c3 = 0x1.5555555555556p-3, c4 = 0x1.5555555555555p-5, c5 = 0x1.11111111109b5p-7, c6 = 0x1.6c16c16c167e2p-10,
         c7 = 0x1.a01a01a7c2efep-13, c8 = 0x1.a01a01a47a591p-16, c9 = 0x1.71de0db2f6b19p-19,
         c10 = 0x1.27e4e1f7222cbp-22, c11 = 0x1.af389ecfc4b9cp-26, c12 = 0x1.1f66d948a47d2p-29;
};

template <class Constants>
__device__ __forceinline__ double rate_exp_in(double x, const Constants& K) {  // |x| < 700
  const double t = fma(x, K.l2e, K.rnd);  // n in the low bits
  const double n = t - K.rnd;
  const double r = fma(-n, K.lo, fma(-n, K.hi, x));
  double p = fma(K.c12, r, K.c11);
  p = fma(p, r, K.c10);
  p = fma(p, r, K.c9);
  p = fma(p, r, K.c8);
  p = fma(p, r, K.c7);
  p = fma(p, r, K.c6);
  p = fma(p, r, K.c5);
  p = fma(p, r, K.c4);
  p = fma(p, r, K.c3);
  p = fma(p, r, 0.5);
  return ldexp(fma(r, fma(r, p, 1.0), 1.0), __double2loint(t));
}

}  // namespace astr
