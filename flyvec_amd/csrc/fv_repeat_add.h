// n sequential fp32 additions of the same value, in fewer than n steps, bit for bit.
//
// The reference adds 1/f onto ds[h][i] once per occurrence of token i in the windows neuron h
// won (flyvec/src/cuda_funcs.cu:657-672); for a frequent token that is thousands of additions
// onto one element.  The result v_n of  v_{k+1} = fl(v_k + f)  is reproduced exactly by noting
// that while v stays inside one binade (same sign and exponent) its bit pattern moves by a
// constant number of ulps per addition: the exact sum is (m + q + r) ulps with m the integer
// significand of v and q + r = f / ulp, and round-to-nearest turns the fraction r into the same
// 0 or 1 every time.  The one exception, r = 1/2 exactly (ties-to-even looks at the parity of
// m + q), settles after one addition, because every tie result is even.  So: take three real
// additions; if all three results share a binade and the two differences are equal, the state
// is steady and the remaining additions inside the binade are one integer multiply-add on the
// bit pattern (stopping short of the binade's ends); binade crossings, including the passage
// through zero, are taken with real additions.  Fewer than FV_REPEAT_JUMP additions are simply made, eight to a turn: a
// turn that looks for the steady state divides, and the sums of an ordinary minibatch have a few additions to a few dozen.
// Where the line lies, in us of a whole step with 4 (as good as always looking), 32, 48, 64, 96, 256: K = 400, V = 20000,
// B = 10000 51.9 51.6 51.6 51.6 51.6 51.7, with the anti-Hebbian term 68.7 68.3 68.4 68.5 68.5 68.5; K = 209, V = 7919, B =
// 3001 26.8 26.5 26.4 26.4 26.4 26.5; K = 100, V = 2000, B = 10000 38.5 38.5 38.6 38.7 38.9 39.1; K = 60, V = 1000, B =
// 16000 42.0 42.2 42.2 42.3 42.7 -; K = 1000, V = 50000, B = 50000 406.8 404.8 404.6 404.7 404.8 -. (Replays of the launch by itself
// say otherwise: the elements it then finds are sentinels.)  Compiles for the host too, where the tests check it against the plain loop.
#pragma once

#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define FV_HD __host__ __device__ __forceinline__
#else
#define FV_HD static inline
#endif

FV_HD uint32_t fv_f2u(float x) {
  uint32_t u;
  memcpy(&u, &x, sizeof u);
  return u;
}

FV_HD float fv_u2f(uint32_t u) {
  float x;
  memcpy(&x, &u, sizeof x);
  return x;
}

// One rounded addition; never fused with a neighbouring multiply.
FV_HD float fv_add1(float a, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __fadd_rn(a, b);
#else
  volatile float r = a + b;
  return r;
#endif
}

#ifndef FV_REPEAT_JUMP
#define FV_REPEAT_JUMP 48u
#endif

FV_HD float fv_add_repeat(float v, float f, uint32_t n) {
  while (n >= FV_REPEAT_JUMP) {
    const float v1 = fv_add1(v, f), v2 = fv_add1(v1, f), v3 = fv_add1(v2, f);
    n -= 3;
    v = v3;
    const uint32_t b1 = fv_f2u(v1), b2 = fv_f2u(v2);
    uint32_t b3 = fv_f2u(v3);
    if (b3 == b2) return v;  // f is absorbed: every further addition returns v again
    const uint32_t se = b1 >> 23;  // sign and exponent
    if (se == (b2 >> 23) && se == (b3 >> 23) && (se & 0xffu) != 0u && (se & 0xffu) != 0xffu) {
      const int32_t d1 = (int32_t)(b2 - b1), d2 = (int32_t)(b3 - b2);
      if (d1 == d2) {
        // the bit pattern grows when the magnitude grows, whatever the sign
        const uint32_t mant = b3 & 0x7fffffu;
        // ulps left inside the binade. Shrinking magnitudes stop one ulp short of the binade's
        // lowest value: a sum that rounds onto it may lie below it, where the spacing is finer.
        const uint32_t room = d1 > 0 ? 0x7fffffu - mant : (mant ? mant - 1u : 0u);
        const uint32_t step = d1 > 0 ? (uint32_t)d1 : (uint32_t)(-d1);
        uint32_t k = room / step;
        if (k > n) k = n;
        b3 = d1 > 0 ? b3 + k * step : b3 - k * step;
        v = fv_u2f(b3);
        n -= k;
      }
    }
  }
  for (; n >= 8; n -= 8) {
    v = fv_add1(fv_add1(fv_add1(fv_add1(v, f), f), f), f);
    v = fv_add1(fv_add1(fv_add1(fv_add1(v, f), f), f), f);
  }
  if (n & 4u) v = fv_add1(fv_add1(fv_add1(fv_add1(v, f), f), f), f);
  if (n & 2u) v = fv_add1(fv_add1(v, f), f);
  if (n & 1u) v = fv_add1(v, f);
  return v;
}
