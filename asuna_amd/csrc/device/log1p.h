// log(1 + x) of the denoiser's features.  Plain C++ apart from the reciprocal
// the caller passes, so that it can be evaluated on a CPU.
#pragma once

#include <stdint.h>

namespace ashd {

// log(1 + x) for x >= 0 (or infinity), within 0.54 units in the last place.
// u = 1 + x rounds by c; u = 2^k m with m in [1/sqrt 2, sqrt 2), and
// log m = 2 atanh(s), s = f / (2 + f), f = m - 1, by the series to s^11
// (|s| <= 0.1716: the rest is below 4e-11).  With k = 0, f is x itself.  s keeps
// the remainder of its division, k ln 2 is split so that its first part is exact,
// and the largest terms are added last, with their error.  That holds with rcp one
// unit off.  (The device library's log1pf measures 0.563, mean error 0.1516 as
// here.)  About 45 instructions; that function's 120 were a third of the time of the
// denoiser's first layers.
template <class Rcp> __host__ __device__ inline float log1pPos(float x, Rcp rcp) {
  const float u = 1.0f + x;
  uint32_t bits;
  __builtin_memcpy(&bits, &u, 4);
  const uint32_t mbits = (bits & 0x7fffffu) | 0x3f800000u;
  float m;
  __builtin_memcpy(&m, &mbits, 4);
  const bool high = m > 1.41421356f;
  const int k = int(bits >> 23) - (high ? 126 : 127);
  m = high ? 0.5f * m : m;
  const float f = k ? m - 1.0f : x, c = k ? x - (u - 1.0f) : 0.0f;
  const float kf = float(k);
  const float d = 2.0f + f, dl = f - (d - 2.0f);  // 2 + f = d + dl
  const float r = rcp(d), s = f * r;
  const float sl = __builtin_fmaf(-s, dl, __builtin_fmaf(-s, d, f)) * r;  // f / (2 + f) = s + sl
  const float z = s * s, w = 2.0f * sl, dw = __builtin_fmaf(w, z, w);     // 2 atanh(s + sl) = 2 atanh(s) + 2 sl (1 + z)
  const float p = z * __builtin_fmaf(
                          z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, 1.0f / 11, 1.0f / 9), 1.0f / 7), 1.0f / 5),
                          1.0f / 3);
  const float s2 = 2.0f * s;
  const float kh = kf * 0.693145752f;  // 45426 / 2^16: exact for |k| <= 128
  const float t = kh + s2, tl = s2 - (t - kh);
  // k (ln 2 - 45426 / 2^16) + log(1 + c / u) + what s2 leaves of the series
  const float lo = __builtin_fmaf(kf, 1.42860677e-06f, __builtin_fmaf(s2, p, __builtin_fmaf(c, rcp(u), dw)));
  const float l = t + (tl + lo);
  return x < 5.96046448e-08f || x > 3.40282347e+38f ? x : l;  // below 2^-24 x is nearest; infinity
}

}  // namespace ashd
