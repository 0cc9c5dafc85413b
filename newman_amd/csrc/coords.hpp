// coords.hpp - the high-precision pixel map of computeRow / findProbe / pointAt
// (mandelbrot.cpp:271, 275, 86-87, 287-288), re = center.re + k * sz.re, im =
// center.im + j * sz.im, each step truncated at the working precision, for one
// column or row: the device makes a frame's coordinate tables with it.  The same
// truncating arithmetic as hpfloat.cpp on mantissas of a fixed number of limbs;
// compiled for the host too, where a check compares it with hpfloat.cpp.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "engine.hpp"

namespace nm {

// value = sign * 0.m * 2^exp, m top-aligned: m[ML - 1] is the most significant limb
// (its top bit set unless the value is 0), unused low limbs are 0
template <int ML>
struct hpd {
  int sign;
  int64_t exp;
  uint64_t m[ML];
};

template <int ML>
__host__ __device__ inline hpd<ML> hpd_load(const HpVal& v) {
  hpd<ML> r;
  r.sign = v.sign;
  r.exp = v.exp;
  for (int i = 0; i < ML; i++) {
    const int s = v.L - ML + i;
    r.m[i] = s >= 0 && v.sign ? v.m[s] : 0;
  }
  return r;
}

// the top L limbs
template <int ML>
__host__ __device__ inline void hpd_trunc(hpd<ML>& r, int L) {
  for (int i = 0; i < ML; i++)
    if (i < ML - L) r.m[i] = 0;
}

__host__ __device__ inline int hpd_clz(uint64_t x) { return x ? __builtin_clzll(x) : 64; }

// a * k at L limbs
template <int ML>
__host__ __device__ inline hpd<ML> hpd_mul_si(const hpd<ML>& a, long k, int L) {
  hpd<ML> r;
  r.sign = 0;
  r.exp = 0;
  for (int i = 0; i < ML; i++) r.m[i] = 0;
  if (a.sign == 0 || k == 0) return r;
  const uint64_t u = k < 0 ? (uint64_t)(-k) : (uint64_t)k;  // |k| < 2^31: frame indices
  uint64_t p[ML + 1];
  unsigned __int128 c = 0;
  for (int i = 0; i < ML; i++) {
    c += (unsigned __int128)a.m[i] * u;
    p[i] = (uint64_t)c;
    c >>= 64;
  }
  p[ML] = (uint64_t)c;
  const int lead = hpd_clz(p[ML]);  // 33 .. 64: the product is at least the mantissa
  for (int i = 0; i < ML; i++) r.m[i] = lead == 64 ? p[i] : (p[i + 1] << lead) | (p[i] >> (64 - lead));
  r.sign = k < 0 ? -a.sign : a.sign;
  r.exp = a.exp + 64 - lead;
  hpd_trunc(r, L);
  return r;
}

// a + s b at L limbs (s = 1 or -1)
template <int ML>
__host__ __device__ inline hpd<ML> hpd_add(const hpd<ML>& a, const hpd<ML>& b, int s, int L) {
  const int sb = s * b.sign;
  if (sb == 0 || a.sign == 0) {
    hpd<ML> r = sb == 0 ? a : b;
    if (sb != 0) r.sign = sb;
    hpd_trunc(r, L);
    return r;
  }
  bool less = a.exp < b.exp;  // |a| < |b|
  if (a.exp == b.exp)
    for (int i = 0; i < ML; i++)  // the last differing limb decides
      if (a.m[i] != b.m[i]) less = a.m[i] < b.m[i];
  constexpr int N = ML + 3;  // two guard limbs below, one carry limb above
  uint64_t X[N], Y[N];
  X[0] = X[1] = X[N - 1] = Y[0] = Y[1] = Y[N - 1] = 0;
  for (int i = 0; i < ML; i++) {
    X[i + 2] = less ? b.m[i] : a.m[i];
    Y[i + 2] = less ? a.m[i] : b.m[i];
  }
  const int64_t ex = less ? b.exp : a.exp, sh = ex - (less ? a.exp : b.exp);
  const int sx = less ? sb : a.sign;
  uint64_t lost = 0;  // bits of Y shifted out
  const int64_t ls = sh / 64 < N ? sh / 64 : N;
  for (int64_t t = 0; t < ls; t++) {
    lost |= Y[0];
    for (int i = 0; i + 1 < N; i++) Y[i] = Y[i + 1];
    Y[N - 1] = 0;
  }
  const int bs = (int)(sh % 64);
  if (bs) {
    lost |= Y[0] << (64 - bs);
    for (int i = 0; i + 1 < N; i++) Y[i] = (Y[i] >> bs) | (Y[i + 1] << (64 - bs));
    Y[N - 1] >>= bs;
  }
  if (a.sign == sb) {
    unsigned __int128 c = 0;
    for (int i = 0; i < N; i++) {
      c += (unsigned __int128)X[i] + Y[i];
      X[i] = (uint64_t)c;
      c >>= 64;
    }
  } else {
    uint64_t br = lost ? 1 : 0;  // exact = X - Y - fraction: its floor borrows one
    for (int i = 0; i < N; i++) {
      const unsigned __int128 d = (unsigned __int128)X[i] - Y[i] - br;
      X[i] = (uint64_t)d;
      br = (uint64_t)(d >> 127);
    }
  }
  hpd<ML> r;
  const int64_t e = ex + 64;
  int up = 0;
  while (up < N && X[N - 1] == 0) {
    for (int i = N - 1; i > 0; i--) X[i] = X[i - 1];
    X[0] = 0;
    up++;
  }
  const int lead = up == N ? 0 : hpd_clz(X[N - 1]);
  for (int i = 0; i < ML; i++) r.m[i] = lead ? (X[i + 3] << lead) | (X[i + 2] >> (64 - lead)) : X[i + 3];
  r.sign = up == N ? 0 : sx;
  r.exp = up == N ? 0 : e - 64 * (int64_t)up - lead;
  hpd_trunc(r, L);
  return r;
}

// bits of the mantissa that a double at exponent e holds (fewer than 53 below 2^-1021)
__host__ __device__ inline int hpd_keep(int64_t e) { return e - 53 < -1074 ? (int)(e + 1074) : 53; }

// truncated to a double (mpf_get_d)
template <int ML>
__host__ __device__ inline double hpd_get_d(const hpd<ML>& a) {
  if (a.sign == 0) return 0.0;
  if (a.exp > 1024) return a.sign * HUGE_VAL;
  const int keep = hpd_keep(a.exp);
  if (keep <= 0) return 0.0 * a.sign;
  const double d = ldexp((double)(a.m[ML - 1] >> (64 - keep)), (int)(a.exp - keep));
  return a.sign < 0 ? -d : d;
}

// the nearest double to what truncation to a double leaves (ties to even)
template <int ML>
__host__ __device__ inline double hpd_rest(const hpd<ML>& a) {
  if (a.sign == 0 || a.exp > 1024) return 0.0;
  const int cut = hpd_keep(a.exp);
  uint64_t w[ML];
  for (int i = 0; i < ML; i++) w[i] = a.m[i];
  if (cut > 0) w[ML - 1] &= (1ull << (64 - cut)) - 1ull;
  int64_t e = a.exp;
  int up = 0;
  while (up < ML && w[ML - 1] == 0) {
    for (int i = ML - 1; i > 0; i--) w[i] = w[i - 1];
    w[0] = 0;
    up++;
  }
  if (up == ML) return 0.0;
  const int lead = hpd_clz(w[ML - 1]);
  if (lead) {
    for (int i = ML - 1; i > 0; i--) w[i] = (w[i] << lead) | (w[i - 1] >> (64 - lead));
    w[0] <<= lead;
  }
  e -= 64 * (int64_t)up + lead;
  const int keep = hpd_keep(e);
  if (keep <= 0) return 0.0;
  uint64_t q = w[ML - 1] >> (64 - keep);
  const uint64_t half = 1ull << (63 - keep), low = w[ML - 1] & (2 * half - 1);
  uint64_t below = low & (half - 1);
  for (int i = 0; i < ML - 1; i++) below |= w[i];
  if ((low & half) && (below || (q & 1))) q++;
  const double d = ldexp((double)q, (int)(e - keep));
  return a.sign < 0 ? -d : d;
}

// a * b at L limbs
template <int ML>
__host__ __device__ inline hpd<ML> hpd_mul(const hpd<ML>& a, const hpd<ML>& b, int L) {
  hpd<ML> r;
  r.sign = a.sign * b.sign;
  uint64_t t[2 * ML];
#pragma unroll
  for (int i = 0; i < 2 * ML; i++) t[i] = 0;
#pragma unroll
  for (int i = 0; i < ML; i++) {
    unsigned __int128 c = 0;
#pragma unroll
    for (int j = 0; j < ML; j++) {
      c += (unsigned __int128)a.m[i] * b.m[j] + t[i + j];
      t[i + j] = (uint64_t)c;
      c >>= 64;
    }
    t[i + ML] = (uint64_t)c;
  }
  const int lead = t[2 * ML - 1] >> 63 ? 0 : 1;  // both mantissas are at least 1/2
#pragma unroll
  for (int i = 0; i < ML; i++)
    r.m[i] = r.sign == 0 ? 0 : lead ? (t[ML + i] << 1) | (t[ML + i - 1] >> 63) : t[ML + i];
  r.exp = r.sign == 0 ? 0 : a.exp + b.exp - lead;
  hpd_trunc(r, L);
  return r;
}

// a double as it is
template <int ML>
__host__ __device__ inline hpd<ML> hpd_from_d(double d) {
  hpd<ML> r;
  int e = 0;
  const bool zero = d == 0.0 || !(fabs(d) <= 1.7976931348623157e308);
  const double f = zero ? 0.0 : frexp(fabs(d), &e);
  for (int i = 0; i < ML; i++) r.m[i] = 0;
  r.m[ML - 1] = (uint64_t)ldexp(f, 64);
  r.exp = zero ? 0 : e;
  r.sign = zero ? 0 : d < 0.0 ? -1 : 1;
  return r;
}

// the nearest double (ties to even), by way of the truncated one
template <int ML>
__host__ __device__ inline double hpd_nearest(const hpd<ML>& a, int L) {
  const double t = hpd_get_d(a);
  if (a.sign == 0 || !(fabs(t) <= 1.7976931348623157e308)) return t;
  const hpd<ML> r = hpd_add(a, hpd_from_d<ML>(t), -1, L);
  if (r.sign == 0) return t;
  union {
    double d;
    uint64_t u;
  } up, low;
  low.d = t;
  if (t == 0.0) up.u = 1ull | (a.sign < 0 ? 1ull << 63 : 0);
  else up.u = low.u + 1;  // one step away from zero
  const hpd<ML> half = hpd_from_d<ML>((up.d - t) * 0.5);
  int c = r.exp > half.exp ? 1 : r.exp < half.exp ? -1 : 0;
  if (c == 0)
    for (int i = 0; i < ML; i++)  // the last differing limb decides
      if (r.m[i] != half.m[i]) c = r.m[i] > half.m[i] ? 1 : -1;
  return c > 0 ? up.d : c < 0 ? t : (low.u & 1) ? up.d : t;
}

// the coordinate of offset k: center + k * size at L limbs
template <int ML>
__host__ __device__ inline hpd<ML> hpd_pixel(const HpVal& center, const HpVal& size, long k, int L) {
  return hpd_add(hpd_load<ML>(center), hpd_mul_si(hpd_load<ML>(size), k, L), 1, L);
}

// The tables of `frames` frames of nr x nc: column tables at t (frame after frame,
// nc each), row tables behind them.  Plain path (series false): the truncated
// coordinate in hi and its remainder in lo; series path: the truncated difference
// from the reference point in hi.
struct CoordTables {
  double *chi, *clo, *rhi, *rlo;
};
// returns 0, or 1 after a launch error; `hp` holds one FrameHp per frame, in device
// memory (hp_dev) or, for a single frame, by value (hp_one)
int coords_launch(void* stream, const FrameHp* hp_one, const FrameHp* hp_dev, int frames, int nr, int nc, int limbs,
                  bool series, CoordTables t);

}  // namespace nm
