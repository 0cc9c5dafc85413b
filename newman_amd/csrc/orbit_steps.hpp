// orbit_steps.hpp - the arithmetic of the device's reference tables (orbit.hip), for
// the host too, where a check runs the same passes over an orbit: a recurrence's step,
// its terms, what a value's doubles hang on, and the bound on what another order of
// operations can change.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "coords.hpp"

namespace nm {

template <int ML>
__host__ __device__ __forceinline__ hpd<ML> hpd_small(int v) {  // 0 or 1
  hpd<ML> r;
  r.sign = v;
  r.exp = v;
  for (int i = 0; i < ML; i++) r.m[i] = 0;
  if (v) r.m[ML - 1] = 1ull << 63;
  return r;
}

// one part (0 real, 1 imaginary) of factor v (+ 1) + u1 + u2: v that part of the value,
// o the other; twice: the factor stands for twice its value; u1, u2 may be null
template <int ML>
__host__ __device__ __forceinline__ hpd<ML> sweep_part(int part, const hpd<ML>& fr, const hpd<ML>& fi,
                                                       const hpd<ML>& v, const hpd<ML>& o, bool twice, bool one,
                                                       const hpd<ML>* u1, const hpd<ML>* u2, int L) {
  hpd<ML> s = hpd_add(hpd_mul(fr, v, L), hpd_mul(fi, o, L), part == 0 ? -1 : 1, L);
  if (twice && s.sign) s.exp++;
  if (one && part == 0) s = hpd_add(s, hpd_small<ML>(1), 1, L);
  if (u1) s = hpd_add(s, *u1, 1, L);
  if (u2) s = hpd_add(s, *u2, 1, L);
  return s;
}

// one part of the terms of B (b null: A^2) or C (2 A B), in the order the recurrence
// adds them: real parts a_r b_r and -a_i b_i, imaginary a_r b_i and a_i b_r (for A^2
// the one product doubled); a and b point at (re, im)
template <int ML>
__host__ __device__ __forceinline__ void terms_part(int part, const hpd<ML>* a, const hpd<ML>* b, int L, hpd<ML>& u1,
                                                    hpd<ML>& u2) {
  const hpd<ML>* w = b ? b : a;
  u1 = hpd_mul(a[0], w[part], L);
  u2 = hpd_mul(a[1], w[1 - part], L);
  if (part == 0) u2.sign = -u2.sign;
  if (b) {
    if (u1.sign) u1.exp++;
    if (u2.sign) u2.exp++;
  } else if (part == 1) {
    if (u1.sign) u1.exp++;
    u2 = hpd_small<ML>(0);
  }
}

// The run of equal bits behind a value's first 53: with r of them the value is at
// least 2^(exp - 54 - r) from any other truncation to 53 bits.  kNoRun: a zero, or
// equal bits down to the last one.
constexpr uint16_t kNoRun = 0xffff;
template <int ML>
__host__ __device__ __forceinline__ uint16_t hpd_run(const hpd<ML>& v, int L) {
  if (v.sign == 0) return kNoRun;
  const uint64_t flip = (v.m[ML - 1] >> 10) & 1 ? ~0ull : 0ull;  // the first bit behind
  const uint64_t low = (v.m[ML - 1] ^ flip) & ((1ull << 11) - 1);
  if (low) return (uint16_t)(hpd_clz(low) - 53);
  int run = 11;
  bool on = true;
  for (int i = ML - 2; i >= 0; i--)
    if (on && i >= ML - L) {
      const uint64_t x = v.m[i] ^ flip;
      run += hpd_clz(x);
      on = x == 0;
    }
  return on ? kNoRun : (uint16_t)run;
}

// Whether the doubles that the device made of A, B and C are the host's.  Both follow
// Y_i+1 = 2 x_i Y_i + u_i, each product and sum truncated at L limbs, but from chunk 1
// on the device starts every chunk at a value made by way of the chunks' products and
// sums.  Let D_i bound |device - host|:
//   * up to the end of chunk 0 the operations are the same: D = 0;
//   * where a chunk starts, D grows by the distance from the previous chunk's end to
//     the value the chunk starts at, which the device measures (gap: its exponents);
//   * a step takes D to 2 |x| D, plus what the two u differ by (B: 2 |A| D_A + D_A^2,
//     C: 2 (|A| D_B + |B| D_A + D_A D_B)), plus the truncations of both: a part takes
//     two products, their sum and up to two terms, each off by less than e = 2^(1 - 64
//     L) of itself, in all 5 W + 3 U of e with W = 2 |x| (|Y| + D), U >= |u|; both
//     sides and both parts 16 (W + U) e at the most.
// A double is the host's where D is below the distance to its neighbours (hpd_run).
// D_i is kept in units of 2^(E_i) e, E_i the larger exponent of Y_i's parts.  What
// cancels in a step raises D against Y_i+1 as far as it does the true error, so no
// assumption about the orbit is left.  real: the orbit lies on the real axis and every
// imaginary part is an exact zero.  Zd: the orbit as the kernels read it (Zd[i + 1] = x_i).
// trace (a check's): 3 len values, D of every index as far as the bound does.
// It is 0.2 ms of one host thread for a length of 8000, 2.8 for 100,000.
inline bool orbit_tables_hold(const double* Zd, int len, int L, int chunk, bool real, const int32_t* const (&ex)[3],
                              const uint16_t* const (&run)[3], const int32_t* const (&gap)[3],
                              double* trace = nullptr) {
  auto pow2 = [](int64_t k) {  // rounded up below 2^-1000, infinite past 2^1000
    if (k > 1000) return HUGE_VAL;
    const uint64_t u = (uint64_t)(std::max<int64_t>(k, -1000) + 1023) << 52;
    double d;
    std::memcpy(&d, &u, 8);
    return d;
  };
  constexpr double kRoot2 = 1.4142136, kRound = 16.0;
  const int64_t unit = 64 * (int64_t)L - 1;  // e = 2^-unit
  const double e = pow2(-unit);
  double d[3] = {0.0, 0.0, 0.0};
  int64_t E[3] = {0, 0, 0};
  auto larger = [&](int s, int i) { return std::max(ex[s][2 * (size_t)i], ex[s][2 * (size_t)i + 1]); };
  for (int i = chunk; i + 1 < len; i++) {
    const bool start = i % chunk == 0;
    const double zx = Zd[2 * (size_t)(i + 1)], zy = Zd[2 * (size_t)(i + 1) + 1];
    const double f = std::max(2.0 * std::sqrt(zx * zx + zy * zy), 0x1p-480);  // above a square that underflows
    int64_t E1[3];
    double n[3];
    for (int s = 0; s < 3; s++) {
      if (i == chunk) E[s] = larger(s, i);
      E1[s] = larger(s, i + 1);
      if (E[s] == kFxZeroExp || E1[s] == kFxZeroExp) return false;
      double own = d[s];
      if (start)
        for (int p = 0; p < 2; p++) {
          const int32_t g = gap[s][2 * (size_t)(i / chunk - 1) + p];
          if (g != kFxZeroExp) own += pow2(g - E[s] + unit);
        }
      double u, du;  // |u| and the difference of the two u, in the units of Y_i+1
      if (s == 0) {
        u = pow2(-E1[0]);
        du = 0.0;
      } else if (s == 1) {
        const double q = pow2(2 * E1[0] - E1[1]);
        u = 2.0 * q;
        du = q * n[0] * (2.0 * kRoot2 + n[0] * e);
      } else {
        const double q = pow2(E1[0] + E1[1] - E1[2]);
        u = 4.0 * q;
        du = 2.0 * q * (kRoot2 * (n[0] + n[1]) + n[0] * n[1] * e);
      }
      const double g = f * pow2(E[s] - E1[s]);
      n[s] = (g * own + kRound * (g * (kRoot2 + own * e) + u) + du) * (1.0 + 0x1p-40);  // rounded up
      if (!(n[s] < 0x1p900)) return false;
      if (trace) trace[3 * (size_t)(i + 1) + s] = n[s];
      for (int p = 0; p < (real ? 1 : 2); p++) {
        const size_t t = 2 * (size_t)(i + 1) + p;
        if (run[s][t] == kNoRun) return false;
        const int64_t room = (int64_t)ex[s][t] - E1[s] - 54 - run[s][t] + unit;
        if (room <= 0 || n[s] >= pow2(std::min<int64_t>(room, 1000))) return false;
      }
    }
    for (int s = 0; s < 3; s++) {
      d[s] = n[s];
      E[s] = E1[s];
    }
  }
  return true;
}

}  // namespace nm
