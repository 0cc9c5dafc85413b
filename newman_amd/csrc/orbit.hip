// orbit.hip - what a reference's high-precision orbit gives the kernels: the orbit in
// doubles with its remainders, and the series coefficients A, B, C (mandelbrot.cpp:
// 112-131) at the working precision, truncated to doubles.
//
// The coefficients are three linear recurrences with the same factors, Y_i = 2 x_{i-1}
// Y_{i-1} + u_i (u: 1 for A, A_i^2 for B, 2 A_i B_i for C).  One after the other they
// are a chain of 18 products per index, 1.5 us of one host thread (11.8 ms for 8000
// indices, a third of a 38 ms pass on a moved view).  Here each recurrence is cut in
// chunks on three levels of about cbrt(len) each: every chunk's product and its sum
// from 0, the same over the chunks of a group, then the values at each group's and
// each chunk's start, then all values from there, so that the longest chain is 5
// cbrt(len) steps (100 for 8000).  A step is two products and three sums per lane, the
// real part in an even lane and the imaginary part in the odd one beside it.  What
// bounds it is the latency of that arithmetic (carries run through a lane's limbs),
// with a few waves in flight.  The orbit in doubles, a lane per value, took the host
// another 5 ms each for the screening's orbit and the reference's.  precompute() with
// the host's tables and with these (orbit lengths 3000, 8000, 20000, 100000 at 3, 4, 4
// and 8 limbs): 13.1 -> 6.9, 35.5 -> 15.9, 86.1 -> 37.7, 598 -> 237 ms (0.1, 0.2, 0.5
// and 2.8 ms of them the bound below), most of what is left the host's chain of the
// orbit itself.
//
// A chunk's first value comes by another order of operations than the host's chain, so
// its last bits differ (the first chunk's do not).  What is kept of a value is its
// truncation to 53 bits, which the difference changes only where it reaches the value's
// neighbours.  The kernels give each value's distance to those and each chunk's step at
// its start, orbit_tables_hold() (orbit_steps.hpp) bounds the difference along the
// orbit from them, and where the bound does not do the host makes the tables.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "coords.hpp"
#include "orbit.hpp"
#include "orbit_steps.hpp"

namespace nm {

namespace {

// the value of the lane's neighbour (lanes 2 k and 2 k + 1)
__device__ __forceinline__ uint32_t beside(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);  // quad_perm 1, 0, 3, 2
}
__device__ __forceinline__ uint64_t beside(uint64_t v) {
  return (uint64_t)beside((uint32_t)(v >> 32)) << 32 | beside((uint32_t)v);
}
template <int ML>
__device__ __forceinline__ hpd<ML> beside(const hpd<ML>& a) {
  hpd<ML> r;
  r.sign = (int)beside((uint32_t)a.sign);
  r.exp = (int64_t)beside((uint64_t)a.exp);
#pragma unroll
  for (int i = 0; i < ML; i++) r.m[i] = beside(a.m[i]);
  return r;
}

// One pass over a level: chunk q of the n elements, v = factor v + terms for each of
// them in turn.  Values are pairs (re, im); every pointer may be null.
template <int ML>
struct Sweep {
  const hpd<ML>*factor, *u1, *u2;  // terms: u1 + u2
  int twice;                       // the factor stands for twice its value
  int one;                         // a term 1 for each element
  int n, chunk, L;
  const hpd<ML>* start;  // each chunk's first v (null: first)
  int first;
  hpd<ML>*end, *before, *after;  // v at a chunk's end; at each element, before or after its step
  hpd<ML>* product;              // products of the factors (grid y = 1): no terms, from 1
};

template <int ML>
__global__ __launch_bounds__(64) void k_sweep(Sweep<ML> w) {
  const int t = blockIdx.x * 64 + threadIdx.x, part = t & 1, chunks = (w.n + w.chunk - 1) / w.chunk;
  const bool live = (t >> 1) < chunks, product = blockIdx.y != 0;
  const int q = live ? t >> 1 : chunks - 1;
  const int e0 = q * w.chunk, e1 = min(w.n, e0 + w.chunk);  // chunks * chunk < n + chunk: in 32 bits
  hpd<ML> v = hpd_small<ML>(part == 0 ? (product ? 1 : w.first) : 0);
  if (w.start && !product) v = w.start[2 * q + part];
  hpd<ML> fr = w.factor[2 * e0], fi = w.factor[2 * e0 + 1];
  for (int e = e0; e < e1; e++) {
    const int nx = min(e + 1, e1 - 1);
    const hpd<ML> nr = w.factor[2 * nx], ni = w.factor[2 * nx + 1];  // the next step's
    if (w.before && live && !product) w.before[2 * e + part] = v;
    const hpd<ML> o = beside(v);
    const size_t u = 2 * (size_t)e + part;
    const hpd<ML> s = sweep_part(part, fr, fi, v, o, w.twice != 0, !product && w.one,
                                 product || !w.u1 ? nullptr : w.u1 + u, product || !w.u2 ? nullptr : w.u2 + u, w.L);
    v = s;
    if (w.after && live && !product) w.after[2 * e + part] = v;
    fr = nr;
    fi = ni;
  }
  if (!live) return;
  if (product) w.product[2 * q + part] = v;
  else if (w.end) w.end[2 * q + part] = v;
}

// the terms of B (bs null) or C at i = 1 .. n (terms_part)
template <int ML>
__global__ __launch_bounds__(64) void k_terms(const hpd<ML>* as, const hpd<ML>* bs, int n, int L, hpd<ML>* u1,
                                              hpd<ML>* u2) {
  const int t = blockIdx.x * 64 + threadIdx.x, part = t & 1, e = t >> 1;
  if (e >= n) return;
  hpd<ML> p, s;
  terms_part(part, as + 2 * (e + 1), bs ? bs + 2 * (e + 1) : (const hpd<ML>*)nullptr, L, p, s);
  u1[t] = p;
  u2[t] = s;
}

// the factors' orbit in doubles: Zd[k + 1] = nearest(x[k]), Xlo[k] = nearest(x[k] - Zd[k + 1])
template <int ML>
__global__ __launch_bounds__(64) void k_orbit(const hpd<ML>* x, int len, int L, double* Zd, double* Xlo) {
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t < 2) Zd[t] = 0.0;
  if (t >= 2 * (len + 1)) return;
  const hpd<ML> v = x[t];
  const double d = hpd_nearest(v, L);
  Zd[t + 2] = d;
  if (t < 2 * len) Xlo[t] = hpd_nearest(hpd_add(v, hpd_from_d<ML>(d), -1, L), L);
}

// Y_0 .. Y_{len - 1} truncated to doubles (mpf_get_d), as mantissa and exponent, and
// with the bits that the truncation hangs on; for chunks 1 .. n1 - 1 the exponents of
// the step from the previous chunk's end to their start
template <int ML>
__global__ __launch_bounds__(64) void k_emit(const hpd<ML>* y, int len, int L, const hpd<ML>* starts,
                                             const hpd<ML>* ends, int n1, double* d, double* m, int32_t* e,
                                             uint16_t* run, int32_t* gap) {
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t < 2 * (n1 - 1)) {
    const hpd<ML> g = hpd_add(starts[t + 2], ends[t], -1, L);
    gap[t] = g.sign ? (int32_t)g.exp : kFxZeroExp;
  }
  if (t >= 2 * len) return;
  const hpd<ML> v = y[t];
  d[t] = hpd_get_d(v);
  const double f = v.sign * ldexp((double)(v.m[ML - 1] >> 11), -53);
  m[t] = v.sign ? f : 0.0;
  e[t] = v.sign ? (int32_t)v.exp : kFxZeroExp;
  run[t] = hpd_run(v, L);
}

template <int ML>
__global__ __launch_bounds__(64) void k_first(hpd<ML>* y, int first) {
  if (threadIdx.x < 2) y[threadIdx.x] = hpd_small<ML>(threadIdx.x == 0 ? first : 0);
}

template <int ML>
void sweep(hipStream_t s, const Sweep<ML>& w) {
  const int chunks = (w.n + w.chunk - 1) / w.chunk;
  hipLaunchKernelGGL(k_sweep<ML>, dim3((unsigned)((2 * chunks + 63) / 64), w.product ? 2 : 1), dim3(64), 0, s, w);
}

}  // namespace

OrbitTables::~OrbitTables() { release(); }

void OrbitTables::release() {
  if (buf_) (void)hipFree(buf_);
  buf_ = nullptr;
  bytes_ = 0;
}

bool OrbitTables::room(size_t bytes) {
  if (bytes <= bytes_) return true;
  release();
  if (hipMalloc((void**)&buf_, bytes) != hipSuccess) {
    (void)hipGetLastError();
    buf_ = nullptr;
    return false;
  }
  bytes_ = bytes;
  return true;
}

template <int ML>
bool OrbitTables::go(void* stream, const HpVal* x, int len, int L, bool series, SaReferenceHost& r) {
  typedef hpd<ML> V;
  hipStream_t s = (hipStream_t)stream;
  const int n = len - 1;  // steps of the recurrences
  const int c = std::max(1, (int)std::ceil(std::cbrt((double)n)));
  const int n1 = (n + c - 1) / c, n2 = (n1 + c - 1) / c;
  size_t off = 0;
  auto place = [&](size_t bytes) {
    const size_t o = off;
    off += (bytes + 255) & ~(size_t)255;
    return o;
  };
  const size_t count = 2 * (size_t)len;
  const size_t ox = place((count + 2) * sizeof(V)), oz = place((count + 4) * 8), ol = place(count * 8);
  size_t oy[3], od[3], om[3], oe[3], ou[2], os[6], orun = 0, ogap = 0;
  const size_t gaps = 2 * (size_t)(n1 - 1);  // of each series
  if (series) {
    for (int k = 0; k < 3; k++) {
      oy[k] = place(count * sizeof(V));
      od[k] = place(count * 8);
      om[k] = place(count * 8);
      oe[k] = place(count * 4);
    }
    for (size_t& o : ou) o = place(count * sizeof(V));
    for (int k = 0; k < 6; k++) os[k] = place(2 * (size_t)(k < 3 ? n1 : n2) * sizeof(V));  // products, ends, starts
    orun = place(3 * count * 2);
    ogap = place(3 * gaps * 4);
  }
  if (!room(off)) return false;
  V* dx = (V*)(buf_ + ox);
  std::vector<V> hx(count + 2);
  std::vector<uint16_t> run;
  std::vector<int32_t> gap;
  // also where a table's allocation throws: the copies out of and into them are over first
  struct Wait {
    hipStream_t s;
    ~Wait() { (void)hipStreamSynchronize(s); }
  } wait{s};
  for (size_t k = 0; k < count + 2; k++) hx[k] = hpd_load<ML>(x[k]);
  bool ok = hipMemcpyAsync(dx, hx.data(), hx.size() * sizeof(V), hipMemcpyHostToDevice, s) == hipSuccess;
  hipLaunchKernelGGL(k_orbit<ML>, dim3((unsigned)((count + 2 + 63) / 64)), dim3(64), 0, s, (const V*)dx, len, L,
                     (double*)(buf_ + oz), (double*)(buf_ + ol));
  if (series) {
    V *P1 = (V*)(buf_ + os[0]), *E1 = (V*)(buf_ + os[1]), *S1 = (V*)(buf_ + os[2]);
    V *P2 = (V*)(buf_ + os[3]), *E2 = (V*)(buf_ + os[4]), *S2 = (V*)(buf_ + os[5]);
    V *u1 = (V*)(buf_ + ou[0]), *u2 = (V*)(buf_ + ou[1]);
    const unsigned blocks = (unsigned)((count + 63) / 64);
    for (int k = 0; k < 3; k++) {
      V* y = (V*)(buf_ + oy[k]);
      const V *t1 = k ? u1 : nullptr, *t2 = k ? u2 : nullptr;
      if (k)
        hipLaunchKernelGGL(k_terms<ML>, dim3((unsigned)((2 * (size_t)n + 63) / 64)), dim3(64), 0, s,
                           (const V*)(buf_ + oy[0]), k == 2 ? (const V*)(buf_ + oy[1]) : (const V*)nullptr, n, L, u1, u2);
      const int one = k == 0, first = k == 0;
      V *p1 = k == 0 ? P1 : nullptr, *p2 = k == 0 ? P2 : nullptr;  // the products are the same for all three
      sweep<ML>(s, {dx, t1, t2, 1, one, n, c, L, nullptr, 0, E1, nullptr, nullptr, p1});
      sweep<ML>(s, {P1, E1, nullptr, 0, 0, n1, c, L, nullptr, 0, E2, nullptr, nullptr, p2});
      sweep<ML>(s, {P2, E2, nullptr, 0, 0, n2, n2, L, nullptr, first, nullptr, S2, nullptr, nullptr});
      sweep<ML>(s, {P1, E1, nullptr, 0, 0, n1, c, L, S2, 0, nullptr, S1, nullptr, nullptr});
      sweep<ML>(s, {dx, t1, t2, 1, one, n, c, L, S1, 0, E1, nullptr, y + 2, nullptr});
      hipLaunchKernelGGL(k_first<ML>, dim3(1), dim3(64), 0, s, y, first);
      hipLaunchKernelGGL(k_emit<ML>, dim3(blocks), dim3(64), 0, s, (const V*)y, len, L, (const V*)S1, (const V*)E1, n1,
                         (double*)(buf_ + od[k]), (double*)(buf_ + om[k]), (int32_t*)(buf_ + oe[k]),
                         (uint16_t*)(buf_ + orun) + k * count, (int32_t*)(buf_ + ogap) + k * gaps);
    }
  }
  ok = ok && hipGetLastError() == hipSuccess;
  auto fetch = [&](auto& v, size_t o, size_t size) {
    v.resize(size);
    ok = ok && hipMemcpyAsync(v.data(), buf_ + o, size * sizeof(v[0]), hipMemcpyDeviceToHost, s) == hipSuccess;
  };
  fetch(r.Zd, oz, count + 4);
  fetch(r.Xlo, ol, count);
  if (series) {
    std::vector<double>*fd[3] = {&r.A, &r.B, &r.C}, *fm[3] = {&r.Am, &r.Bm, &r.Cm};
    std::vector<int32_t>* fe[3] = {&r.Ae, &r.Be, &r.Ce};
    for (int k = 0; k < 3; k++) {
      fetch(*fd[k], od[k], count);
      fetch(*fm[k], om[k], count);
      fetch(*fe[k], oe[k], count);
    }
    fetch(run, orun, 3 * count);
    fetch(gap, ogap, 3 * gaps);
  }
  ok = hipStreamSynchronize(s) == hipSuccess && ok;
  if (!ok) (void)hipGetLastError();
  if (bytes_ > kKeep) release();
  if (!ok || !series) return ok;
  bool real = true;
  for (size_t k = 1; k < count && real; k += 2) real = x[k].sign == 0;
  return orbit_tables_hold(r.Zd.data(), len, L, c, real, {r.Ae.data(), r.Be.data(), r.Ce.data()},
                           {run.data(), run.data() + count, run.data() + 2 * count},
                           {gap.data(), gap.data() + gaps, gap.data() + 2 * gaps});
}

bool OrbitTables::make(void* stream, const HpVal* x, int len, int L, bool series, SaReferenceHost& r) {
  if (len < kMinLen || L > kMaxLimbs) return false;
  if (L <= 4) return go<4>(stream, x, len, L, series, r);
  if (L <= 6) return go<6>(stream, x, len, L, series, r);
  if (L <= 8) return go<8>(stream, x, len, L, series, r);
  return go<kMaxLimbs>(stream, x, len, L, series, r);
}

}  // namespace nm
