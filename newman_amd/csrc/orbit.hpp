// orbit.hpp - a reference's tables from its high-precision orbit, on the device (see
// orbit.hip).
#pragma once
#include <cstddef>
#include <cstdint>

#include "engine.hpp"

namespace nm {

class OrbitTables {
 public:
  static constexpr int kMaxLimbs = 16;
  // a precompute of length 512 takes 1.34 ms with the host's tables and 1.03 with these,
  // 1024 2.69 and 1.43; 256 0.67 and 0.80 (4 limbs)
  static constexpr int kMinLen = 1024;
  // Zd and Xlo of r, and with `series` A .. Ce, for the orbit x (2 (len + 1) values of
  // L limbs, real and imaginary parts in turn).  False where the host has to make
  // them (r may then be partly filled): more than kMaxLimbs limbs, an orbit shorter
  // than kMinLen, no memory, or coefficients whose doubles the order of operations
  // could change (orbit_tables_hold).
  bool make(void* stream, const HpVal* x, int len, int L, bool series, SaReferenceHost& r);
  ~OrbitTables();

 private:
  static constexpr size_t kKeep = (size_t)256 << 20;  // device memory kept between calls
  char* buf_ = nullptr;
  size_t bytes_ = 0;
  template <int ML>
  bool go(void* stream, const HpVal* x, int len, int L, bool series, SaReferenceHost& r);
  bool room(size_t bytes);
  void release();
};

}  // namespace nm
