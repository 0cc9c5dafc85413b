// series_chain.hpp - the series coefficients A, B, C of a reference orbit as one chain
// of high-precision operations, the recurrence exactly as the reference writes it
// (mandelbrot.cpp:112-131, A[i], B[i] on the right-hand side of B[i], C[i]).  Only the
// truncated doubles the per-pixel work reads, and their floatexp form, are kept: A .. Ce
// of r.  L: the working precision in limbs.
#pragma once
#include "engine.hpp"
#include "hpfloat.hpp"

namespace nm {

void series_chain(const HPComplex* X, int len, int L, SaReferenceHost& r);

}  // namespace nm
