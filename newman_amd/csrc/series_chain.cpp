// series_chain.cpp - see series_chain.hpp
#include "series_chain.hpp"

namespace nm {

void series_chain(const HPComplex* X, int len, int L, SaReferenceHost& r) {
  r.A.assign(2 * (size_t)len, 0.0);
  r.B.assign(2 * (size_t)len, 0.0);
  r.C.assign(2 * (size_t)len, 0.0);
  r.Am.assign(2 * (size_t)len, 0.0);
  r.Bm.assign(2 * (size_t)len, 0.0);
  r.Cm.assign(2 * (size_t)len, 0.0);
  r.Ae.assign(2 * (size_t)len, kFxZeroExp);
  r.Be.assign(2 * (size_t)len, kFxZeroExp);
  r.Ce.assign(2 * (size_t)len, kFxZeroExp);
  r.Am[0] = 0.5;
  r.Ae[0] = 1;
  hpf Ar(L), Ai(L), Br(L), Bi(L), Cr(L), Ci(L), nAr(L), nAi(L), nBr(L), nBi(L), nCr(L), nCi(L), t(L);
  hpf one(2);
  hp_set_d(one, 1.0);
  hp_set_d(Ar, 1.0);
  r.A[0] = 1.0;
  for (int i = 1; i < len; i++) {
    const hpf& xr = X[i - 1].re;
    const hpf& xi = X[i - 1].im;
    hp_mul(nAr, xr, Ar); hp_mul(t, xi, Ai); hp_sub(nAr, nAr, t); times2(nAr); hp_add(nAr, nAr, one);
    hp_mul(nAi, xr, Ai); hp_mul(t, xi, Ar); hp_add(nAi, nAi, t); times2(nAi);
    hp_mul(nBr, xr, Br); hp_mul(t, xi, Bi); hp_sub(nBr, nBr, t); times2(nBr);
    hp_mul(t, nAr, nAr); hp_add(nBr, nBr, t);
    hp_mul(t, nAi, nAi); hp_sub(nBr, nBr, t);
    hp_mul(nBi, xr, Bi); hp_mul(t, xi, Br); hp_add(nBi, nBi, t);
    hp_mul(t, nAr, nAi); hp_add(nBi, nBi, t); times2(nBi);
    hp_mul(nCr, xr, Cr); hp_mul(t, xi, Ci); hp_sub(nCr, nCr, t);
    hp_mul(t, nAr, nBr); hp_add(nCr, nCr, t);
    hp_mul(t, nAi, nBi); hp_sub(nCr, nCr, t); times2(nCr);
    hp_mul(nCi, xr, Ci); hp_mul(t, xi, Cr); hp_add(nCi, nCi, t);
    hp_mul(t, nAr, nBi); hp_add(nCi, nCi, t);
    hp_mul(t, nAi, nBr); hp_add(nCi, nCi, t); times2(nCi);
    hp_copy_prec(Ar, nAr); hp_copy_prec(Ai, nAi);
    hp_copy_prec(Br, nBr); hp_copy_prec(Bi, nBi);
    hp_copy_prec(Cr, nCr); hp_copy_prec(Ci, nCi);
    r.A[2 * i] = Ar.get_d(); r.A[2 * i + 1] = Ai.get_d();
    r.B[2 * i] = Br.get_d(); r.B[2 * i + 1] = Bi.get_d();
    r.C[2 * i] = Cr.get_d(); r.C[2 * i + 1] = Ci.get_d();
    const hpf* hv[6] = {&Ar, &Ai, &Br, &Bi, &Cr, &Ci};
    std::vector<double>* fm[3] = {&r.Am, &r.Bm, &r.Cm};
    std::vector<int32_t>* fe[3] = {&r.Ae, &r.Be, &r.Ce};
    for (int k = 0; k < 6; k++) {
      long e = 0;
      const double m = hv[k]->get_d_2exp(&e);
      (*fm[k / 2])[2 * i + k % 2] = m;
      (*fe[k / 2])[2 * i + k % 2] = m == 0.0 ? kFxZeroExp : (int32_t)e;
    }
  }
}

}  // namespace nm
