// skipnet.hip - the learned series-skip predictor: a 132-64-64-1 MLP (ReLU, FP32)
// with hand-written HIP forward, backward and Adam kernels, and its training
// loop.  It predicts, per tile, the first index at which the series approximation
// becomes unstable at the tile's probe point (as the scaled rank of that index
// among the candidate indices of the reference's thresholds); the render side
// validates every prediction with the reference's stability test and falls back
// to the plain probe search.
//
// Parameters, one flat FP32 array (kParams = 12737):
//   W1[64][132], b1[64], W2[64][64], b2[64], W3[64], b3
// Forward: h1 = relu(W1 x + b1), h2 = relu(W2 h1 + b2), y = W3 . h2 + b3.
// Loss: mean over the batch of (y - t)^2.  Gradients are reduced over the batch in
// a fixed order (deterministic, no atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "skipnet.hpp"

namespace nm {

namespace {

constexpr int kIn = SkipNet::kIn, kH = SkipNet::kHidden;
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH, oB3 = oW3 + kH;
static_assert(oB3 + 1 == SkipNet::kParams, "parameter layout");

// The contractions run on the FP32 matrix units (v_mfma_f32_16x16x4_f32): lane l
// gives A[row l % 16][k = l / 16] and B[k = l / 16][column l % 16] and holds
// C[row 4 (l / 16) + i][column l % 16].  Which four k's a step takes is free (the
// sum over k in another order), so a lane group takes k's that lie together.
typedef float v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4f mfma4(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int kRows = 16;     // samples per workgroup of k_rows
constexpr int kPad = kH + 4;  // LDS row stride of the hidden layers

// One workgroup of 4 waves per 16 samples, wave w computing hidden units 16 w ..
// 16 w + 15: the forward pass and, with TRAIN, every per-sample delta of the
// backward pass: dY = 2 (y - t) / n, dH2 = dY W3 (h2 > 0), dH1 = W2^T dH2 (h1 > 0).
// Sample b is row idx[b] of X and T (row b without idx).  It is bound by the
// latency of its loads (a batch of 256 is 16 workgroups), so all weights are loaded
// before the first product needs them.  (One wave per sample and a launch each for
// the batch's gather, forward pass and deltas took 16 us per batch of 256.)
template <bool TRAIN>
__global__ __launch_bounds__(256) void k_rows(const float* __restrict__ X, const float* __restrict__ T,
                                              const int* __restrict__ idx, const float* __restrict__ P, int n,
                                              float* __restrict__ H1, float* __restrict__ H2, float* __restrict__ Y,
                                              float* __restrict__ DY, float* __restrict__ D2, float* __restrict__ D1) {
  __shared__ float h1[kRows][kPad], h2[kRows][kPad], d2[kRows][kPad];
  __shared__ float dys[kRows];
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4, u = 16 * (threadIdx.x >> 6) + r;
  const int s0 = blockIdx.x * kRows;
  const int sr = min(s0 + r, n - 1);
  // layer 1, k = 32 q + kk (kk = 0 .. 31), then k = 128 + q
  const float* xr = X + (size_t)(idx ? idx[sr] : sr) * kIn;
  const float* w1 = P + oW1 + u * kIn;
  const float* w2 = P + oW2 + u * kH + 16 * q;
  v4f xa[8], wa[8], wb[4];
  float wt[16];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    wa[k] = *(const v4f*)(w1 + 32 * q + 4 * k);
    xa[k] = *(const v4f*)(xr + 32 * q + 4 * k);
  }
  const float xl = xr[128 + q], wl = w1[128 + q];
#pragma unroll
  for (int k = 0; k < 4; k++) wb[k] = *(const v4f*)(w2 + 4 * k);
  const float b1 = P[oB1 + u], b2 = P[oB2 + u];
  const float w3 = P[oW3 + u];
  if (TRAIN) {
#pragma unroll
    for (int k = 0; k < 16; k++) wt[k] = P[oW2 + (16 * q + k) * kH + u];
  }
  v4f c = {b1, b1, b1, b1};
#pragma unroll
  for (int k = 0; k < 32; k++) c = mfma4(xa[k >> 2][k & 3], wa[k >> 2][k & 3], c);
  c = mfma4(xl, wl, c);
  v4f a1;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    a1[i] = c[i] > 0.0f ? c[i] : 0.0f;
    h1[4 * q + i][u] = a1[i];
  }
  __syncthreads();
  // layer 2, k = 16 q + kk
  c = {b2, b2, b2, b2};
#pragma unroll
  for (int k = 0; k < 16; k++) c = mfma4(h1[r][16 * q + k], wb[k >> 2][k & 3], c);
  v4f a2;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    a2[i] = c[i] > 0.0f ? c[i] : 0.0f;
    h2[4 * q + i][u] = a2[i];
  }
  __syncthreads();
  // the output: four lanes per sample, 16 hidden units each
  if (threadIdx.x < 64) {
    float y = q == 0 ? P[oB3] : 0.0f;
#pragma unroll
    for (int k = 0; k < 16; k++) y = fmaf(P[oW3 + 16 * q + k], h2[r][16 * q + k], y);
    y += __shfl_xor(y, 16);
    y += __shfl_xor(y, 32);
    const float dy = TRAIN ? 2.0f * (y - T[idx ? idx[sr] : sr]) / (float)n : 0.0f;
    if (q == 0) {
      dys[r] = dy;
      if (s0 + r < n) {
        Y[s0 + r] = y;
        if (TRAIN) DY[s0 + r] = dy;
      }
    }
  }
  if (!TRAIN) return;
  __syncthreads();
  v4f g2;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    g2[i] = a2[i] > 0.0f ? dys[4 * q + i] * w3 : 0.0f;
    d2[4 * q + i][u] = g2[i];
  }
  __syncthreads();
  c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int k = 0; k < 16; k++) c = mfma4(d2[r][16 * q + k], wt[k], c);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int s = s0 + 4 * q + i;
    if (s < n) {
      const size_t o = (size_t)s * kH + u;
      H1[o] = a1[i];
      H2[o] = a2[i];
      D2[o] = g2[i];
      D1[o] = a1[i] > 0.0f ? c[i] : 0.0f;
    }
  }
}

// The parameter gradients, one 16 x 16 tile of one product per workgroup, summed
// over the batch: dW1 | db1 = D1^T [X | 1], dW2 | db2 = D2^T [H1 | 1], dW3 | db3 =
// DY^T [H2 | 1] (a bias is the column of ones).  The four waves take every fourth
// step of four samples and their sums are added in wave order, so the result does
// not depend on timing.  With G the gradients are stored, else Adam (Kingma & Ba,
// 2015; c1 = 1 - beta1^t, c2 = 1 - beta2^t) updates each parameter where its
// gradient arises.  One more workgroup (loss not null) sums the batch's squared
// errors.  (One thread per parameter over the whole batch took 65 us for 256
// samples: a chain of dependent loads and adds in 50 workgroups.)
constexpr int kTiles1 = 4 * 9, kTiles2 = 4 * 5, kTiles3 = 5, kGradTiles = kTiles1 + kTiles2 + kTiles3;
struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;
};
__global__ __launch_bounds__(256) void k_grads(const float* __restrict__ X, const float* __restrict__ T,
                                               const int* __restrict__ idx, const float* __restrict__ H1,
                                               const float* __restrict__ H2, const float* __restrict__ Y,
                                               const float* __restrict__ DY, const float* __restrict__ D2,
                                               const float* __restrict__ D1, int n, float* __restrict__ G,
                                               float* __restrict__ P, float* __restrict__ M, float* __restrict__ V,
                                               AdamArgs ad, float* __restrict__ loss) {
  __shared__ float red[4][16][17];
  const int tid = threadIdx.x;
  if (blockIdx.x == kGradTiles) {  // mean squared error
    float* acc = &red[0][0][0];
    float s = 0.0f;
    for (int b = tid; b < n; b += 256) {
      const float d = Y[b] - T[idx ? idx[b] : b];
      s += d * d;
    }
    acc[tid] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if (tid < off) acc[tid] += acc[tid + off];
      __syncthreads();
    }
    if (tid == 0) *loss = acc[0] / (float)n;
    return;
  }
  const int lane = tid & 63, w = tid >> 6, r = lane & 15, q = lane >> 4;
  const int t = blockIdx.x;
  const int prob = t < kTiles1 ? 0 : t < kTiles1 + kTiles2 ? 1 : 2;
  const int u = prob == 0 ? t : prob == 1 ? t - kTiles1 : t - kTiles1 - kTiles2;
  const int ncol = prob == 0 ? kIn : kH, tcol = prob == 0 ? 9 : 5;
  const int j0 = 16 * (u / tcol), c0 = 16 * (u % tcol);
  const float* L = prob == 0 ? D1 : prob == 1 ? D2 : DY;
  const float* R = prob == 0 ? X : prob == 1 ? H1 : H2;
  const int ldl = prob == 2 ? 1 : kH, lj = prob == 2 ? 0 : j0 + r, lc = min(c0 + r, ncol - 1);
  const bool lok = prob != 2 || r == 0;
  const bool one = c0 + r == ncol, rok = c0 + r < ncol;
  const int* rows = prob == 0 ? idx : nullptr;
  v4f c = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int kUn = 8;  // steps of 16 samples in flight
  for (int b0 = 0; b0 < n; b0 += 16 * kUn) {
    float a[kUn], b[kUn];
#pragma unroll
    for (int k = 0; k < kUn; k++) {
      const int s = b0 + 16 * k + 4 * w + q, sc = min(s, n - 1);
      const float lv = L[(size_t)sc * ldl + lj];
      const float rv = R[(size_t)(rows ? rows[sc] : sc) * ncol + lc];
      a[k] = lok && s < n ? lv : 0.0f;
      b[k] = rok ? rv : one ? 1.0f : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < kUn; k++) c = mfma4(a[k], b[k], c);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) red[w][4 * q + i][r] = c[i];
  __syncthreads();
  const int row = tid >> 4, col = tid & 15, cc = c0 + col, jj = j0 + row;
  if (cc > ncol || (prob == 2 && row != 0)) return;
  const float g = ((red[0][row][col] + red[1][row][col]) + red[2][row][col]) + red[3][row][col];
  const bool bias = cc == ncol;
  const int p = prob == 0   ? (bias ? oB1 + jj : oW1 + jj * kIn + cc)
                : prob == 1 ? (bias ? oB2 + jj : oW2 + jj * kH + cc)
                            : (bias ? oB3 : oW3 + cc);
  if (G) {
    G[p] = g;
    return;
  }
  const float m = ad.b1 * M[p] + (1.0f - ad.b1) * g;
  const float v = ad.b2 * V[p] + (1.0f - ad.b2) * g * g;
  M[p] = m;
  V[p] = v;
  P[p] -= ad.lr * (m / ad.c1) / (sqrtf(v / ad.c2) + ad.eps);
}

uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

}  // namespace

#define SN_HIP(expr)                                                    \
  do {                                                                  \
    hipError_t e_ = (expr);                                             \
    if (e_ != hipSuccess) {                                             \
      err_ = std::string(#expr) + ": " + hipGetErrorString(e_);         \
      return NM_ERR_HIP;                                                \
    }                                                                   \
  } while (0)

SkipNet::SkipNet() : params(kParams, 0.0f), mean(kIn, 0.0f), scale(kIn, 1.0f) {}

SkipNet::~SkipNet() { release(); }

void SkipNet::release() {
  for (void* p : {(void*)dP, (void*)dG, (void*)dM, (void*)dV, (void*)dX, (void*)dT, (void*)dH1, (void*)dH2, (void*)dY,
                  (void*)dDY, (void*)dD1, (void*)dD2, (void*)dIdx, (void*)dLoss})
    if (p) (void)hipFree(p);
  dP = dG = dM = dV = dX = dT = dH1 = dH2 = dY = dDY = dD1 = dD2 = dLoss = nullptr;
  dIdx = nullptr;
  capX = capB = capI = 0;
}

// He-uniform initialisation from a seed (deterministic)
void SkipNet::init(uint64_t seed) {
  uint64_t s = seed;
  auto uni = [&](float a) { return (float)(((splitmix(s) >> 11) * (1.0 / 9007199254740992.0)) * 2.0 - 1.0) * a; };
  const float a1 = std::sqrt(6.0f / kIn), a2 = std::sqrt(6.0f / kH);
  for (int i = 0; i < kH * kIn; i++) params[oW1 + i] = uni(a1);
  for (int i = 0; i < kH; i++) params[oB1 + i] = 0.0f;
  for (int i = 0; i < kH * kH; i++) params[oW2 + i] = uni(a2);
  for (int i = 0; i < kH; i++) params[oB2 + i] = 0.0f;
  for (int i = 0; i < kH; i++) params[oW3 + i] = uni(a2);
  params[oB3] = 0.0f;
}

// device buffers for nx rows of input, batches of nb, ni row indices (grow-only)
int SkipNet::reserve(size_t nx, size_t nb, size_t ni) {
  if (!dP) {
    SN_HIP(hipMalloc((void**)&dP, kParams * 4));
    SN_HIP(hipMalloc((void**)&dG, kParams * 4));
    SN_HIP(hipMalloc((void**)&dM, kParams * 4));
    SN_HIP(hipMalloc((void**)&dV, kParams * 4));
    SN_HIP(hipMalloc((void**)&dLoss, kMaxEpochsAtOnce * 4));
  }
  auto again = [&](auto** p, size_t count) {
    if (*p) SN_HIP(hipFree(*p));
    *p = nullptr;
    SN_HIP(hipMalloc((void**)p, count * 4));
    return (int)NM_OK;
  };
  int st;
  if (nx > capX) {
    capX = 0;
    if ((st = again(&dX, nx * kIn)) || (st = again(&dT, nx))) return st;
    capX = nx;
  }
  if (nb > capB) {
    capB = 0;
    for (float** p : {&dH1, &dH2, &dD1, &dD2})
      if ((st = again(p, nb * kH))) return st;
    if ((st = again(&dY, nb)) || (st = again(&dDY, nb))) return st;
    capB = nb;
  }
  if (ni > capI) {
    capI = 0;
    if ((st = again(&dIdx, ni))) return st;
    capI = ni;
  }
  return NM_OK;
}

void SkipNet::normalise(const float* raw, size_t n, std::vector<float>& out) const {
  out.resize(n * kIn);
  for (size_t b = 0; b < n; b++)
    for (int k = 0; k < kIn; k++) out[b * kIn + k] = (raw[b * kIn + k] - mean[k]) * scale[k];
}

// sums per feature in row order, all features side by side (one feature after the
// other walked the rows 132 times: 1 ms for 2040 rows)
void SkipNet::fit_normaliser(const float* raw, size_t n) {
  double s[kIn] = {}, s2[kIn] = {};
  for (size_t b = 0; b < n; b++)
    for (int k = 0; k < kIn; k++) {
      const double v = raw[b * kIn + k];
      s[k] += v;
      s2[k] += v * v;
    }
  for (int k = 0; k < kIn; k++) {
    const double mu = s[k] / (double)n, var = std::max(0.0, s2[k] / (double)n - mu * mu);
    mean[k] = (float)mu;
    scale[k] = var > 1e-12 ? (float)(1.0 / std::sqrt(var)) : 1.0f;
  }
}

int SkipNet::predict(const float* raw, size_t n, float* y) {
  if (n == 0) return NM_OK;
  int st = reserve(n, n, 0);
  if (st) return st;
  std::vector<float> xn;
  normalise(raw, n, xn);
  SN_HIP(hipMemcpy(dP, params.data(), kParams * 4, hipMemcpyHostToDevice));
  SN_HIP(hipMemcpy(dX, xn.data(), n * kIn * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_rows<false>, dim3((unsigned)((n + kRows - 1) / kRows)), dim3(256), 0, 0, (const float*)dX,
                     (const float*)nullptr, (const int*)nullptr, (const float*)dP, (int)n, (float*)nullptr,
                     (float*)nullptr, dY, (float*)nullptr, (float*)nullptr, (float*)nullptr);
  SN_HIP(hipGetLastError());
  SN_HIP(hipMemcpy(y, dY, n * 4, hipMemcpyDeviceToHost));
  return NM_OK;
}

// one batch: rows idx[0 .. n) of dX and dT (rows 0 .. n - 1 without idx); the
// gradients into G, or with a null G an Adam step; loss: where its loss goes, or null
int SkipNet::batch(const int* idx, int n, float* G, const AdamStep& a, float* loss) {
  hipLaunchKernelGGL(k_rows<true>, dim3((n + kRows - 1) / kRows), dim3(256), 0, 0, (const float*)dX, (const float*)dT,
                     idx, (const float*)dP, n, dH1, dH2, dY, dDY, dD2, dD1);
  SN_HIP(hipGetLastError());
  const AdamArgs ad{a.lr, 0.9f, 0.999f, 1e-8f, a.c1, a.c2};
  hipLaunchKernelGGL(k_grads, dim3(kGradTiles + (loss ? 1 : 0)), dim3(256), 0, 0, (const float*)dX, (const float*)dT,
                     idx, (const float*)dH1, (const float*)dH2, (const float*)dY, (const float*)dDY, (const float*)dD2,
                     (const float*)dD1, n, G, dP, dM, dV, ad, loss);
  SN_HIP(hipGetLastError());
  return NM_OK;
}

// loss and gradient of one batch (inputs already normalised), for checks
int SkipNet::gradient(const float* xn, const float* t, size_t n, float* grad, float* loss) {
  int st = reserve(n, n, 0);
  if (st) return st;
  SN_HIP(hipMemcpy(dP, params.data(), kParams * 4, hipMemcpyHostToDevice));
  SN_HIP(hipMemcpy(dX, xn, n * kIn * 4, hipMemcpyHostToDevice));
  SN_HIP(hipMemcpy(dT, t, n * 4, hipMemcpyHostToDevice));
  st = batch(nullptr, (int)n, dG, AdamStep{}, dLoss);
  if (st) return st;
  SN_HIP(hipMemcpy(grad, dG, kParams * 4, hipMemcpyDeviceToHost));
  if (loss) SN_HIP(hipMemcpy(loss, dLoss, 4, hipMemcpyDeviceToHost));
  return NM_OK;
}

// Two launches per batch, and the host waits once for a group of epochs: their
// row orders go up together and their losses come back together.
int SkipNet::train(const float* raw, const float* t, size_t n, const TrainOpts& o, std::vector<float>* curve) {
  if (n == 0 || o.batch <= 0 || o.epochs <= 0) return NM_ERR_ARG;
  fit_normaliser(raw, n);
  init(o.seed);
  const size_t nb = std::min<size_t>((size_t)o.batch, n);
  // epochs whose row orders are on the device at a time: up to 64, and 16 MB of them
  const int group = (int)std::max<size_t>(
      1, std::min<size_t>({(size_t)o.epochs, (size_t)kMaxEpochsAtOnce, ((size_t)4 << 20) / n}));
  int st = reserve(n, nb, (size_t)group * n);
  if (st) return st;
  std::vector<float> xn;
  normalise(raw, n, xn);
  SN_HIP(hipMemcpy(dX, xn.data(), n * kIn * 4, hipMemcpyHostToDevice));
  SN_HIP(hipMemcpy(dT, t, n * 4, hipMemcpyHostToDevice));
  SN_HIP(hipMemcpy(dP, params.data(), kParams * 4, hipMemcpyHostToDevice));
  SN_HIP(hipMemset(dM, 0, kParams * 4));
  SN_HIP(hipMemset(dV, 0, kParams * 4));
  std::vector<int> perm(n), orders((size_t)group * n);
  for (size_t i = 0; i < n; i++) perm[i] = (int)i;
  uint64_t rs = o.seed ^ 0x5DEECE66Dull;
  double p1 = 1.0, p2 = 1.0;
  if (curve) curve->clear();
  for (int ep0 = 0; ep0 < o.epochs; ep0 += group) {
    const int eps = std::min(group, o.epochs - ep0);
    for (int e = 0; e < eps; e++) {
      for (size_t i = n - 1; i > 0; i--) std::swap(perm[i], perm[splitmix(rs) % (i + 1)]);  // Fisher-Yates
      std::copy(perm.begin(), perm.end(), orders.begin() + (size_t)e * n);
    }
    SN_HIP(hipMemcpy(dIdx, orders.data(), (size_t)eps * n * 4, hipMemcpyHostToDevice));
    for (int e = 0; e < eps; e++) {
      const int ep = ep0 + e;
      const float lr = o.lr * (ep < o.epochs / 2 ? 1.0f : (ep < 3 * o.epochs / 4 ? 0.3f : 0.1f));
      for (size_t s = 0; s + nb <= n; s += nb) {
        p1 *= 0.9f;
        p2 *= 0.999f;
        const AdamStep a{lr, (float)(1.0 - p1), (float)(1.0 - p2)};
        // first batch loss of each epoch (before the step)
        st = batch(dIdx + (size_t)e * n + s, (int)nb, nullptr, a, s == 0 ? dLoss + e : nullptr);
        if (st) return st;
      }
    }
    if (curve) {
      curve->resize((size_t)ep0 + eps);
      SN_HIP(hipMemcpy(curve->data() + ep0, dLoss, (size_t)eps * 4, hipMemcpyDeviceToHost));
    }
  }
  SN_HIP(hipMemcpy(params.data(), dP, kParams * 4, hipMemcpyDeviceToHost));
  trained = true;
  version++;
  return NM_OK;
}

}  // namespace nm
