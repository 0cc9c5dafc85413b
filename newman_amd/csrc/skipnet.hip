// skipnet.hip - the learned series-skip predictor: a 132-64-64-1 MLP (ReLU)
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

// Every sum is taken one term after the other in FP32, each product rounded before
// it is added: hidden units over their inputs, gradients over the batch.  A hidden
// unit within rounding of 0 falls on the other side of its ReLU with any other order
// (one training of 2040 rows in twelve has such a unit, and Adam carries it into
// every parameter), so the order is kept fixed rather than given to matrix units: a
// chain of 256 additions is 0.9 us, and the products and loads beside it are what the
// layout below is for.
//
// The device's parameters: the forward weights four inputs at a time, [k / 4][unit]
// [k % 4], W2 also by its rows for the backward pass, so that a wave (lane = unit)
// reads 1 KB of them at a time.
constexpr int dW1 = 0, dB1 = dW1 + kH * kIn, dW2 = dB1 + kH, dB2 = dW2 + kH * kH, dW3 = dB2 + kH, dB3 = dW3 + kH,
              dW2t = dB3 + 4, kDevParams = dW2t + kH * kH;
static_assert(kIn % 4 == 0 && kH == 64 && dW2t % 4 == 0, "parameter layout on the device");
__host__ __device__ constexpr int at4(int k, int unit) { return ((k >> 2) * kH + unit) * 4 + (k & 3); }

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRows = 4;  // samples per workgroup of k_rows, a wave each

// s + w[0] x[0] + w[1] x[1] + ..., in that order
template <int K4>
__device__ __forceinline__ float chain(float s, const v4f (&w)[K4], const float* x) {
#pragma unroll
  for (int k = 0; k < K4; k++) {
    const v4f v = *(const v4f*)(x + 4 * k);
#pragma unroll
    for (int i = 0; i < 4; i++) s += w[k][i] * v[i];
  }
  return s;
}
template <int K4>
__device__ __forceinline__ void weights4(v4f (&w)[K4], const float* p, int j) {
#pragma unroll
  for (int k = 0; k < K4; k++) w[k] = *(const v4f*)(p + (k * kH + j) * 4);
}

// features standardised in place: (x - mean) scale
__global__ __launch_bounds__(256) void k_standardise(const float* __restrict__ mean, const float* __restrict__ scale,
                                                     long count, float* __restrict__ X) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < count; i += gridDim.x * 256L) {
    const int k = (int)(i % kIn);
    X[i] = (X[i] - mean[k]) * scale[k];
  }
}

// One wave per sample, lane j its hidden unit j: the forward pass and, with TRAIN,
// every delta of the backward pass: dY = 2 (y - t) / n, dH2 = dY W3 (h2 > 0), dH1 =
// W2^T dH2 (h1 > 0).  Sample b is row idx[b] of X and T (row b without idx); XB gets
// the batch's rows for the gradients.  It is bound by latency (a batch of 256 is 256
// waves: the weights' loads, then some 330 dependent additions), so a sample has a
// wave of its own and the weights are loaded before the sums that need them begin.
template <bool TRAIN>
__global__ __launch_bounds__(64 * kRows) void k_rows(const float* __restrict__ X, const float* __restrict__ T,
                                                     const int* __restrict__ idx, const float* __restrict__ P, int n,
                                                     float* __restrict__ XB, float* __restrict__ H1,
                                                     float* __restrict__ H2, float* __restrict__ Y,
                                                     float* __restrict__ DY, float* __restrict__ D2,
                                                     float* __restrict__ D1) {
  __shared__ __align__(16) float xs[kRows][kIn], h1[kRows][kH], h2[kRows][kH], d2[kRows][kH];
  const int j = threadIdx.x & 63, w = threadIdx.x >> 6, s = blockIdx.x * kRows + w;
  const bool live = s < n;
  const int b = min(s, n - 1);
  const size_t row = idx ? idx[b] : b;
  if (j < kIn / 4) {
    const v4f v = *(const v4f*)(X + row * kIn + 4 * j);
    *(v4f*)&xs[w][4 * j] = v;
    if (TRAIN && live) *(v4f*)(XB + (size_t)s * kIn + 4 * j) = v;
  }
  v4f wa[kIn / 4], wb[kH / 4], wt[kH / 4];
  weights4(wa, P + dW1, j);
  weights4(wb, P + dW2, j);
  const float b1 = P[dB1 + j], b2 = P[dB2 + j], w3 = P[dW3 + j], b3 = P[dB3];
  const float t = TRAIN ? T[row] : 0.0f;
  __syncthreads();
  float a1 = chain(b1, wa, xs[w]);
  a1 = a1 > 0.0f ? a1 : 0.0f;
  h1[w][j] = a1;
  if (TRAIN) weights4(wt, P + dW2t, j);
  __syncthreads();
  float a2 = chain(b2, wb, h1[w]);
  a2 = a2 > 0.0f ? a2 : 0.0f;
  h2[w][j] = w3 * a2;  // the output's terms
  __syncthreads();
  float y = b3;
#pragma unroll
  for (int k = 0; k < kH / 4; k++) {
    const v4f v = *(const v4f*)&h2[w][4 * k];
#pragma unroll
    for (int i = 0; i < 4; i++) y += v[i];
  }
  if (live && j == 0) Y[s] = y;
  if (!TRAIN) return;
  const float dy = 2.0f * (y - t) / (float)n;
  const float g2 = a2 > 0.0f ? dy * w3 : 0.0f;
  d2[w][j] = g2;
  __syncthreads();
  const float g1 = chain(0.0f, wt, d2[w]);
  if (!live) return;
  const size_t o = (size_t)s * kH + j;
  H1[o] = a1;
  H2[o] = a2;
  D2[o] = g2;
  D1[o] = a1 > 0.0f ? g1 : 0.0f;
  if (j == 0) DY[s] = dy;
}

// The parameter gradients, one 8 x 8 tile of one product per wave, a lane per
// parameter, summed over the batch in its order: dW1 | db1 = D1^T [XB | 1], dW2 | db2
// = D2^T [H1 | 1], dW3 | db3 = DY^T [H2 | 1] (a bias is the column of ones).  The
// tile's columns of 256 samples come at once and lie in LDS by column, so that a lane
// reads four samples at a time.  With G the gradients are stored, else Adam (Kingma &
// Ba, 2015; c1 = 1 - beta1^t, c2 = 1 - beta2^t) updates each parameter where its
// gradient arises; its old values are loaded before the batch's.  One more workgroup
// (loss not null) sums the batch's squared errors.  (One thread per parameter that
// reads the batch from memory took 65 us for 256 samples.)
constexpr int kTile = 8;
constexpr int kCols1 = (kIn + kTile) / kTile, kCols2 = (kH + kTile) / kTile;  // the bias among them
constexpr int kTiles1 = kH / kTile * kCols1, kTiles2 = kH / kTile * kCols2, kTiles3 = kCols2;
constexpr int kGradTiles = kTiles1 + kTiles2 + kTiles3;
constexpr int kChunk = 256;        // samples in LDS
constexpr int kCol = kChunk + 4;   // LDS stride of a column: eight columns' reads of 16 bytes hit 32 banks
struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;
};
__global__ __launch_bounds__(64) void k_grads(const float* __restrict__ XB, const float* __restrict__ T,
                                              const int* __restrict__ idx, const float* __restrict__ H1,
                                              const float* __restrict__ H2, const float* __restrict__ Y,
                                              const float* __restrict__ DY, const float* __restrict__ D2,
                                              const float* __restrict__ D1, int n, float* __restrict__ G,
                                              float* __restrict__ P, float* __restrict__ M, float* __restrict__ V,
                                              AdamArgs ad, float* __restrict__ loss) {
  __shared__ __align__(16) float ls[kTile][kCol], rs[kTile][kCol];
  const int lane = threadIdx.x;
  if (blockIdx.x == kGradTiles) {  // mean squared error: 256 partial sums, then their tree
    float* acc = &ls[0][0];
    for (int k = lane; k < 256; k += 64) {
      float s = 0.0f;
      for (int b = k; b < n; b += 256) {
        const float d = Y[b] - T[idx ? idx[b] : b];
        s += d * d;
      }
      acc[k] = s;
    }
    for (int off = 128; off > 0; off >>= 1) {
      __syncthreads();
      for (int k = lane; k < off; k += 64) acc[k] += acc[k + off];
    }
    if (lane == 0) *loss = acc[0] / (float)n;
    return;
  }
  const int t = blockIdx.x;
  const int prob = t < kTiles1 ? 0 : t < kTiles1 + kTiles2 ? 1 : 2;
  const int u = prob == 0 ? t : prob == 1 ? t - kTiles1 : t - kTiles1 - kTiles2;
  const int ncol = prob == 0 ? kIn : kH, tcol = prob == 0 ? kCols1 : kCols2;
  const int j0 = kTile * (u / tcol), c0 = kTile * (u % tcol);
  // this lane's parameter: flat index p (< 0: none), place on the device at and at2
  const int jr = lane >> 3, kc = lane & 7, j = j0 + jr, c = c0 + kc;
  const bool bias = c == ncol;
  int p = -1, at = 0, at2 = -1;
  if (c <= ncol && (prob != 2 || jr == 0)) {
    if (prob == 0) {
      p = bias ? oB1 + j : oW1 + j * kIn + c;
      at = bias ? dB1 + j : dW1 + at4(c, j);
    } else if (prob == 1) {
      p = bias ? oB2 + j : oW2 + j * kH + c;
      at = bias ? dB2 + j : dW2 + at4(c, j);
      at2 = bias ? -1 : dW2t + at4(j, c);
    } else {
      p = bias ? oB3 : oW3 + c;
      at = bias ? dB3 : dW3 + c;
    }
  }
  const bool step = !G && p >= 0;
  const float m0 = step ? M[p] : 0.0f, v0 = step ? V[p] : 0.0f, p0 = step ? P[at] : 0.0f;
  // a lane loads four columns of one sample in 32
  const int half = 4 * (lane & 1), bq = lane >> 1;
  const float* R = prob == 0 ? XB : prob == 1 ? H1 : H2;
  const float* L = prob == 0 ? D1 : D2;
  const v4f none = {0.0f, 0.0f, 0.0f, 0.0f}, ones = {1.0f, 0.0f, 0.0f, 0.0f};
  const int rc = c0 + half;  // ncol is a multiple of 4
  constexpr int kLoads = kChunk / 32;
  float g = 0.0f;
  for (int b0 = 0; b0 < n; b0 += kChunk) {
    v4f lv[kLoads], rv[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      const int b = b0 + 32 * i + bq;
      lv[i] = rv[i] = none;
      if (b < n) {
        if (prob != 2) lv[i] = *(const v4f*)(L + (size_t)b * kH + j0 + half);
        else if (half == 0) lv[i][0] = DY[b];
        if (rc < ncol) rv[i] = *(const v4f*)(R + (size_t)b * ncol + rc);
        else if (rc == ncol) rv[i] = ones;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kLoads; i++)
#pragma unroll
      for (int k = 0; k < 4; k++) {
        ls[half + k][32 * i + bq] = lv[i][k];
        rs[half + k][32 * i + bq] = rv[i][k];
      }
    __syncthreads();
    const int m = min(kChunk, n - b0);  // zeros behind the last sample add nothing
#pragma unroll 4
    for (int b = 0; b < m; b += 4) {
      const v4f x = *(const v4f*)&ls[jr][b], z = *(const v4f*)&rs[kc][b];
#pragma unroll
      for (int i = 0; i < 4; i++) g += x[i] * z[i];
    }
  }
  if (p < 0) return;
  if (G) {
    G[p] = g;
    return;
  }
  const float mm = ad.b1 * m0 + (1.0f - ad.b1) * g;
  const float vv = ad.b2 * v0 + (1.0f - ad.b2) * g * g;
  M[p] = mm;
  V[p] = vv;
  const float q = p0 - ad.lr * (mm / ad.c1) / (sqrtf(vv / ad.c2) + ad.eps);
  P[at] = q;
  if (at2 >= 0) P[at2] = q;
}

// flat parameters in the device's layout
std::vector<float> to_device(const std::vector<float>& p) {
  std::vector<float> d(kDevParams, 0.0f);
  for (int j = 0; j < kH; j++) {
    for (int k = 0; k < kIn; k++) d[dW1 + at4(k, j)] = p[oW1 + j * kIn + k];
    for (int k = 0; k < kH; k++) d[dW2 + at4(k, j)] = d[dW2t + at4(j, k)] = p[oW2 + j * kH + k];
    d[dB1 + j] = p[oB1 + j];
    d[dB2 + j] = p[oB2 + j];
    d[dW3 + j] = p[oW3 + j];
  }
  d[dB3] = p[oB3];
  return d;
}
void from_device(const std::vector<float>& d, std::vector<float>& p) {
  for (int j = 0; j < kH; j++) {
    for (int k = 0; k < kIn; k++) p[oW1 + j * kIn + k] = d[dW1 + at4(k, j)];
    for (int k = 0; k < kH; k++) p[oW2 + j * kH + k] = d[dW2 + at4(k, j)];
    p[oB1 + j] = d[dB1 + j];
    p[oB2 + j] = d[dB2 + j];
    p[oW3 + j] = d[dW3 + j];
  }
  p[oB3] = d[dB3];
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
                  (void*)dDY, (void*)dD1, (void*)dD2, (void*)dIdx, (void*)dLoss, (void*)dXB, (void*)dNorm})
    if (p) (void)hipFree(p);
  dP = dG = dM = dV = dX = dT = dH1 = dH2 = dY = dDY = dD1 = dD2 = dLoss = dXB = dNorm = nullptr;
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
    SN_HIP(hipMalloc((void**)&dP, kDevParams * 4));
    SN_HIP(hipMalloc((void**)&dG, kParams * 4));
    SN_HIP(hipMalloc((void**)&dM, kParams * 4));
    SN_HIP(hipMalloc((void**)&dV, kParams * 4));
    SN_HIP(hipMalloc((void**)&dLoss, kMaxEpochsAtOnce * 4));
    SN_HIP(hipMalloc((void**)&dNorm, 2 * kIn * 4));
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
    if ((st = again(&dY, nb)) || (st = again(&dDY, nb)) || (st = again(&dXB, nb * kIn))) return st;
    capB = nb;
  }
  if (ni > capI) {
    capI = 0;
    if ((st = again(&dIdx, ni))) return st;
    capI = ni;
  }
  return NM_OK;
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

// n rows of features to dX, standardised with mean and scale where `norm` is set
int SkipNet::inputs(const float* raw, size_t n, bool norm) {
  if (norm) {
    SN_HIP(hipMemcpy(dNorm, mean.data(), kIn * 4, hipMemcpyHostToDevice));
    SN_HIP(hipMemcpy(dNorm + kIn, scale.data(), kIn * 4, hipMemcpyHostToDevice));
  }
  SN_HIP(hipMemcpy(dX, raw, n * kIn * 4, hipMemcpyHostToDevice));
  if (!norm) return NM_OK;
  const size_t count = n * kIn;
  hipLaunchKernelGGL(k_standardise, dim3((unsigned)std::min<size_t>(2048, (count + 255) / 256)), dim3(256), 0, 0,
                     (const float*)dNorm, (const float*)(dNorm + kIn), (long)count, dX);
  SN_HIP(hipGetLastError());
  return NM_OK;
}

// the parameters to dP
int SkipNet::weights() {
  const std::vector<float> d = to_device(params);
  SN_HIP(hipMemcpy(dP, d.data(), kDevParams * 4, hipMemcpyHostToDevice));
  return NM_OK;
}

int SkipNet::predict(const float* raw, size_t n, float* y) {
  if (n == 0) return NM_OK;
  int st;
  if ((st = reserve(n, n, 0)) || (st = weights()) || (st = inputs(raw, n, true))) return st;
  hipLaunchKernelGGL(k_rows<false>, dim3((unsigned)((n + kRows - 1) / kRows)), dim3(64 * kRows), 0, 0,
                     (const float*)dX, (const float*)nullptr, (const int*)nullptr, (const float*)dP, (int)n,
                     (float*)nullptr, (float*)nullptr, (float*)nullptr, dY, (float*)nullptr, (float*)nullptr,
                     (float*)nullptr);
  SN_HIP(hipGetLastError());
  SN_HIP(hipMemcpy(y, dY, n * 4, hipMemcpyDeviceToHost));
  return NM_OK;
}

// one batch: rows idx[0 .. n) of dX and dT (rows 0 .. n - 1 without idx); the
// gradients into G, or with a null G an Adam step; loss: where its loss goes, or null
int SkipNet::batch(const int* idx, int n, float* G, const AdamStep& a, float* loss) {
  hipLaunchKernelGGL(k_rows<true>, dim3((n + kRows - 1) / kRows), dim3(64 * kRows), 0, 0, (const float*)dX,
                     (const float*)dT, idx, (const float*)dP, n, dXB, dH1, dH2, dY, dDY, dD2, dD1);
  SN_HIP(hipGetLastError());
  const AdamArgs ad{a.lr, 0.9f, 0.999f, 1e-8f, a.c1, a.c2};
  hipLaunchKernelGGL(k_grads, dim3(kGradTiles + (loss ? 1 : 0)), dim3(64), 0, 0, (const float*)dXB, (const float*)dT,
                     idx, (const float*)dH1, (const float*)dH2, (const float*)dY, (const float*)dDY, (const float*)dD2,
                     (const float*)dD1, n, G, dP, dM, dV, ad, loss);
  SN_HIP(hipGetLastError());
  return NM_OK;
}

// loss and gradient of one batch (inputs already normalised), for checks
int SkipNet::gradient(const float* xn, const float* t, size_t n, float* grad, float* loss) {
  int st;
  if ((st = reserve(n, n, 0)) || (st = weights()) || (st = inputs(xn, n, false))) return st;
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
  int st;
  if ((st = reserve(n, nb, (size_t)group * n)) || (st = weights()) || (st = inputs(raw, n, true))) return st;
  SN_HIP(hipMemcpy(dT, t, n * 4, hipMemcpyHostToDevice));
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
  std::vector<float> d(kDevParams);
  SN_HIP(hipMemcpy(d.data(), dP, kDevParams * 4, hipMemcpyDeviceToHost));
  from_device(d, params);
  trained = true;
  version++;
  return NM_OK;
}

}  // namespace nm
