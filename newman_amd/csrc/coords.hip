// coords.hip - a frame set's coordinate tables, made on the device from the centre
// and sample size: one thread per column and per row of every frame.  The host made
// them one high-precision operation after the other (0.3 us an entry: 4 ms for a
// 7680 x 4320 frame, half of a 640 x 480 call that keeps no tables) and copied them:
// that call 565 -> 256 us, the first pass of a 7680 x 4320 plain view 8.2 -> 4.9 ms.
// The threads are few (some 12,000 at the most for one frame) and the work of each a
// chain of carries, so workgroups of one wave spread them over the CUs.
#include "coords.hpp"

namespace nm {

namespace {

template <int ML>
__device__ __forceinline__ void coords_entry(const FrameHp& h, bool series, bool row, long k, double* hi, double* lo) {
  const hpd<ML> p = hpd_pixel<ML>(row ? h.cim : h.cre, row ? h.sim : h.sre, k, h.L);
  if (series) {
    *hi = hpd_get_d(hpd_add(p, hpd_load<ML>(row ? h.x0im : h.x0re), -1, h.L));
  } else {
    *hi = hpd_get_d(p);
    *lo = hpd_rest(p);
  }
}

template <int ML>
__device__ __forceinline__ void coords_all(const FrameHp& h, int f, int nr, int nc, bool series, CoordTables t, int i) {
  const bool row = i >= nc;
  const int j = row ? i - nc : i;
  const size_t o = (size_t)f * (row ? nr : nc) + j;
  coords_entry<ML>(h, series, row, row ? row_offset(j, nr) : column_offset(j, nc), (row ? t.rhi : t.chi) + o,
                   (row ? t.rlo : t.clo) + o);
}

template <int ML>
__global__ __launch_bounds__(64) void k_coords_one(FrameHp h, int nr, int nc, bool series, CoordTables t) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nr + nc) coords_all<ML>(h, 0, nr, nc, series, t, i);
}
template <int ML>
__global__ __launch_bounds__(64) void k_coords(const FrameHp* h, int nr, int nc, bool series, CoordTables t) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nr + nc) coords_all<ML>(h[blockIdx.y], blockIdx.y, nr, nc, series, t, i);
}

template <int ML>
void go(hipStream_t s, const FrameHp* one, const FrameHp* dev, int frames, int nr, int nc, bool series, CoordTables t) {
  const unsigned blocks = (unsigned)(((int64_t)nr + nc + 63) / 64);
  if (one) {
    hipLaunchKernelGGL(k_coords_one<ML>, dim3(blocks), dim3(64), 0, s, *one, nr, nc, series, t);
    return;
  }
  for (int f = 0; f < frames; f += 65535) {  // grid y limit
    const int n = frames - f < 65535 ? frames - f : 65535;
    CoordTables u = t;
    u.chi += (size_t)f * nc;
    u.rhi += (size_t)f * nr;
    if (!series) {
      u.clo += (size_t)f * nc;
      u.rlo += (size_t)f * nr;
    }
    hipLaunchKernelGGL(k_coords<ML>, dim3(blocks, n), dim3(64), 0, s, dev + f, nr, nc, series, u);
  }
}

}  // namespace

int coords_launch(void* stream, const FrameHp* hp_one, const FrameHp* hp_dev, int frames, int nr, int nc, int limbs,
                  bool series, CoordTables t) {
  hipStream_t s = (hipStream_t)stream;
  // limbs: the most that any of the values holds; a table entry's work grows with
  // the limbs it is compiled for
  if (limbs <= 4) go<4>(s, hp_one, hp_dev, frames, nr, nc, series, t);
  else if (limbs <= 8) go<8>(s, hp_one, hp_dev, frames, nr, nc, series, t);
  else if (limbs <= 16) go<16>(s, hp_one, hp_dev, frames, nr, nc, series, t);
  else go<kHpMaxLimbs>(s, hp_one, hp_dev, frames, nr, nc, series, t);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

}  // namespace nm
