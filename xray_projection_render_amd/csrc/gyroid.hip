// gyroid.hip - kernels of the gyroid march (gyroid_march.hpp), one wave per
// workgroup on the ray tiles of march.hip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gyroid_march.hpp"
#include "two_pass.hpp"

namespace xrp {

constexpr int kGyroTileI = 32, kGyroTileJ = 2;

struct GyroPixel {
  int v, i, j;
  bool valid;
};
__device__ __forceinline__ GyroPixel gyro_pixel(const MarchParams& p) {
  const int lane = threadIdx.x;
  const int tiles_j = (p.res + kGyroTileJ - 1) / kGyroTileJ;
  const int ti = blockIdx.x / tiles_j, tj = blockIdx.x - ti * tiles_j;
  GyroPixel q;
  q.v = blockIdx.y;
  q.i = ti * kGyroTileI + lane / kGyroTileJ;
  q.j = tj * kGyroTileJ + lane % kGyroTileJ;
  q.valid = q.i < p.res && q.j < p.res;
  return q;
}

template <int DEF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8))) void
gyro_try_kernel(MarchParams p) {
  __shared__ uint32_t kbuf[64 * kGyroDefer];
  const GyroPixel q = gyro_pixel(p);
  RayCounts rc;
  TryState ts;
  ts.ks = kbuf + threadIdx.x * kGyroDefer;
  const double T = gyro_T_simple<DEF, true, false>(p, q.v, q.i, q.j, q.valid, rc, &ts);
  try_finish(p, q.v, q.i, q.j, q.valid, T, ts, rc);
}

template <int DEF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5))) void
gyro_hier_try_kernel(MarchParams p) {
  __shared__ uint32_t kbuf[64 * kGyroDefer];
  __shared__ GyroRuns runs;
  const GyroPixel q = gyro_pixel(p);
  RayCounts rc;
  TryState ts;
  ts.ks = kbuf + threadIdx.x * kGyroDefer;
  const double T = gyro_T_hier<DEF, true, false>(p, q.v, q.i, q.j, q.valid, rc, &ts, runs);
  try_finish<true>(p, q.v, q.i, q.j, q.valid, T, ts, rc);
}

// The passes between (two_pass.hpp).  The first pass lists the membership it
// used in bit 31.
template <int DEF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void
gyro_check_kernel(MarchParams p) {
  two_pass_check(
      p, [](int, int, int, bool) {},
      [&](unsigned item, const double (&o)[3], const double (&d)[3], const double (&s)[1]) {
        return gyro_exact<DEF>(p, o, d, s[0]) != ((item >> 31) != 0u);
      });
}
template <int DEF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void
gyro_resolve_kernel(MarchParams p) {
  two_pass_resolve(
      p, [](int, int, int, bool) {},
      [&](const double (&o)[3], const double (&d)[3], double s) {
        return gyro_exact<DEF>(p, o, d, s) ? p.gyro_rho : 0.0;
      });
}

template <int DEF, int INTEG, bool AUDIT, int H = 1>
__device__ __forceinline__ double gyro_T(const MarchParams& p, int v, int i, int j, bool valid,
                                         RayCounts& rc) {
  if constexpr (INTEG == INT_HIERARCHICAL) {
    __shared__ GyroRuns runs;
    return gyro_T_hier<DEF, false, AUDIT, H>(p, v, i, j, valid, rc, nullptr, runs);
  } else {
    return gyro_T_simple<DEF, false, AUDIT>(p, v, i, j, valid, rc, nullptr);
  }
}

// One pass.
template <int DEF, int INTEG, bool AUDIT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void
gyro_kernel(MarchParams p) {
  const GyroPixel q = gyro_pixel(p);
  RayCounts rc;
  const double T = gyro_T<DEF, INTEG, AUDIT>(p, q.v, q.i, q.j, q.valid, rc);
  if (q.valid) store_pixel(p, q.v, q.i, q.j, T);
  flush_counts(p, rc);
}

// Last of the two passes: the listed rays, 64 per wave in list order (simple),
// or 4 with 16 lanes each (hierarchical: few rays, but with long chains of
// visits and guard-band samples, so the pass lasts as long as its slowest
// wave: 8074 rays of 25 M 1.18 -> 0.45 ms).
template <int INTEG>
struct GyroAgain {
  static constexpr int lanes = INTEG == INT_HIERARCHICAL ? 16 : 1;
};
template <int DEF, int INTEG>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void
gyro_redo_kernel(MarchParams p) {
  constexpr int H = GyroAgain<INTEG>::lanes;
  constexpr unsigned rays = 64 / H;
  const unsigned n = min(p.counts[0], p.redo_cap);
  const unsigned rr = (unsigned)p.res * (unsigned)p.res;
  RayCounts rc;
  for (unsigned base = blockIdx.x * rays; base < n; base += gridDim.x * rays) {
    const unsigned e = base + threadIdx.x / H;
    const bool valid = e < n && threadIdx.x % H == 0;
    const unsigned id = valid ? p.redo_list[e] : 0u;
    const unsigned v = id / rr, pix = id - v * rr;
    const int i = (int)(pix / (unsigned)p.res), j = (int)(pix - (unsigned)i * p.res);
    const double T = gyro_T<DEF, INTEG, false, H>(p, (int)v, i, j, valid, rc);
    if (valid) store_pixel(p, (int)v, i, j, T);
  }
  flush_counts(p, rc);
}

template <int DEF>
static int launch_def(const MarchParams& p, int integrator, hipStream_t s) {
  const bool hier = integrator == INT_HIERARCHICAL;
  const dim3 block(64);
  const dim3 grid(((p.res + kGyroTileI - 1) / kGyroTileI) * ((p.res + kGyroTileJ - 1) / kGyroTileJ),
                  p.n_views);
  if (p.audit && hier) {
    hipLaunchKernelGGL((gyro_kernel<DEF, INT_HIERARCHICAL, true>), grid, block, 0, s, p);
  } else if (p.audit) {
    hipLaunchKernelGGL((gyro_kernel<DEF, INT_SIMPLE, true>), grid, block, 0, s, p);
  } else if (p.redo_list) {
    const dim3 lists(std::min((p.defer_cap + 63u) / 64u, 8192u));
    const dim3 again(std::min((p.redo_cap + 63u) / 64u, 8192u));
    if (hier) {
      hipLaunchKernelGGL((gyro_hier_try_kernel<DEF>), grid, block, 0, s, p);
      hipLaunchKernelGGL((gyro_check_kernel<DEF>), lists, block, 0, s, p);
      hipLaunchKernelGGL((gyro_redo_kernel<DEF, INT_HIERARCHICAL>), again, block, 0, s, p);
    } else {
      hipLaunchKernelGGL((gyro_try_kernel<DEF>), grid, block, 0, s, p);
      hipLaunchKernelGGL((gyro_resolve_kernel<DEF>), lists, block, 0, s, p);
      hipLaunchKernelGGL((gyro_redo_kernel<DEF, INT_SIMPLE>), again, block, 0, s, p);
    }
  } else if (hier) {
    hipLaunchKernelGGL((gyro_kernel<DEF, INT_HIERARCHICAL, false>), grid, block, 0, s, p);
  } else {
    hipLaunchKernelGGL((gyro_kernel<DEF, INT_SIMPLE, false>), grid, block, 0, s, p);
  }
  return (int)hipGetLastError();
}

int launch_gyroid(const MarchParams& p, int integrator, void* stream) {
  if (p.gyro <= 0 || (integrator == INT_HIERARCHICAL && !p.fine_n))
    return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  if (p.n_defs == 0) return launch_def<GYRO_STRAIGHT>(p, integrator, s);
  if (p.gyro_tanh) return launch_def<GYRO_TANH>(p, integrator, s);
  return launch_def<GYRO_CHAIN>(p, integrator, s);
}

}  // namespace xrp
