// batch.hip - many scenes and views of uneven size in one persistent launch.
//
// The host flattens a batch into work items (scene, view, tile), grouped by
// (precision, integrator, interval march or not) and ordered within a group
// by estimated total work, smallest first.  Jobs of the interval march run in
// line.hip's form of this kernel.  Each wave of the persistent grid takes the
// next item from an atomic counter, marches its pixel tile (wave_rows x
// wave_cols blocks of 8x8 rays, one block after another) with the same
// per-ray code as the per-scene kernel (march_ray.hpp), and stamps the
// scene's first-start and last-end wall-clock times for per-scene latency.
// Every wave leaves the loop once the counter passes the item count, so the
// grid always drains.
#include <hip/hip_runtime.h>

#include "batch_items.hpp"
#include "march.hpp"
#include "march_ray.hpp"

namespace xrp {

// Two waves per SIMD: the batched scenes' hot path (gyroids, up to 200
// primitives) spills at 4 waves per SIMD and measured slower there, and
// without the cap the allocation passes 256 registers (1 wave per SIMD; the
// hierarchical form ran 16 scenes in 1,223 ms there, 751 ms at 2).  With
// registers to spare the guarded march queues its FP64 re-evaluations per
// wave (march_ray.hpp), 24 % faster on the 32-scene batch.
template <int PREC, int INTEG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void batch_kernel(BatchGroup g,
                                                    const MarchParams* __restrict__ jobs) {
  batch_items(g, jobs, [](const MarchParams& p, int v, int i, int j, bool valid, RayCounts& rc) {
    march_ray<PREC, INTEG, 4, kBlock, true>(p, v, i, j, valid, rc);
  });
}

__global__ void batch_reset_kernel(uint32_t* counters, int n_counters,
                                   unsigned long long* t_first, unsigned long long* t_done,
                                   int n_jobs, unsigned long long* stats, int n_stats) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n_counters) counters[k] = 0u;
  if (k < n_jobs) {
    t_first[k] = ~0ull;
    t_done[k] = 0ull;
  }
  if (k < n_stats) stats[k] = 0ull;
}

int launch_batch(const BatchGroup& g, int precision, int integrator, int workgroups,
                 void* stream) {
  hipStream_t s = (hipStream_t)stream;
  dim3 block(256);
  dim3 grid(workgroups);
  if (precision == PREC_FP64) {
    if (integrator == INT_HIERARCHICAL)
      hipLaunchKernelGGL((batch_kernel<PREC_FP64, INT_HIERARCHICAL>), grid, block, 0, s, g,
                         g.jobs);
    else
      hipLaunchKernelGGL((batch_kernel<PREC_FP64, INT_SIMPLE>), grid, block, 0, s, g, g.jobs);
  } else {
    if (integrator == INT_HIERARCHICAL)
      hipLaunchKernelGGL((batch_kernel<PREC_GUARDED, INT_HIERARCHICAL>), grid, block, 0, s, g,
                         g.jobs);
    else
      hipLaunchKernelGGL((batch_kernel<PREC_GUARDED, INT_SIMPLE>), grid, block, 0, s, g,
                         g.jobs);
  }
  return (int)hipGetLastError();
}

int launch_batch_reset(uint32_t* counters, int n_counters, unsigned long long* t_first,
                       unsigned long long* t_done, int n_jobs, unsigned long long* stats,
                       int n_stats, void* stream) {
  int n = n_counters > n_jobs ? n_counters : n_jobs;
  if (n_stats > n) n = n_stats;
  if (n <= 0) return 0;
  hipLaunchKernelGGL(batch_reset_kernel, dim3((n + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, counters, n_counters, t_first, t_done, n_jobs, stats,
                     n_stats);
  return (int)hipGetLastError();
}

}  // namespace xrp
