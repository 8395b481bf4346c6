// batch_items.hpp - work-queue bookkeeping shared by the batched persistent
// kernels (batch.hip, line.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "march.hpp"
#include "march_ray.hpp"

namespace xrp {

// Adds the wave's sum of v; nothing, on a wave-uniform condition, where it is
// zero.
__device__ __forceinline__ void wave_add(unsigned long long* p, unsigned long long v,
                                         unsigned long long* sink) {
  if (!__ballot(v != 0ull)) return;
  v = wave_sum(v);
  atomicAdd(lane_slot(p, sink), first_lane() ? v : 0ull);
}

// Close a wave's run of items of scene `job`: its stats, once, and its
// last-end stamp.  All conditions are wave-uniform (job and p.stats are).
__device__ __forceinline__ void close_run(const BatchGroup& g,
                                          const MarchParams* __restrict__ jobs, int job,
                                          const RayCounts& rc) {
  const MarchParams& p = jobs[job];
  if (p.stats) {
    wave_add(p.stats + ST_SAMPLES, rc.samples, g.sink);
    wave_add(p.stats + ST_REEVAL, rc.reeval, g.sink);
    wave_add(p.stats + ST_AUDIT_MISS, rc.miss, g.sink);
    wave_add(p.stats + ST_FINE, rc.fine, g.sink);
    wave_add(p.stats + ST_SKIPPED, rc.skipped, g.sink);
  }
  atomicMax(lane_slot(g.t_done + job, g.sink), (unsigned long long)wall_clock64());
}

// Every wave of a persistent grid takes items until the counter passes the
// last one, without LDS or barriers of the loop's own (the interval march keeps
// a wave's run slots and child list in LDS, line.hip); march(p, v, i, j, valid,
// rc) renders one pixel per lane, called by every lane of the wave.
template <class March>
__device__ __forceinline__ void batch_items(const BatchGroup& g,
                                            const MarchParams* __restrict__ jobs, March&& march) {
  const int lane = threadIdx.x & 63;
  const int tile_i = 8 * g.wave_rows, tile_j = 8 * g.wave_cols;
  for (;;) {
    const uint32_t got =
        atomicAdd(lane_slot(g.counter, g.sink), first_lane() ? kItemsPerGrab : 0u);
    const uint32_t t0 = __builtin_amdgcn_readfirstlane(got);
    if (t0 >= g.n_tiles) break;
    const uint32_t t1 = min(t0 + kItemsPerGrab, g.n_tiles);
    int run_job = -1;
    RayCounts rc;
    for (uint32_t t = t0; t < t1; ++t) {
      // job holding item t: last job whose tile_start <= t
      int lo = 0, hi = g.n_jobs - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (g.tile_start[mid] <= t)
          lo = mid;
        else
          hi = mid - 1;
      }
      const int job = __builtin_amdgcn_readfirstlane(lo);
      if (job != run_job) {
        if (run_job >= 0) {
          close_run(g, jobs, run_job, rc);
          rc = RayCounts();
        }
        atomicMin(lane_slot(g.t_first + job, g.sink), (unsigned long long)wall_clock64());
        run_job = job;
      }
      const MarchParams& p = jobs[job];
      const uint32_t local = t - g.tile_start[job];
      const int tiles_i = (p.res + tile_i - 1) / tile_i, tiles_j = (p.res + tile_j - 1) / tile_j;
      const uint32_t per_view = (uint32_t)tiles_i * (uint32_t)tiles_j;
      const int v = (int)(local / per_view);
      const uint32_t rem = local - (uint32_t)v * per_view;
      const int ti = (int)(rem / (uint32_t)tiles_j), tj = (int)(rem - (uint32_t)ti * tiles_j);
      for (int bi = 0; bi < g.wave_rows; ++bi)
        for (int bj = 0; bj < g.wave_cols; ++bj) {
          const int i = ti * tile_i + bi * 8 + (lane >> 3);
          const int j = tj * tile_j + bj * 8 + (lane & 7);
          march(p, v, i, j, i < p.res && j < p.res, rc);
        }
    }
    close_run(g, jobs, run_job, rc);
  }
}

}  // namespace xrp
