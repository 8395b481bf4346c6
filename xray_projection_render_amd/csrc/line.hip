// line.hip - gfx950 kernels of the interval march (line_march.hpp): scenes
// of convex primitives (and wide gyroids) seen along straight object-space
// lines.
//
// Bound by VALU issue on tessellations (6.1e11 instructions a second, half the
// rate of 2-cycle instructions with the roots' minima, selects and
// transcendentals between) and, on collections, by the latency of serial chains
// (2.2e11, 3 waves per SIMD): the runs of every listed child (about 80 FP32
// instructions each) and one pass over the wave's run slots per change of the
// density, where the sampling marches evaluated every listed child at every
// sample they could not settle.  Whole calls, sampling march -> interval march:
// strut lattice 30 x 500^2 7.39 -> 0.88 ms, hierarchical bytes 12 x 512^2 10.0 ->
// 1.05 ms; 60 primitives hierarchical 8 x 256^2 8.59 -> 0.58 ms; three primitives
// 2 x 128^2 0.097 -> 0.041 ms; 10 uneven scenes batched 22.8 -> 1.92 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "batch_items.hpp"
#include "line_march.hpp"
#include "march.hpp"

namespace xrp {

extern __shared__ __align__(16) unsigned char line_lds[];

// Ray tile of one wave: 8 x 8 for collections (a narrow pencil of rays keeps
// few children through the wave's culling), 32 x 2 for tessellations.
template <int KIND>
struct LineTile {
  static constexpr int I = KIND == LINE_TESS ? 32 : 8, J = 64 / I;
};

// Waves per SIMD the kernels are compiled for.
template <int KIND>
struct LineWaves {
  static constexpr int n = KIND == LINE_TESS ? 4 : 3;
};

struct LinePixel {
  int v, i, j;
  bool valid;
};
template <int KIND>
__device__ __forceinline__ LinePixel line_pixel(const MarchParams& p) {
  constexpr int TI = LineTile<KIND>::I, TJ = LineTile<KIND>::J;
  const int lane = threadIdx.x;
  const int tiles_j = (p.res + TJ - 1) / TJ;
  const int ti = blockIdx.x / tiles_j, tj = blockIdx.x - ti * tiles_j;
  LinePixel q;
  q.v = blockIdx.y;
  q.i = ti * TI + lane / TJ;
  q.j = tj * TJ + lane % TJ;
  q.valid = q.i < p.res && q.j < p.res;
  return q;
}

// T of one pixel per lane: the march, then, ray by ray, the ones it stopped.
// The FP64 evaluator is then called with nothing of the march live: called
// from within it, it cost 30-50 spilled registers in the march's loops.
template <int INTEG, bool AUDIT, int KIND>
__device__ __forceinline__ double line_pixel_T(const MarchParams& p, int v, int i, int j,
                                               bool valid, const LineSlots& S, int cap,
                                               RayCounts& rc) {
  bool stopped;
  double T = line_T<INTEG, AUDIT, KIND>(p, v, i, j, valid, S, cap, rc, stopped);
  for (unsigned long long m = __ballot(valid && stopped); __builtin_expect(m != 0ull, 0);
       m &= m - 1ull) {
    const int own = (int)__builtin_ctzll(m);
    const double t = line_T_exact<INTEG>(p, __builtin_amdgcn_readlane(v, own),
                                         __builtin_amdgcn_readlane(i, own),
                                         __builtin_amdgcn_readlane(j, own), own, rc);
    if ((int)(threadIdx.x & 63) == own) T = t;
  }
  return T;
}

template <int INTEG, bool AUDIT, int KIND>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(LineWaves<KIND>::n))) void
line_kernel(MarchParams p) {
  const LineSlots S = line_slots(line_lds, p.line_cap);
  const LinePixel q = line_pixel<KIND>(p);
  RayCounts rc;
  const double T = line_pixel_T<INTEG, AUDIT, KIND>(p, q.v, q.i, q.j, q.valid, S, p.line_cap, rc);
  if (q.valid) store_pixel(p, q.v, q.i, q.j, T);
  flush_counts(p, rc);
}

// First pass of the two-pass form: the stopped rays are appended to
// p.redo_list (one atomic per wave).
template <int KIND>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(LineWaves<KIND>::n))) void
line_try_kernel(MarchParams p) {
  const LineSlots S = line_slots(line_lds, p.line_cap);
  const LinePixel q = line_pixel<KIND>(p);
  RayCounts rc;
  bool stopped;
  const double T = line_T<INT_SIMPLE, false, KIND>(p, q.v, q.i, q.j, q.valid, S, p.line_cap, rc,
                                                   stopped);
  if (q.valid && !stopped) store_pixel(p, q.v, q.i, q.j, T);
  const unsigned long long m = __ballot(q.valid && stopped);
  if (m) {
    unsigned base = 0;
    if ((threadIdx.x & 63) == 0) base = atomicAdd(p.counts, (unsigned)__popcll(m));
    base = (unsigned)__shfl((int)base, 0, 64);
    const unsigned e = base + (unsigned)__popcll(m & __lanemask_lt());
    if (q.valid && stopped) {
      if (e < p.redo_cap)
        p.redo_list[e] = ((unsigned)q.v * (unsigned)p.res + (unsigned)q.i) * (unsigned)p.res +
                         (unsigned)q.j;
      else
        p.counts[3] = 1u;  // no room: the caller renders again in one pass
    }
  }
  flush_counts(p, rc);
}

// Second pass: one listed ray per wave (grid-stride).
__global__ __launch_bounds__(64) void line_redo_kernel(MarchParams p) {
  const unsigned n = min(p.counts[0], p.redo_cap);
  const unsigned rr = (unsigned)p.res * (unsigned)p.res;
  RayCounts rc;
  for (unsigned e = blockIdx.x; e < n; e += gridDim.x) {
    const unsigned id = p.redo_list[e], v = id / rr, pix = id - v * rr;
    const int i = (int)(pix / (unsigned)p.res), j = (int)(pix - (unsigned)i * p.res);
    const double T = line_T_exact<INT_SIMPLE>(p, (int)v, i, j, 0, rc);
    if (threadIdx.x == 0) store_pixel(p, (int)v, i, j, T);
  }
  flush_counts(p, rc);
}

// Batched form: the items of one group (batch.hip), every job of it with
// line != LINE_NONE, one wave per workgroup.  2 waves per SIMD: the item loop
// spills at 3, with the same time (10 scenes 2.70 against 2.69 ms; the run
// slots' LDS admits 2 to 4).
template <int INTEG>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void
batch_line_kernel(BatchGroup g, const MarchParams* __restrict__ jobs) {
  const LineSlots S = line_slots(line_lds, g.line_cap);
  batch_items(g, jobs, [&](const MarchParams& p, int v, int i, int j, bool valid, RayCounts& rc) {
    const double T = line_pixel_T<INTEG, false, LINE_NONE>(p, v, i, j, valid, S, p.line_cap, rc);
    if (valid) store_pixel(p, v, i, j, T);
  });
}

int launch_batch_line(const BatchGroup& g, int integrator, int workgroups, void* stream) {
  if (g.line_cap < 1) return (int)hipErrorInvalidValue;
  const size_t lds = line_lds_bytes(g.line_cap);
  if (integrator == INT_HIERARCHICAL)
    hipLaunchKernelGGL((batch_line_kernel<INT_HIERARCHICAL>), dim3(workgroups), dim3(64), lds,
                       (hipStream_t)stream, g, g.jobs);
  else
    hipLaunchKernelGGL((batch_line_kernel<INT_SIMPLE>), dim3(workgroups), dim3(64), lds,
                       (hipStream_t)stream, g, g.jobs);
  return (int)hipGetLastError();
}

template <int KIND>
static int launch_kind(const MarchParams& p, int integrator, hipStream_t s) {
  constexpr int TI = LineTile<KIND>::I, TJ = LineTile<KIND>::J;
  const dim3 block(64);
  const dim3 grid(((p.res + TI - 1) / TI) * ((p.res + TJ - 1) / TJ), p.n_views);
  const size_t lds = line_lds_bytes(p.line_cap);
  if (integrator == INT_HIERARCHICAL && p.audit) {
    hipLaunchKernelGGL((line_kernel<INT_HIERARCHICAL, true, KIND>), grid, block, lds, s, p);
  } else if (integrator == INT_HIERARCHICAL) {
    hipLaunchKernelGGL((line_kernel<INT_HIERARCHICAL, false, KIND>), grid, block, lds, s, p);
  } else if (p.audit) {
    hipLaunchKernelGGL((line_kernel<INT_SIMPLE, true, KIND>), grid, block, lds, s, p);
  } else if (p.redo_list) {
    hipLaunchKernelGGL((line_try_kernel<KIND>), grid, block, lds, s, p);
    hipLaunchKernelGGL(line_redo_kernel, dim3(std::min(p.redo_cap, 4096u)), block, 0, s, p);
  } else {
    hipLaunchKernelGGL((line_kernel<INT_SIMPLE, false, KIND>), grid, block, lds, s, p);
  }
  return (int)hipGetLastError();
}

int launch_line(const MarchParams& p, int integrator, void* stream) {
  if (p.line_cap < 1 || (p.line != LINE_COLL && p.line != LINE_TESS))
    return (int)hipErrorInvalidValue;
  return p.line == LINE_TESS ? launch_kind<LINE_TESS>(p, integrator, (hipStream_t)stream)
                             : launch_kind<LINE_COLL>(p, integrator, (hipStream_t)stream);
}

}  // namespace xrp
