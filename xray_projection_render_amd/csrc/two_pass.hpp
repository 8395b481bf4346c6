// two_pass.hpp - the end of a first-pass wave, shared by the two-pass marches
// (march.hip, gyroid.hip).
#pragma once
#include "march_ray.hpp"

namespace xrp {

// End of a first-pass wave of the two-pass marches; every lane calls it.
// A ray with nothing deferred stores its pixel (SPEC: every ray not stopped
// does, its listed samples to be checked, and its counts follow its items
// in defer_k: samples, fine samples, settled samples).  The rays with
// deferred items are appended, with T and the items (ts.ks), to the
// resolve pass's lists in lane order (an exclusive scan of the counts over
// the wave, one atomic per wave and list).  The stopped ones, and a wave's deferring rays when
// the lists are full, go to p.redo_list.  The counts of a ray go to rc only
// when it is not marched again.
template <bool SPEC = false>
__device__ __forceinline__ void try_finish(const MarchParams& p, int v, int i, int j,
                                           bool valid, double T, TryState& ts,
                                           RayCounts& rc) {
  const int lane = threadIdx.x & 63;
  const unsigned id = ((unsigned)v * (unsigned)p.res + (unsigned)i) * (unsigned)p.res +
                      (unsigned)j;
  if (valid && !ts.aborted && (SPEC || ts.cnt == 0)) store_pixel(p, v, i, j, T);
  bool defer = valid && !ts.aborted && ts.cnt > 0;
  const unsigned kc = ts.cnt + (SPEC ? 3u : 0u);  // words in defer_k
  const unsigned long long dm = __ballot(defer);
  if (dm) {
    unsigned incl = defer ? kc : 0u;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned t = (unsigned)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += t;
    }
    const unsigned total = (unsigned)__shfl((int)incl, 63, 64);
    unsigned eb = 0, kb = 0;
    if (lane == 0) {
      eb = atomicAdd(p.counts + 1, (unsigned)__popcll(dm));
      kb = atomicAdd(p.counts + 2, total);
    }
    eb = (unsigned)__shfl((int)eb, 0, 64);
    kb = (unsigned)__shfl((int)kb, 0, 64);
    const bool fits = eb + (unsigned)__popcll(dm) <= p.defer_cap && kb + total <= p.k_cap;
    if (defer && fits) {
      const unsigned e = eb + (unsigned)__popcll(dm & __lanemask_lt());
      const unsigned k0 = kb + incl - kc;
      p.defer_T[e] = T;
      p.defer_ray[e] = id;
      p.defer_cnt[e] = ts.cnt;
      p.defer_kfirst[e] = k0;
      for (unsigned c = 0; c < ts.cnt; ++c) p.defer_k[k0 + c] = ts.ks[c];
      if (SPEC) {
        p.defer_k[k0 + ts.cnt] = ts.samples;
        p.defer_k[k0 + ts.cnt + 1] = ts.fine;
        p.defer_k[k0 + ts.cnt + 2] = ts.skipped;
      }
    } else if (defer) {
      // the lists are full: the wave's rays go to the redo list, and its
      // entries below the cap are marked empty for the resolve pass
      const unsigned e = eb + (unsigned)__popcll(dm & __lanemask_lt());
      if (e < p.defer_cap) p.defer_cnt[e] = 0u;
      ts.aborted = true;
    }
  }
  if (valid && !ts.aborted) {
    rc.samples += ts.samples;
    rc.skipped += ts.skipped;
    rc.fine += ts.fine;
  }
  const unsigned long long m = __ballot(valid && ts.aborted);
  if (m) {
    unsigned base = 0;
    if (lane == 0) base = atomicAdd(p.counts, (unsigned)__popcll(m));
    base = (unsigned)__shfl((int)base, 0, 64);
    const unsigned e = base + (unsigned)__popcll(m & __lanemask_lt());
    if (valid && ts.aborted) {
      if (e < p.redo_cap)
        p.redo_list[e] = id;
      else
        p.counts[3] = 1u;  // no room: the caller renders again in one pass
    }
  }
  flush_counts(p.stats, rc);
}

}  // namespace xrp
