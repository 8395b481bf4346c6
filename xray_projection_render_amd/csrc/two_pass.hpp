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
  flush_counts(p, rc);
}

// Check pass of the two-pass hierarchical march: 64 entries per wave
// (grid-stride), their listed samples spread one per lane.  Each listed
// sample, (nn << 4) | m, is at R[nn] for m = 15 and otherwise at
// R[nn-1] + DS/10 plus m more additions of DS/10 (the m-th sample of step
// nn's fine walk, main.go:180-186).  differs(item, origin, direction, {s})
// says whether the FP32 value that the first pass used is not its FP64
// density; a ray with any that differs goes to the redo list, whose pass overwrites its pixel, and its first
// pass counts (after its items) are taken back from the stats.
// One listed sample per lane rather than one ray per lane: on C5 18.6 ->
// 11.3 ms (a wave ran as many rounds as its longest list, 1-14 samples).
// begin(v, i, j, valid) is called by every lane with its own entry's pixel.
template <typename Begin, typename Differs>
__device__ __forceinline__ void two_pass_check(const MarchParams& p, Begin begin,
                                               Differs differs) {
  const unsigned n = min(p.counts[1], p.defer_cap), nk = min(p.counts[2], p.k_cap);
  const unsigned rr = (unsigned)p.res * (unsigned)p.res;
  const double dsf = p.ds_fine;
  unsigned long long reeval = 0, rays = 0, back_s = 0, back_f = 0, back_k = 0;
  for (unsigned base = blockIdx.x * 64u; base < n; base += gridDim.x * 64u) {
    const unsigned e = base + threadIdx.x;
    unsigned cnt = 0u, k0 = 0u, id = 0u;
    if (e < n) {
      cnt = p.defer_cnt[e];
      k0 = p.defer_kfirst[e];
      if (k0 + cnt + 3u > nk) cnt = 0u;
      // an entry marked empty (cnt 0, lists full) has no ray or k0 written
      if (cnt != 0u)
        id = p.defer_ray[e];
      else
        k0 = 0u;
    }
    const unsigned v = id / rr, pix = id - v * rr;
    const int i = (int)(pix / (unsigned)p.res), j = (int)(pix - (unsigned)i * p.res);
    begin((int)v, i, j, cnt != 0u);
    const Ray r = make_ray(p, p.views[p.view_offset + (int)v], i, j);
    // The wave's listed samples, one per lane: lane l of round fb takes
    // sample t = fb + l of the concatenated lists, owned by the ray (lane o)
    // whose inclusive prefix sum of counts is the first above t.
    unsigned incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned u = __shfl_up(incl, off, 64);
      if ((int)threadIdx.x >= off) incl += u;
    }
    const unsigned total = __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
    unsigned long long bad = 0ull;  // lanes whose ray holds a wrong guess
    for (unsigned fb = 0; fb < total; fb += 64u) {
      const unsigned t = fb + threadIdx.x;
      int o = 0;
#pragma unroll
      for (int step = 32; step >= 1; step >>= 1)
        if (__shfl(incl, o + step - 1, 64) <= t) o += step;
      const bool has = t < total;
      const unsigned c = t - (__shfl(incl, o, 64) - __shfl(cnt, o, 64));
      const unsigned ko = __shfl(k0, o, 64);
      double ro[3], rd[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        ro[q] = __shfl(r.o[q], o, 64);
        rd[q] = __shfl(r.d[q], o, 64);
      }
      bool wrong = false;
      if (has) {
        const unsigned item = p.defer_k[ko + c], nn = (item & 0x7fffffffu) >> 4,
                       m = item & 15u;
        double sq[1];
        if (m == 15u) {
          sq[0] = p.s_table[nn];
        } else {
          sq[0] = (nn == 0 ? p.smin : p.s_table[nn - 1]) + dsf;
          for (unsigned q = 0; q < m; ++q) sq[0] += dsf;
        }
        wrong = differs(item, ro, rd, sq);
      }
      for (unsigned long long w = __ballot(wrong); w; w &= w - 1ull) {
        const int l = (int)__builtin_ctzll(w);
        bad |= 1ull << __builtin_amdgcn_readlane(o, l);
      }
    }
    if (cnt == 0u) continue;
    const bool same = ((bad >> threadIdx.x) & 1ull) == 0ull;
    if (same) {
      reeval += cnt;
      ++rays;
    } else {
      back_s += p.defer_k[k0 + cnt];
      back_f += p.defer_k[k0 + cnt + 1];
      back_k += p.defer_k[k0 + cnt + 2];
      const unsigned at = atomicAdd(p.counts, 1u);
      if (at < p.redo_cap)
        p.redo_list[at] = id;
      else
        p.counts[3] = 1u;  // no room: the caller renders again in one pass
    }
  }
  if (unsigned long long* stats = stat_slot(p)) {
    const unsigned long long a = wave_total(reeval), b = wave_total(rays), c = wave_total(back_s),
                             d = wave_total(back_f), f = wave_total(back_k);
    if (threadIdx.x == 0) {
      if (a) atomicAdd(stats + ST_REEVAL, a);
      if (b) atomicAdd(stats + ST_DEFERRED, b);
      // the counts of rays marched again, taken back (mod 2^64)
      if (c) atomicAdd(stats + ST_SAMPLES, 0ull - c);
      if (d) atomicAdd(stats + ST_FINE, 0ull - d);
      if (f) atomicAdd(stats + ST_SKIPPED, 0ull - f);
    }
  }
}

// Resolve pass: 64 entries of the first pass's lists per wave (grid-stride
// over min(counts[1], defer_cap) entries), their deferred samples spread
// one per lane.  Each is evaluated in FP64, its term (rho * dm) * ds staged
// in LDS, and each entry's lane adds its own terms in sample order into Ta,
// as the one-pass march sums its re-evaluated terms; the pixel is T + Ta.
// exact(origin, direction, s) is the FP64 density.
// A wave whose entries did not all fit wrote none of them but their count
// 0 (its rays are in the redo list), and entries past the cap are not read.
template <typename Begin, typename Exact>
__device__ __forceinline__ void two_pass_resolve(const MarchParams& p, Begin begin,
                                                 Exact exact) {
  __shared__ double terms[64];
  const unsigned n = min(p.counts[1], p.defer_cap), nk = min(p.counts[2], p.k_cap);
  const unsigned rr = (unsigned)p.res * (unsigned)p.res;
  const double ds = p.ds, dm = p.dm;
  unsigned long long reeval = 0, rays = 0;
  for (unsigned base = blockIdx.x * 64u; base < n; base += gridDim.x * 64u) {
    const unsigned e = base + threadIdx.x;
    unsigned cnt = 0u, k0 = 0u, id = 0u;
    if (e < n) {
      cnt = p.defer_cnt[e];
      k0 = p.defer_kfirst[e];
      if (k0 + cnt > nk) cnt = 0u;
      // an entry marked empty (cnt 0, lists full) has no ray or k0 written
      if (cnt != 0u)
        id = p.defer_ray[e];
      else
        k0 = 0u;
    }
    const unsigned v = id / rr, pix = id - v * rr;
    const int i = (int)(pix / (unsigned)p.res), j = (int)(pix - (unsigned)i * p.res);
    begin((int)v, i, j, cnt != 0u);
    const Ray r = make_ray(p, p.views[p.view_offset + (int)v], i, j);
    // sample t of the concatenated lists belongs to the lane o whose
    // inclusive prefix sum of counts is the first above t
    unsigned incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned u = __shfl_up(incl, off, 64);
      if ((int)threadIdx.x >= off) incl += u;
    }
    const unsigned excl = incl - cnt;
    const unsigned total = __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
    double Ta = 0.0;
    for (unsigned fb = 0; fb < total; fb += 64u) {
      const unsigned t = fb + threadIdx.x;
      int o = 0;
#pragma unroll
      for (int step = 32; step >= 1; step >>= 1)
        if (__shfl(incl, o + step - 1, 64) <= t) o += step;
      const unsigned c = t - __shfl(excl, o, 64);
      const unsigned ko = __shfl(k0, o, 64);
      double ro[3], rd[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        ro[q] = __shfl(r.o[q], o, 64);
        rd[q] = __shfl(r.d[q], o, 64);
      }
      double term = 0.0;
      if (t < total) {
        const double sk = p.s_table[p.defer_k[ko + c]];
        term = (exact(ro, rd, sk) * dm) * ds;
      }
      terms[threadIdx.x] = term;
      __syncthreads();
      const unsigned lo = excl > fb ? excl : fb, hi = incl < fb + 64u ? incl : fb + 64u;
      for (unsigned x = lo; x < hi; ++x) Ta += terms[x - fb];
      __syncthreads();
    }
    if (cnt != 0u) {
      store_pixel(p, (int)v, i, j, p.defer_T[e] + Ta);
      reeval += cnt;
      ++rays;
    }
  }
  if (unsigned long long* stats = stat_slot(p)) {
    const unsigned long long a = wave_total(reeval), b = wave_total(rays);
    if (threadIdx.x == 0) {
      if (a) atomicAdd(stats + ST_REEVAL, a);
      if (b) atomicAdd(stats + ST_DEFERRED, b);
    }
  }
}

}  // namespace xrp
