// gyroid_march.hpp - guarded march of a tessellated gyroid: a root
// tessellation whose unit cell holds one gyroid with whole periods along
// each cell axis (api.cpp gyroid_plan has the rule), under any deformation
// chain.  The scene is then one periodic level set inside a box, and a march
// over it needs none of the node walk of eval_block.hpp.
//
// The march is bound by VALU issue (first passes: 7.1e11 instructions a second,
// 57 % of the rate of 2-cycle instructions, with a visit's 12 transcendentals of 8
// cycles, selects and minima of 4 between; waves wait for issue half their
// cycles and more, for anything else 7 to 15 %), so everything per visit
// that does not depend on the sample is hoisted, the cell wrap is left out
// (the phase is reduced to [-0.5, 0.5] periods anyway, exactly, by one fma
// against the rounded period count), and each lane runs its own state
// machine: every visit evaluates one sample of every lane that has any left,
// coarse or fine.
//
// A sample whose FP32 | |g| - thickness |, or distance to the box, is within
// its band is evaluated in FP64 (or, in a first pass, listed).  The level's
// band (p.gyro_band) is this evaluation's own error bound.
//
// Between evaluated samples the second-order reach (eval_block.hpp
// gyroid_reach) settles samples forwards, and in the hierarchical march also
// backwards from the right end of a step with a density change: the fine
// samples within reach of either end have that end's density, which leaves
// about one to evaluate where the walk took four or five visits.
//
// Sheared 6^3 gyroid cells against the general march: 16 x 512^2 rays at step
// 0.001, simple, 1.58 -> 0.53 ms; 24 x 1024^2, hierarchical, 17.1 -> 3.84 ms
// (first pass 12.8 -> 3.15, the FP64 passes 4.0 -> 0.54).
//
// Sums: every term is (rho * dm) * ds of one density value, so T is a number
// of equal additions in a fixed order; the marches count and add at the end
// (the same additions, hence the same bits, as march_ray.hpp).
#pragma once
#include "line_march.hpp"
#include "march_ray.hpp"

namespace xrp {

// Runs of inside coarse samples a lane keeps before it adds them (LDS).
constexpr int kGyroRuns = 32;
// Guard-band samples a ray may list in a first pass (LDS: 2 KiB a wave; the
// bands leave most rays none).
constexpr uint32_t kGyroDefer = 8;

// What the march does for the deformation chain: nothing, one tanh
// displacement with its axes as 0 / 1 weights, or the general chain.
enum GyroDef { GYRO_STRAIGHT, GYRO_TANH, GYRO_CHAIN };

// The scene's constants, uniform over the launch.
struct GyroScene {
  float b0, b1, b2, b3, b4, b5, gb;  // the box and its band
  float cx, cy, cz, rv, rv_lo;       // centre, periods per length (two floats)
  float th, band;                    // level and band
  float two_M, e1, e3, inv;          // reach: 2M, slope error (and 3 times), 1/scale
  float per, far, first;             // samples per unit of box distance, of reach times M,
                                     // and of | |g| - th | (1 / |grad g|)
  float A, k, Ak, sx, sy, sz, ax, ay, az;  // GYRO_TANH
};

template <int DEF>
__device__ __forceinline__ GyroScene gyro_scene(const MarchParams& p, float per) {
  const DevNode &t = p.nodes[0], &g = p.nodes[p.gyro];
  GyroScene s;
  s.b0 = t.f[0], s.b1 = t.f[1], s.b2 = t.f[2], s.b3 = t.f[3], s.b4 = t.f[4], s.b5 = t.f[5];
  s.gb = t.g[1];
  s.cx = g.f[0], s.cy = g.f[1], s.cz = g.f[2], s.rv = g.f[6], s.rv_lo = g.f[7];
  s.th = g.f[4], s.band = p.gyro_band;
  s.two_M = 2.0f * g.g[6], s.e1 = g.g[7], s.e3 = 3.0f * g.g[7];
  s.inv = g.g[3];
  // the reach keeps eval_block.hpp's 1e-4 in hand
  s.per = per, s.far = g.g[1] * g.g[5] * per * (1.0f - 1e-4f), s.first = g.g[4] * per;
  if constexpr (DEF == GYRO_TANH) {
    const DevDeform& f = p.defs[0];
    s.A = f.f[0], s.k = f.f[1], s.Ak = f.f[0] * f.f[1];
    s.sx = f.src == 0 ? 1.0f : 0.0f, s.sy = f.src == 1 ? 1.0f : 0.0f;
    s.sz = f.src == 2 ? 1.0f : 0.0f;
    s.ax = f.axis == 0 ? 1.0f : 0.0f, s.ay = f.axis == 1 ? 1.0f : 0.0f;
    s.az = f.axis == 2 ? 1.0f : 0.0f;
  }
  return s;
}

// One sample: inside (by FP32), in a guard band, and the samples ahead and
// behind that have its density.
struct GyroEval {
  bool in, amb;
  float ahead, behind;
};

__device__ __forceinline__ void gyro_phase(float x, float c, const GyroScene& g, float& s,
                                           float& co) {
  const float w = x - c;
  const float n = rintf(w * g.rv);
  const float r = fmaf(w, g.rv_lo, fmaf(w, g.rv, -n));
  s = __builtin_amdgcn_sinf(r);
  co = __builtin_amdgcn_cosf(r);
}

// Reach, times M, to a level at distance c of |g| (less its band) along a ray
// whose slope towards it is as = |slope| in size, off by at most e1: moving
// towards it, and away from it.  Towards: the root of c - (as + e1) s -
// M s^2 / 2, (q - as - e1) / M with q = sqrt((as + e1)^2 + 2 M c).  Away: that
// of c + (as - e1) s - M s^2 / 2, (q' + as - e1) / M, whose q' = sqrt((as -
// e1)^2 + 2 M c) is at least q - 2 e1: one root serves both.  1e-6 q covers
// the rounding of the root and, where they cancel, of the difference: a loss of
// 1e-6 of slope over curvature, 1e-4 of a fine step of 1e-4 on cells of 1/6.
// (2 c / (q + as + e1) does not cancel but divides: simple first pass 559 against
// 499 us, hierarchical 3.25 against 3.15 ms.)
__device__ __forceinline__ void gyro_reach(const GyroScene& g, float c, float as, float& to,
                                           float& away) {
  const float b = as + g.e1;
  const float q = __builtin_amdgcn_sqrtf(fmaf(b, b, g.two_M * c)) * (1.0f - 1e-6f);
  to = q - b;
  away = q + (as - g.e3);
}

template <int DEF>
__device__ __forceinline__ GyroEval gyro_eval(const MarchParams& p, const GyroScene& g, float x,
                                              float y, float z, float vx, float vy, float vz) {
  if constexpr (DEF == GYRO_TANH) {
    const float s = fmaf(g.sx, x, fmaf(g.sy, y, g.sz * z));
    const float vs = fmaf(g.sx, vx, fmaf(g.sy, vy, g.sz * vz));
    const float t = tanh_hw(g.k * s);
    const float dq = g.A * t, dv = g.Ak * fmaf(-t, t, 1.0f) * vs;
    x = fmaf(g.ax, dq, x), y = fmaf(g.ay, dq, y), z = fmaf(g.az, dq, z);
    vx = fmaf(g.ax, dv, vx), vy = fmaf(g.ay, dv, vy), vz = fmaf(g.az, dv, vz);
  } else if constexpr (DEF == GYRO_CHAIN) {
    deform32_jvp(p.defs, p.n_defs, x, y, z, vx, vy, vz);
  }
  const float e = fmaxf(fmaxf(fmaxf(g.b0 - x, x - g.b1), fmaxf(g.b2 - y, y - g.b3)),
                        fmaxf(g.b4 - z, z - g.b5));
  float sx, cx, sy, cy, sz, cz;
  gyro_phase(x, g.cx, g, sx, cx);
  gyro_phase(y, g.cy, g, sy, cy);
  gyro_phase(z, g.cz, g, sz, cz);
  const float gg = fmaf(sx, cy, fmaf(sy, cz, sz * cx));
  const float ag = fabsf(gg), a = ag - g.th;
  const float g1 = fmaf(fmaf(cx, cy, -sz * sx), vx,
                        fmaf(fmaf(cy, cz, -sx * sy), vy, fmaf(cz, cx, -sy * sz) * vz)) *
                   g.inv;
  GyroEval o;
  const bool in_box = e < -g.gb;
  o.in = e <= 0.0f && a < 0.0f;
  // in the box's band a sample clear of the level is 0 on either side
  o.amb = !(e > g.gb) && a < g.band && (!in_box || a > -g.band);
  // The level nearest, on g's side of zero, and (inside the sheet) the other
  // one: |g| falls towards that one, and towards the nearest from outside.
  const bool falls = (gg < 0.0f) != (g1 < 0.0f);  // |g| along the ray
  float to1, away1, to2, away2;
  const float c1 = fabsf(a) - g.band;
  gyro_reach(g, c1, fabsf(g1), to1, away1);
  gyro_reach(g, ag + g.th - g.band, fabsf(g1), to2, away2);
  const bool near1 = falls == (a >= 0.0f);
  const float fa = fminf(near1 ? to1 : away1, falls ? to2 : away2);
  const float fb = fminf(near1 ? away1 : to1, falls ? away2 : to2);
  const float r1 = c1 * g.first, box = (fabsf(e) - g.gb) * g.per;
  o.ahead = in_box ? fminf(fmaxf(r1, fa * g.far), box) : box;
  o.behind = in_box ? fminf(fmaxf(r1, fb * g.far), box) : box;
  return o;
}

// FP64 membership at distance s along the ray (density64's operations; the
// constants through scalar loads).
template <int DEF>
__device__ __forceinline__ bool gyro_exact(const MarchParams& p, const double (&o)[3],
                                           const double (&d)[3], double s) {
  double x = o[0] + d[0] * s, y = o[1] + d[1] * s, z = o[2] + d[2] * s;
  const LineNodes N = (LineNodes)line_uniform(p.nodes);
  const LineDefs D = (LineDefs)line_uniform(p.defs);
  if constexpr (DEF == GYRO_TANH) {
    DevDeform f;
    f.kind = D_TANH;
    f.axis = D[0].axis;
    f.src = D[0].src;
    f.d[0] = D[0].d[0];
    f.d[1] = D[0].d[1];
    deform64(&f, 1, x, y, z);
  } else if constexpr (DEF == GYRO_CHAIN) {
    line_deform64(D, p.n_defs, x, y, z);
  }
  if (!line_wrap64(N, x, y, z)) return false;
  double c[14];
#pragma unroll
  for (int q = 0; q < 5; ++q) c[q] = N[p.gyro].d[q];
  return line_gyroid64(c, x, y, z);
}

// T + c added n times, in order.
__device__ __forceinline__ double gyro_add(double T, double c, unsigned n) {
  for (; n >= 4u; n -= 4u) {
    T += c;
    T += c;
    T += c;
    T += c;
  }
  for (; n; --n) T += c;
  return T;
}

// Appends an item to a ray's list; false when it has too many.
__device__ __forceinline__ bool gyro_list(const MarchParams& p, TryState& ts, uint32_t item) {
  const uint32_t most = min(p.defer_max, kGyroDefer);
  if (ts.cnt < most) ts.ks[ts.cnt] = item;
  return ++ts.cnt <= most;
}

// Optical depth of pixel (i, j) of view v, simple integrator.  Every lane of
// the wave calls it together.  TRY: guard-band samples are listed and their
// terms left out, as march_T_guarded_inline<1, true> does.  Otherwise a lane
// at such a sample waits until no lane of the wave can go on, and all that
// wait evaluate theirs in FP64 together.  AUDIT: every other sample is
// evaluated in FP64 too and compared.
template <int DEF, bool TRY, bool AUDIT>
__device__ __forceinline__ double gyro_T_simple(const MarchParams& p, int v, int i, int j,
                                                bool valid, RayCounts& rc, TryState* ts) {
  const double ds = p.ds;
  const GyroScene g = gyro_scene<DEF>(p, p.skip_inv);
  Ray r;
  r.o[0] = r.o[1] = r.o[2] = 0.0;
  r.d[0] = r.d[1] = r.d[2] = 0.0;
  int k = 0, k_hi = -1;
  if (valid) {
    r = make_ray(p, p.views[p.view_offset + v], i, j);
    double t_in, t_out;
    if (clip_ray(p, r, t_in, t_out)) clip_range(p, t_in, t_out, k, k_hi);
  }
  const float d0 = (float)r.d[0], d1 = (float)r.d[1], d2 = (float)r.d[2];
  const unsigned n_samples = k_hi >= k ? (unsigned)(k_hi - k + 1) : 0u;
  const double c = (p.gyro_rho * p.dm) * ds;
  double Ta = 0.0;
  unsigned hits = 0, n_skip = 0, n_reeval = 0, n_miss = 0;
  bool wait = false;
  for (;;) {
    bool go = k <= k_hi;
    if constexpr (!TRY) {
      go = go && !wait;
      if (!__ballot(go)) {
        if (!__ballot(wait)) break;
        if (wait) {
          if (gyro_exact<DEF>(p, r.o, r.d, p.s_table[k])) Ta += c;
          ++n_reeval;
          ++k;
          wait = false;
        }
        continue;
      }
    } else {
      if (!__ballot(go)) break;
    }
    if (go) {
      const double s = fma((double)k, ds, p.smin);
      const GyroEval o =
          gyro_eval<DEF>(p, g, (float)fma(r.d[0], s, r.o[0]), (float)fma(r.d[1], s, r.o[1]),
                           (float)fma(r.d[2], s, r.o[2]), d0, d1, d2);
      if (o.amb) {
        if constexpr (TRY) {
          if (!gyro_list(p, *ts, (uint32_t)k)) {
            ts->aborted = true;
            k = k_hi;
          }
          ++k;
        } else {
          wait = true;
        }
      } else {
        int m = 0;
        if (o.ahead >= 1.0f) m = min(o.ahead < 65536.0f ? (int)o.ahead : 65536, k_hi - k);
        if constexpr (AUDIT) {
          for (int q = 0; q <= m; ++q)
            if (gyro_exact<DEF>(p, r.o, r.d, p.s_table[k + q]) != o.in) ++n_miss;
        }
        if (o.in) hits += (unsigned)(m + 1);
        n_skip += (unsigned)m;
        k += m + 1;
      }
    }
  }
  const double T = gyro_add(p.flat_field, c, hits);
  if constexpr (TRY) {
    ts->samples = n_samples;
    ts->skipped = n_skip;
  } else {
    rc.samples += n_samples;
    rc.reeval += n_reeval;
    rc.miss += n_miss;
    rc.skipped += n_skip;
  }
  return T + Ta;
}

// A wave's runs and fine sums in LDS.
struct GyroRuns {
  uint16_t len[kGyroRuns][64];  // DS terms of a run; top bit: no DS/10 term before them
  double fine[16];              // the sum of n DS/10 terms, in order
};

// Optical depth of pixel (i, j) of view v, hierarchical integrator; every
// lane of the wave calls it together.  The march is on the fine grid: coarse
// sample n, at R[n], is fine index 10 (n + 1), and fine sample m of step n
// (main.go:180-186: R[n-1] + DS/10, then DS/10 further while left of R[n];
// p.fine_n[n] of them) is 10 n + m + 1.  TRY: guard-band samples keep their FP32 densities
// and are listed as march_T_hier<TRY> does, with the FP32 membership in bit
// 31; otherwise the lanes wait for each other, and AUDIT compares, as in the
// simple march.  H > 1: only every H-th lane has a ray, and the H lanes from
// it on evaluate its next H coarse (or the step's next H fine) samples at
// once: such rays run along the level, with many guard-band samples in a row.
template <int DEF, bool TRY, bool AUDIT, int H = 1>
__device__ __forceinline__ double gyro_T_hier(const MarchParams& p, int v, int i, int j,
                                              bool valid, RayCounts& rc, TryState* ts,
                                              GyroRuns& R) {
  const double DS = p.ds, dsf = p.ds_fine;
  const int lane = threadIdx.x & 63;
  const double rr = p.gyro_rho * p.dm, c_fine = rr * dsf, c_DS = rr * DS;
  {
    // lane q's sum of q terms
    const double f = gyro_add(0.0, c_fine, (unsigned)(lane & 15));
    if (lane < 16) R.fine[lane] = f;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const GyroScene g = gyro_scene<DEF>(p, p.skip_inv * 10.0f);  // skip_inv is per DS
  Ray r;
  r.o[0] = r.o[1] = r.o[2] = 0.0;
  r.d[0] = r.d[1] = r.d[2] = 0.0;
  int n = 0, n_hi = -1;
  if (valid) {
    r = make_ray(p, p.views[p.view_offset + v], i, j);
    double t_in, t_out;
    if (clip_ray(p, r, t_in, t_out)) {
      n_hi = p.K - 1;
      if (p.clip) {
        const double a = floor((t_in - p.smin) / DS) - 3.0;
        const double b = ceil((t_out - p.smin) / DS) + 3.0;
        n = a > 0.0 ? (a < (double)p.K ? (int)a : p.K) : 0;
        n_hi = b < (double)(p.K - 1) ? (b > -1.0 ? (int)b : -1) : p.K - 1;
      }
    }
  }
  const float d0 = (float)r.d[0], d1 = (float)r.d[1], d2 = (float)r.d[2];
  const unsigned n_samples = n_hi >= n ? (unsigned)(n_hi - n + 1) : 0u;
  double T = p.flat_field, Tf = 0.0;
  unsigned n_skip = 0, n_fine = 0, n_reeval = 0, n_miss = 0;
  unsigned run = 0, runs = 0;  // DS terms of the open run; runs kept
  bool prev = false;           // the last coarse sample's density is not 0
  int left = 0;                // fine samples of step n settled from its left end
  // the step in its fine walk: fine sample m next, those from m_hi on have
  // the right end's density (cur), nf samples, the right end's reach
  bool fine = false, cur = false;
  int m = 0, m_hi = 0, nf = 0, inside = 0;
  float reach = 0.0f;
  bool wait = false;
  // H > 1: bit q says whether sample known_at + q, fine ones of step n or
  // (not known_fine) coarse ones, is inside
  unsigned known = 0;
  int known_at = -H;
  bool known_fine = false;
  // adds the kept runs to T
  auto drain = [&]() {
    for (unsigned q = 0; q < runs; ++q) {
      const unsigned l = R.len[q][lane];
      if (!(l & 0x8000u)) T += c_fine;
      T = gyro_add(T, c_DS, l & 0x7fffu);
    }
    runs = 0;
  };
  auto close = [&](unsigned l) {
    if (runs == (unsigned)kGyroRuns) drain();
    R.len[runs][lane] = (uint16_t)l;
    ++runs;
  };
  // the open run: bit 15 as in GyroRuns::len
  auto extend = [&](unsigned l) {
    while ((run & 0x7fffu) + l > 0x7fffu) {
      l -= 0x7fffu - (run & 0x7fffu);
      close(run | 0x7fffu);
      run = 0x8000u;
    }
    run += l;
  };
  // fine sample q of step nn, or its right end (q < 0)
  auto at = [&](int nn, int q) {
    if (q < 0) return p.s_table[nn];
    double s = (nn == 0 ? p.smin : p.s_table[nn - 1]) + dsf;
    for (int t = 0; t < q; ++t) s += dsf;
    return s;
  };
  auto audit = [&](int q, int end, bool in) {
    for (; q < end; ++q)
      if (gyro_exact<DEF>(p, r.o, r.d, at(n, q)) != in) ++n_miss;
  };
  for (;;) {
    bool go = n <= n_hi;
    bool exact = false, ein = false;
    if constexpr (!TRY) {
      if (!__ballot(go && !wait)) {
        if (!__ballot(wait)) break;
        if constexpr (H > 1) {
          const int own = lane & ~(H - 1), h = lane & (H - 1);
          double o[3], d[3];
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            o[c] = __shfl(r.o[c], own, 64);
            d[c] = __shfl(r.d[c], own, 64);
          }
          const int f = __shfl(fine ? 1 : 0, own, 64), nn = __shfl(n, own, 64);
          const int q = __shfl(fine ? m : n, own, 64) + h;
          const int end = __shfl(fine ? nf : n_hi + 1, own, 64);
          bool bit = false;
          if (__shfl(wait ? 1 : 0, own, 64) && q < end)
            bit = gyro_exact<DEF>(p, o, d, at(f ? nn : q, f ? q : -1));
          const unsigned long long mask = __ballot(bit);
          if (wait) {
            known = (unsigned)(mask >> own) & ((1u << H) - 1u);
            known_at = q;
            known_fine = fine;
            ein = known & 1u;
            ++n_reeval;
          }
        } else if (wait) {
          ein = gyro_exact<DEF>(p, r.o, r.d, at(n, fine ? m : -1));
          ++n_reeval;
        }
        exact = wait;
        go = wait;
        wait = false;
      } else {
        go = go && !wait;
      }
    } else {
      if (!__ballot(go)) break;
    }
    if (!go) continue;
    GyroEval o;
    if (!TRY && exact) {
      o.in = ein;
      o.amb = true;
    } else {
      const int q = fine ? 10 * n + m + 1 : 10 * n + 10;
      const double s = fma((double)q, dsf, p.smin);
      o = gyro_eval<DEF>(p, g, (float)fma(r.d[0], s, r.o[0]), (float)fma(r.d[1], s, r.o[1]),
                          (float)fma(r.d[2], s, r.o[2]), d0, d1, d2);
      if (o.amb) {
        if constexpr (TRY) {
          if (!gyro_list(p, *ts, ((uint32_t)n << 4) | (o.in ? 0x80000000u : 0u) |
                                     (fine ? (uint32_t)m : 15u))) {
            ts->aborted = true;
            n = n_hi + 1;
            continue;
          }
        } else {
          const int q = (fine ? m : n) - known_at;
          if (H > 1 && fine == known_fine && q >= 0 && q < H) {
            o.in = (known >> q) & 1u;
            ++n_reeval;
          } else {
            wait = true;
            continue;
          }
        }
      }
    }
    if (o.amb) o.ahead = o.behind = 0.0f;
    bool done;  // coarse sample n is complete, with density cur
    if (!fine) {
      if (AUDIT && !o.amb) audit(-1, 0, o.in);
      cur = o.in;
      reach = o.ahead;
      done = true;
      if (cur != prev) {
        nf = (int)p.fine_n[n];
        // from m_hi on within reach behind R[n] (sample 9 - t is t DS/10 from it)
        m_hi = nf;
        if (o.behind > 1e-4f) m_hi = min(nf, max(0, (int)ceilf(9.0f - o.behind)));
        m = min(left, m_hi);
        inside = prev ? m : 0;
        if constexpr (AUDIT) {
          audit(0, m, prev);
          audit(m_hi, nf, cur);
        }
        n_skip += (unsigned)(m + nf - m_hi);
        n_fine += (unsigned)nf;
        fine = true;
        done = m >= m_hi;
      }
    } else {
      const int t = 1 + (o.ahead >= 1.0f ? min((int)fminf(o.ahead, 64.0f), m_hi - m - 1) : 0);
      if constexpr (AUDIT) audit(o.amb ? m + 1 : m, m + t, o.in);
      if (o.in) inside += t;
      n_skip += (unsigned)(t - 1);
      m += t;
      done = m >= m_hi;
    }
    if (done) {
      if (fine) {
        // the step's density change: its fine sum, and the start or end of a run
        if (cur) inside += nf - m_hi;
        Tf += R.fine[inside & 15];
        if (prev) close(run);
        run = 0;
        fine = false;
        if (H > 1 && known_fine) known_at = -H;
      } else if (cur) {
        extend(1u);
      }
      int t = 0;
      float f = reach * 0.1f;
      if (f >= 1.0f) t = min(f < 65536.0f ? (int)f : 65536, n_hi - n);
      if constexpr (AUDIT) {
        for (int q = 1; q <= t; ++q)
          if (gyro_exact<DEF>(p, r.o, r.d, p.s_table[n + q]) != cur) ++n_miss;
      }
      if (cur && t > 0) extend((unsigned)t);
      n_skip += (unsigned)t;
      left = (int)fminf(fmaxf(fmaf(-10.0f, (float)t, reach * (1.0f - 1e-6f)), 0.0f), 15.0f);
      prev = cur;
      n += t + 1;
    }
  }
  if (prev) close(run);
  drain();
  if constexpr (TRY) {
    ts->samples = n_samples;
    ts->fine = n_fine;
    ts->skipped = n_skip;
  } else {
    rc.samples += n_samples;
    rc.reeval += n_reeval;
    rc.miss += n_miss;
    rc.fine += n_fine;
    rc.skipped += n_skip;
  }
  return T + Tf;
}

}  // namespace xrp
