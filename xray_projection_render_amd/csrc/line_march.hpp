// line_march.hpp - the interval march: scenes whose rays stay straight in
// object space (affine, linear and rigid deformations) and whose primitives
// meet a line in intervals.
//
// The marches of march_ray.hpp find where the density along a ray changes by
// evaluating the tree at samples and stepping by safe radii.  Along a
// straight line those places can be computed: a sphere, box, parallelepiped
// or cylinder is convex, so it holds one run of consecutive samples, whose
// ends are the roots of a linear or quadratic equation.  This march computes
// every child's run of sample indices once per ray (per cell of a
// tessellation), then walks from one change of the density to the next and
// adds each stretch of equal terms in one step.  A gyroid child contributes
// the runs its own safe reach (eval_block.hpp) finds.
//
// Exactness.  The roots are FP32, each with a bound on its error (below); a
// sample whose position is further than the bound from every root has the
// reference's membership.  One that is not is decided by the primitive's
// FP64 test at the reference's own sample position (main.go:148-150), so the
// densities summed are the reference's.  Terms of one run are added as
// (count * term): one rounding where the reference has `count`.
//
// Sample index x.  Simple integrator: x = k, position s_table[k].
// Hierarchical (main.go:159-199): steps of DS/10; coarse sample R[n] is
// x = 10 (n + 1) and the j-th sample of its step's fine walk x = 10 n + j.
#pragma once
#include <hip/hip_runtime.h>

#include "march_ray.hpp"

namespace xrp {

// Per-wave LDS of the interval march: one slot per run of a child, [slot]
// [lane] the run's first index and one past its last, 16 bits each, relative
// to the segment's start (both 0: none), and the child's density per slot.
struct LineSlots {
  uint32_t* span;  // [cap][64]
  double* rho;     // [cap]
};
constexpr size_t line_lds_bytes(int cap) { return (size_t)cap * (64 * 4 + 8); }
// Longest segment (16-bit relative indices).
constexpr int kLineSegment = 60000;
// Ambiguous samples of one child tested one by one before the whole stretch
// is left to the full FP64 evaluator.
constexpr int kLineTests = 8;

__device__ __forceinline__ LineSlots line_slots(unsigned char* lds, int cap) {
  LineSlots s;
  s.rho = (double*)lds;
  s.span = (uint32_t*)(lds + (size_t)cap * 8);
  return s;
}

// One ray of the interval march: world ray, object-space line q(s) = A + B s
// and its FP32 copy, the lane's index range [x0, x1).
struct LineRay {
  Ray r;
  double A[3], B[3];
  float b[3], ib[3];  // B and its componentwise reciprocals
  float bb, bl;       // |B|^2, |B|
  int x0, x1;
};

// Reference position parameter of index x.
template <int INTEG>
__device__ __forceinline__ double line_s(const MarchParams& p, int x) {
  if constexpr (INTEG == INT_SIMPLE) {
    return p.s_table[x];
  } else {
    const int n = x / 10, j = x - 10 * n;
    double s = n == 0 ? p.smin : p.s_table[n - 1];
    for (int q = 0; q < j; ++q) s += p.ds_fine;
    return s;
  }
}

// Running integral: runs of equal density in index order.  Adjacent runs of
// one density merge, so the sums do not depend on how the march cut the ray
// into segments.
template <int INTEG>
struct LineSum {
  double T, cur = 0.0;
  int a, b;  // pending run [a, b) of density cur
  // hierarchical: fine sum and toggle state of the step in progress
  double S = 0.0;
  bool prev_zero = true;
  unsigned runs = 0, fine = 0;

  __device__ __forceinline__ void start(double flat, int x) {
    T = flat;
    a = b = x;
  }
  // rho10: density of a tenth fine sample just before a coarse sample that
  // starts the run (differs from rho only on exact ties)
  __device__ __forceinline__ void flush(const MarchParams& p, double rho10) {
    if (b <= a) return;
    const double rr = cur * p.dm;
    if constexpr (INTEG == INT_SIMPLE) {
      T += (double)(b - a) * (rr * p.ds);
    } else {
      const double f = rr * p.ds_fine;
      const int xc = ((a + 9) / 10) * 10;
      if (xc >= b) {
        S += (double)(b - a) * f;
      } else {
        S += (double)(xc - a) * f;
        const bool z = rr == 0;
        if (z != prev_zero) {
          // main.go:180-188: left += DS/10 while left < right, from R[n-1]
          const int n = xc / 10 - 1;
          double left = n == 0 ? p.smin : p.s_table[n - 1];
#pragma unroll
          for (int q = 0; q < 10; ++q) left += p.ds_fine;
          const bool ten = left < p.s_table[n];
          if (ten) S += (rho10 * p.dm) * p.ds_fine;
          fine += ten ? 10u : 9u;
          T += S;
          T += f;
        } else {
          T += rr * p.ds;
        }
        prev_zero = z;
        const int m = (b - 1 - xc) / 10;  // further coarse samples of the run
        T += (double)m * (rr * p.ds);
        S = (double)(b - 1 - (xc + 10 * m)) * f;
      }
    }
    a = b;
  }
  __device__ __forceinline__ void push(const MarchParams& p, double rho, int to) {
    if (rho != cur) {
      flush(p, cur);
      cur = rho;
    }
    b = to;
  }
};

// ---------------------------------------------------------------------------
// Runs of a line in a convex primitive, as parameters along the line (units
// of s from the origin of w): the primitive holds every point of (ia, ib)
// and none outside [oa, ob].
// ---------------------------------------------------------------------------
struct LineSpan {
  float oa, ob, ia, ib;
};
constexpr float kLineU = 1.2e-7f;  // 2^-23 and a little: two FP32 roundings

__device__ __forceinline__ float line_rcp(float x) {  // finite, sign kept
  const float m = fmaxf(fabsf(x), 1e-12f);
  return copysignf(__builtin_amdgcn_rcpf(m), x);
}

// Slab lo <= c + g s <= hi (ig = 1/g): each end is off by at most e |1/g|, e
// bounding the errors of c and of g s in c's units.
__device__ __forceinline__ void line_slab(LineSpan& q, float c, float lo, float hi, float ig,
                                          float e) {
  const float t1 = (lo - c) * ig, t2 = (hi - c) * ig;
  const float d = e * fabsf(ig);
  const float a = fminf(t1, t2), b = fmaxf(t1, t2);
  q.oa = fmaxf(q.oa, a - d);
  q.ob = fminf(q.ob, b + d);
  q.ia = fmaxf(q.ia, a + d);
  q.ib = fminf(q.ib, b - d);
}

// |e0 + e1 s| < r.  w bounds |e0|, |e1 s| at every s where the primitive can
// hold the point, and the lengths e0 and e1 were projected from.  There the
// computed e0 + e1 s is within e of the exact vector, so the runs of radius
// r + e and r - e enclose the exact one from outside and inside; E covers
// both squares, d the roundings of the roots themselves.
__device__ __forceinline__ void line_round(LineSpan& q, const float (&e0)[3],
                                           const float (&e1)[3], float r, float r2, float w,
                                           float bl, float eps) {
  const float a = fmaxf(fmaf(e1[0], e1[0], fmaf(e1[1], e1[1], e1[2] * e1[2])),
                        1e-14f * bl * bl);
  const float ia = __builtin_amdgcn_rcpf(a), ie = __builtin_amdgcn_rsqf(a);
  const float s0 = -fmaf(e0[0], e1[0], fmaf(e0[1], e1[1], e0[2] * e1[2])) * ia;
  const float m0 = fmaf(e1[0], s0, e0[0]), m1 = fmaf(e1[1], s0, e0[1]),
              m2 = fmaf(e1[2], s0, e0[2]);
  const float h2 = r2 - fmaf(m0, m0, fmaf(m1, m1, m2 * m2));
  const float e = fmaf(7.0f * kLineU, w, eps);
  const float E = fmaf(2.5f * r + 2.0f * e, e, 4.0f * kLineU * r2);
  const float ho = __builtin_amdgcn_sqrtf(fmaxf(h2 + E, 0.0f) * ia);
  const float hi = __builtin_amdgcn_sqrtf(fmaxf(h2 - E, 0.0f) * ia);
  const float d = 4.0f * kLineU * fmaf(w, ie, ho);
  const bool out = h2 + E < 0.0f, none = !(h2 - E > 0.0f);
  q.oa = fmaxf(q.oa, out ? 1e30f : s0 - ho - d);
  q.ob = fminf(q.ob, out ? -1e30f : s0 + ho + d);
  q.ia = fmaxf(q.ia, none ? 1e30f : s0 - hi + d);
  q.ib = fminf(q.ib, none ? -1e30f : s0 + hi - d);
}

// w: the line's origin relative to the node's reference point (f[0..2]), b
// its direction per unit of s.  f[13..15] hold sizes the error bounds use
// (flatten in scene.cpp).
__device__ __forceinline__ LineSpan line_span(const DevNode& n, const LineRay& L, float w0,
                                              float w1, float w2, float eps) {
  LineSpan q = {-1e30f, 1e30f, -1e30f, 1e30f};
  const float b0 = L.b[0], b1 = L.b[1], b2 = L.b[2];
  switch (n.kind) {
    case K_SPHERE: {
      const float e0[3] = {w0, w1, w2}, e1[3] = {b0, b1, b2};
      const float w = __builtin_amdgcn_sqrtf(fmaf(w0, w0, fmaf(w1, w1, w2 * w2)));
      line_round(q, e0, e1, n.f[14], n.f[3], w + n.f[14], L.bl, eps);
      break;
    }
    case K_BOX: {
      line_slab(q, w0, -n.f[3], n.f[3], L.ib[0], fmaf(4.0f * kLineU, fabsf(w0) + n.f[3], eps));
      line_slab(q, w1, -n.f[4], n.f[4], L.ib[1], fmaf(4.0f * kLineU, fabsf(w1) + n.f[4], eps));
      line_slab(q, w2, -n.f[5], n.f[5], L.ib[2], fmaf(4.0f * kLineU, fabsf(w2) + n.f[5], eps));
      break;
    }
    case K_PPED: {
      const float w = fabsf(w0) + fabsf(w1) + fabsf(w2) + n.f[14];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float m0 = n.f[3 + k], m1 = n.f[6 + k], m2 = n.f[9 + k];
        const float c = fmaf(m0, w0, fmaf(m1, w1, m2 * w2));
        const float g = fmaf(m0, b0, fmaf(m1, b1, m2 * b2));
        // |row of M^-1| <= f[13]
        line_slab(q, c, 0.0f, 1.0f, line_rcp(g),
                  fmaf(n.f[13], fmaf(5.0f * kLineU, w, eps), 4.0f * kLineU));
      }
      break;
    }
    default: {  // K_CYL
      const float v0 = n.f[3], v1 = n.f[4], v2 = n.f[5], vv = n.f[6], ivv = n.f[7];
      const float t0 = fmaf(w0, v0, fmaf(w1, v1, w2 * v2));
      const float t1 = fmaf(b0, v0, fmaf(b1, v1, b2 * v2));
      const float c0 = t0 * ivv, c1 = t1 * ivv;
      const float e0[3] = {fmaf(-c0, v0, w0), fmaf(-c0, v1, w1), fmaf(-c0, v2, w2)};
      const float e1[3] = {fmaf(-c1, v0, b0), fmaf(-c1, v1, b1), fmaf(-c1, v2, b2)};
      const float w = __builtin_amdgcn_sqrtf(fmaf(w0, w0, fmaf(w1, w1, w2 * w2))) + n.f[13];
      line_round(q, e0, e1, n.f[14], n.f[8], w + n.f[14], L.bl, eps);
      line_slab(q, t0, 0.0f, vv, line_rcp(t1), n.f[13] * fmaf(5.0f * kLineU, w, eps));
      break;
    }
  }
  return q;
}

// The FP64 evaluators are called (rarely) out of line: inlined, they set the
// register budget of the whole march (200-240 VGPRs, 2 waves per SIMD).
// Their pointers and node index are the same on every lane.  In a function
// the compiler cannot tell, and reads the node records with vector loads,
// one memory latency per field (a 36-strut cell: 0.33 ms per call, most of
// the kernel where a column of rays lies in a cell face); through the
// constant address space they come as scalar loads.
typedef const DevNode __attribute__((address_space(4))) * LineNodes;
typedef const DevDeform __attribute__((address_space(4))) * LineDefs;
__device__ __forceinline__ unsigned long long line_uniform(const void* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v),
                 hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}
// One primitive's FP64 density at an object-space (cell-local) point.
__device__ __forceinline__ double line_leaf64(LineNodes N, int c, double X, double Y, double Z) {
  DevNode k;
  k.kind = N[c].kind;
#pragma unroll
  for (int q = 0; q < 14; ++q) k.d[q] = N[c].d[q];
  switch (k.kind) {
    case K_SPHERE: return sphere64(k, X, Y, Z);
    case K_BOX: return box64(k, X, Y, Z);
    case K_PPED: return pped64(k, X, Y, Z);
    case K_CYL: return cyl64(k, X, Y, Z);
  }
  // gyroid64's operations (objects.go:1014-1032)
  X = (X - k.d[0]) / k.d[3];
  Y = (Y - k.d[1]) / k.d[3];
  Z = (Z - k.d[2]) / k.d[3];
  const double g = sin(X) * cos(Y) + sin(Y) * cos(Z) + sin(Z) * cos(X);
  return fabs(g) < k.d[4] ? k.d[5] : 0.0;
}
// The deformations line_plan admits (deform64's operations).
__device__ __forceinline__ void line_deform64(LineDefs D, int nd, double& x, double& y,
                                              double& z) {
  for (int k = 0; k < nd; ++k) {
    DevDeform f;
    f.kind = D[k].kind;
#pragma unroll
    for (int q = 0; q < 9; ++q) f.d[q] = D[k].d[q];
    deform64(&f, 1, x, y, z);
  }
}
// objects.go:568-582; false outside the tessellation's bounds or the cell.
__device__ __forceinline__ bool line_wrap64(LineNodes N, double& X, double& Y, double& Z) {
  double b[12];
#pragma unroll
  for (int q = 0; q < 12; ++q) b[q] = N[0].d[q];
  if (X < b[0] || X > b[1] || Y < b[2] || Y > b[3] || Z < b[4] || Z > b[5]) return false;
  const double dx = b[9] - b[6], dy = b[10] - b[7], dz = b[11] - b[8];
  X = X - dx * floor((X - b[6]) / dx);
  Y = Y - dy * floor((Y - b[7]) / dy);
  Z = Z - dz * floor((Z - b[8]) / dz);
  return !(X < b[6] || X > b[9] || Y < b[7] || Y > b[10] || Z < b[8] || Z > b[11]);
}
// Density of the whole tree (one of line_plan's forms) at a world point; the
// root collection's children limited to idx[0 .. n) when n >= 0 (Cull).
__device__ __noinline__ double line_density64(const DevNode* nodes, const DevDeform* defs,
                                              int n_defs, double x, double y, double z,
                                              const int16_t* idx, int n) {
  const LineNodes N = (LineNodes)line_uniform(nodes);
  n = __builtin_amdgcn_readfirstlane(n);
  line_deform64((LineDefs)line_uniform(defs), __builtin_amdgcn_readfirstlane(n_defs), x, y, z);
  const int kind = N[0].kind;
  int c = 0;
  bool in = true;
  if (kind == K_TESS) {
    in = line_wrap64(N, x, y, z);
    c = N[0].first;
  } else if (kind != K_COLL) {
    return line_leaf64(N, 0, x, y, z);
  }
  const bool greedy = N[c].greedy != 0;
  const int end = n < 0 ? N[c].next : 0x7fffffff;
  double sum = 0.0;
  bool hit = false;
  int t = 0;
  c = n < 0 ? N[c].first : 0;
  while (n < 0 ? c < end : t < n) {
    if (n >= 0) c = __builtin_amdgcn_readfirstlane((int)idx[t++]);
    const double rho = line_leaf64(N, c, x, y, z);
    if (!hit) {
      hit = greedy && rho > 0.0;
      sum = hit ? rho : sum + rho;
    }
    if (n < 0) c = N[c].next;
  }
  if (!hit) sum = sum < 0.0 ? 0.0 : (sum > 1.0 ? 1.0 : sum);
  return in ? sum : 0.0;
}
// Membership of a world point in node `node`, in the unit cell's wrap when
// tess is set.
__device__ __noinline__ bool line_member64(const DevNode* nodes, const DevDeform* defs,
                                           int n_defs, int node, bool tess, double X, double Y,
                                           double Z) {
  const LineNodes N = (LineNodes)line_uniform(nodes);
  line_deform64((LineDefs)line_uniform(defs), __builtin_amdgcn_readfirstlane(n_defs), X, Y, Z);
  if (tess) (void)line_wrap64(N, X, Y, Z);
  return line_leaf64(N, __builtin_amdgcn_readfirstlane(node), X, Y, Z) != 0.0;
}
// A gyroid's g at a world point (gyroid64's operations) and its derivative
// along the object-space direction b.
struct LineG {
  double g, g1;
};
__device__ __noinline__ LineG line_gyroid64(const DevNode* nodes, const DevDeform* defs,
                                            int n_defs, int node, double X, double Y, double Z,
                                            double b0, double b1, double b2) {
  line_deform64((LineDefs)line_uniform(defs), __builtin_amdgcn_readfirstlane(n_defs), X, Y, Z);
  const LineNodes N = (LineNodes)line_uniform(nodes) + __builtin_amdgcn_readfirstlane(node);
  const double sc = N->d[3];
  const double x = (X - N->d[0]) / sc, y = (Y - N->d[1]) / sc, z = (Z - N->d[2]) / sc;
  const double sx = sin(x), cx = cos(x), sy = sin(y), cy = cos(y), sz = sin(z), cz = cos(z);
  LineG r;
  r.g = sx * cy + sy * cz + sz * cx;
  r.g1 = ((cx * cy - sz * sx) * b0 + (cy * cz - sx * sy) * b1 + (cz * cx - sy * sz) * b2) / sc;
  return r;
}

// FP64 membership of index x in one primitive (of the unit cell with TESS),
// at the reference's sample position (main.go:148-150).  tie: at a coarse
// index, whether the tenth sample of the fine walk before it (a few ulps
// away, where the walk's additions end short of it) differs.
template <int INTEG, bool TESS>
__device__ __forceinline__ bool line_exact(const MarchParams& p, const LineRay& L, int node,
                                           int x, bool& tie) {
  const double s = line_s<INTEG>(p, x);
  const bool in = line_member64(p.nodes, p.defs, p.n_defs, node, TESS,
                                L.r.o[0] + L.r.d[0] * s, L.r.o[1] + L.r.d[1] * s,
                                L.r.o[2] + L.r.d[2] * s);
  tie = false;
  if (INTEG == INT_HIERARCHICAL && x % 10 == 0) {
    const double s9 = line_s<INTEG>(p, x - 1) + p.ds_fine;
    tie = s9 < s && in != line_member64(p.nodes, p.defs, p.n_defs, node, TESS,
                                        L.r.o[0] + L.r.d[0] * s9, L.r.o[1] + L.r.d[1] * s9,
                                        L.r.o[2] + L.r.d[2] * s9);
  }
  return in;
}

// FP64 density of the whole tree at parameter s of the ray o + d s.
__device__ __forceinline__ double line_density(const MarchParams& p, const double (&o)[3],
                                               const double (&d)[3], double s, const Cull& cl) {
  return line_density64(p.nodes, p.defs, p.n_defs, o[0] + d[0] * s, o[1] + d[1] * s,
                        o[2] + d[2] * s, cl.idx, cl.n);
}

// State of one ray of the interval march beside its sum.
struct LineState {
  int wa = 0x7fffffff, wb = 0;  // indices left to the full FP64 evaluator, [wa, wb)
  unsigned reeval = 0;
  bool aborted = false;  // TRY: an index needed FP64
};

// Child run [lo, he) of indices within [la, lb), from the span q about index
// xc (iu: indices per unit of s).  Indices between the outer and the inner
// span are decided in FP64.
template <int INTEG, bool TESS, bool TRY>
__device__ __forceinline__ void line_run(const MarchParams& p, const LineRay& L,
                                         const LineSpan& q, int node, int xc, int la, int lb,
                                         float iu, LineState& st, int& lo, int& he) {
  const float fa = (float)(la - xc), fb = (float)(lb - xc);
  // first index at or past the start, one past the last index before the end
  const int oa = xc + (int)ceilf(fminf(fmaxf(q.oa * iu, fa), fb));
  const int ob = xc + (int)fminf(fmaxf(floorf(q.ob * iu) + 1.0f, fa), fb);
  lo = xc + (int)ceilf(fminf(fmaxf(q.ia * iu, fa), fb));
  he = xc + (int)fminf(fmaxf(floorf(q.ib * iu) + 1.0f, fa), fb);
  if (he < lo) he = lo;
  const bool amb = ob > oa && (oa != lo || ob != he);
  if (__ballot(amb)) {
    if (amb) {
      if constexpr (TRY) {
        st.aborted = true;
      } else {
        const bool inner = he > lo;
        const int i0 = lo, i1 = he;
        int first = 0x7fffffff, last = -1, cnt = 0, tests = 0;
        bool wide = false;
        for (int x = oa; x < ob;) {
          if (inner && x == i0) {
            first = min(first, i0);
            last = i1 - 1;
            cnt += i1 - i0;
            x = i1;
            continue;
          }
          if (++tests > kLineTests) {
            wide = true;
            break;
          }
          bool tie;
          if (line_exact<INTEG, TESS>(p, L, node, x, tie)) {
            first = min(first, x);
            last = x;
            ++cnt;
          }
          ++st.reeval;
          if (tie) {
            st.wa = min(st.wa, x);
            st.wb = max(st.wb, x + 1);
          }
          ++x;
        }
        if (!wide && cnt != (cnt ? last - first + 1 : 0)) wide = true;
        lo = cnt ? first : la;
        he = cnt ? last + 1 : la;
        if (wide) {
          st.wa = min(st.wa, oa);
          st.wb = max(st.wb, ob);
        }
      }
    }
  }
}

// Density at index x (relative to the segment) over the wave's n slots, and
// the next index at which it changes.
__device__ __forceinline__ double line_scan(const LineSlots& S, int n, unsigned x, bool greedy,
                                            bool clamp, unsigned& next) {
  const uint32_t* sp = S.span + (threadIdx.x & 63);
  double sum = 0.0;
  bool hit = false;
  next = 0xffffffffu;
  if (!greedy) {
    for (int t = 0; t < n; ++t) {
      const uint32_t u = sp[64 * t];
      const unsigned lo = u >> 16, he = u & 0xffffu;
      next = min(next, x < lo ? lo : (x < he ? he : 0xffffffffu));
      const double r = S.rho[t];
      sum += x >= lo && x < he ? r : 0.0;
    }
  } else {
    for (int t = 0; t < n; ++t) {
      const uint32_t u = sp[64 * t];
      const unsigned lo = u >> 16, he = u & 0xffffu;
      next = min(next, x < lo ? lo : (x < he ? he : 0xffffffffu));
      const double r = S.rho[t];
      if (x >= lo && x < he && !hit) {
        if (r > 0.0) {
          sum = r;
          hit = true;
        } else {
          sum += r;
        }
      }
    }
  }
  if (clamp && !hit) sum = sum < 0.0 ? 0.0 : (sum > 1.0 ? 1.0 : sum);
  return sum;
}

// Runs of e over lanes 0 .. cnt of the wave, indices x0 + lane, added to the
// owner's sum.
template <int INTEG>
__device__ __forceinline__ void line_push_lanes(const MarchParams& p, int own, int first,
                                                int cnt, int x0, double e, LineSum<INTEG>& sum) {
  const int lane = (int)(threadIdx.x & 63) - first;
  const double before = __shfl_up(e, 1, 64);
  unsigned long long starts =
      __ballot(lane >= 0 && lane < cnt && (lane == 0 || e != before)) >> first;
  while (starts) {
    const int b = (int)__builtin_ctzll(starts);
    starts &= starts - 1ull;
    const int to = starts ? (int)__builtin_ctzll(starts) : cnt;
    const double v = __shfl(e, first + b, 64);
    if ((int)(threadIdx.x & 63) == own) sum.push(p, v, x0 + to);
  }
}

// The FP64 window of one lane of the wave (`own`), from its x on: up to 64
// indices (hierarchical: coarse indices, then the fine walks of the steps
// that toggle) evaluated by the whole tree, one per lane; the owner adds the
// runs.
template <int INTEG>
__device__ __forceinline__ void line_window(const MarchParams& p, const LineRay& L, int own,
                                            int& x, int xe, const Cull& cl, LineState& st,
                                            LineSum<INTEG>& sum) {
  const int lane = threadIdx.x & 63;
  const int x0 = __builtin_amdgcn_readlane(x, own);
  int end = min(__builtin_amdgcn_readlane(xe, own), __builtin_amdgcn_readlane(st.wb, own));
  double o[3], d[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    o[c] = __shfl(L.r.o[c], own, 64);
    d[c] = __shfl(L.r.d[c], own, 64);
  }
  int evals = 0;
  if (INTEG == INT_SIMPLE) {
    end = min(end, x0 + 64);
    double e = 0.0;
    if (lane < end - x0) e = line_density(p, o, d, line_s<INTEG>(p, x0 + lane), cl);
    line_push_lanes<INTEG>(p, own, 0, end - x0, x0, e, sum);
    evals = end - x0;
  } else {
    // coarse indices xc + 10 lane
    const int xc = ((x0 + 9) / 10) * 10;
    const int cc = min(64, end > xc ? (end - xc + 9) / 10 : 0);
    if (cc == 64) end = min(end, xc + 631);
    if (lane == own) sum.flush(p, sum.cur);
    double e = 0.0;
    if (lane < cc) e = line_density(p, o, d, line_s<INTEG>(p, xc + 10 * lane), cl);
    const bool z = e * p.dm == 0;
    const unsigned long long zm = __ballot(z);
    const bool pz = __builtin_amdgcn_readlane((int)sum.prev_zero, own) != 0;
    unsigned long long tog = zm ^ ((zm << 1) | (pz ? 1ull : 0ull));
    if (cc < 64) tog &= (1ull << cc) - 1ull;
    evals = cc;
    const double before = __shfl_up(e, 1, 64);
    unsigned long long starts = __ballot(lane < cc && (lane == 0 || e != before)) | tog;
    if (cc < 64) starts &= (1ull << cc) - 1ull;
    // six toggled steps at a time: lane 10 q + j holds fine sample j + 1 of
    // the q-th, j = 9 its tenth, a few ulps before the coarse index
    unsigned long long left = tog, done = 0ull;
    double f = 0.0;
    bool ten = false;
    int group = 0;
    while (starts) {
      const int k = (int)__builtin_ctzll(starts);
      if ((tog >> k) & 1ull && !((done >> k) & 1ull)) {
        int step = -1;
        for (int q = 0; q < 6 && left; ++q) {
          const int kk = (int)__builtin_ctzll(left);
          left &= left - 1ull;
          done |= 1ull << kk;
          if (lane / 10 == q) step = kk;
        }
        group = 0;
        f = 0.0;
        ten = false;
        if (step >= 0) {
          const int xk = xc + 10 * step, j = lane % 10;
          double s = line_s<INTEG>(p, j < 9 ? xk - 9 + j : xk - 1);
          bool need = j == 9 || xk - 9 + j >= x0;
          if (j == 9) {
            s += p.ds_fine;
            need = s < p.s_table[xk / 10 - 1];
            ten = need;
          }
          if (need) f = line_density(p, o, d, s, cl);
        }
        evals += 10;
      }
      starts &= starts - 1ull;
      const int to = starts ? (int)__builtin_ctzll(starts) : cc;
      const double v = __shfl(e, k, 64);
      if ((tog >> k) & 1ull) {
        // fine samples of the step, then its coarse index by itself
        const int xk = xc + 10 * k, lo = max(xk - 9, x0);
        line_push_lanes<INTEG>(p, own, 10 * group + (lo - (xk - 9)), xk - lo, lo, f, sum);
        const double f10 = __shfl(f, 10 * group + 9, 64);
        const bool has = __shfl((int)ten, 10 * group + 9, 64) != 0;
        if (lane == own) {
          sum.flush(p, sum.cur);
          sum.push(p, v, xk + 1);
          sum.flush(p, has ? f10 : v);
        }
        ++group;
      }
      if (lane == own) sum.push(p, v, xc + 10 * (to - 1) + 1);
    }
    // fine samples past the last coarse index of the window
    const int xl = cc > 0 ? xc + 10 * (cc - 1) + 1 : x0;
    if (end > xl) {
      double g = 0.0;
      if (lane < end - xl) g = line_density(p, o, d, line_s<INTEG>(p, xl + lane), cl);
      line_push_lanes<INTEG>(p, own, 0, end - xl, xl, g, sum);
      evals += end - xl;
    }
  }
  if (lane == own) {
    x = end;
    st.reeval += (unsigned)evals;
    sum.runs += (unsigned)evals;
  }
}

// Walk the runs of [x, xe) (absolute indices, slots relative to base).
template <int INTEG, bool TRY>
__device__ __forceinline__ void line_events(const MarchParams& p, const LineRay& L,
                                            const LineSlots& S, int n, int base, int x, int xe,
                                            bool greedy, bool clamp, const Cull& cl,
                                            LineState& st, LineSum<INTEG>& sum,
                                            RayCounts& rc) {
  while (__ballot(x < xe)) {
    const bool win = !TRY && x < xe && x >= st.wa && x < st.wb;
    if (x < xe && !win) {
      unsigned nx;
      const double rho = line_scan(S, n, (unsigned)(x - base), greedy, clamp, nx);
      int to = nx == 0xffffffffu ? xe : min(base + (int)nx, xe);
      if (!TRY && x < st.wa && st.wa < st.wb) to = min(to, st.wa);
      ++sum.runs;
      if constexpr (!TRY) {
        if (p.audit) {
          for (int k = x; k < to; ++k)
            if (line_density(p, L.r.o, L.r.d, line_s<INTEG>(p, k), cl) != rho) ++rc.miss;
        }
      }
      sum.push(p, rho, to);
      x = to;
    }
    if constexpr (!TRY) {
      for (unsigned long long m = __ballot(win); m; m &= m - 1ull)
        line_window<INTEG>(p, L, (int)__builtin_ctzll(m), x, xe, cl, st, sum);
    }
  }
}

// The lane's ray, object-space line and index range (empty without a pixel,
// for a NaN ray and for a ray that misses the clip box).
template <int INTEG>
__device__ __forceinline__ void line_setup(const MarchParams& p, int v, int i, int j, bool valid,
                                           LineRay& L, RayCounts& rc) {
  L.r.o[0] = L.r.o[1] = L.r.o[2] = 0.0;
  L.r.d[0] = L.r.d[1] = 0.0;
  L.r.d[2] = 1.0;
  L.x0 = L.x1 = 0;
  if (valid) {
    L.r = make_ray(p, p.views[p.view_offset + v], i, j);
    double t_in, t_out;
    if (clip_ray(p, L.r, t_in, t_out)) {
      int a, b;
      if constexpr (INTEG == INT_SIMPLE) {
        clip_range(p, t_in, t_out, a, b);
        if (a <= b) {
          L.x0 = a;
          L.x1 = b + 1;
        }
      } else {
        a = 0;
        b = p.K - 1;
        if (p.clip) {
          const double lo = floor((t_in - p.smin) / p.ds) - 3.0;
          const double hi = ceil((t_out - p.smin) / p.ds) + 3.0;
          a = lo > 0.0 ? (lo < (double)p.K ? (int)lo : p.K) : 0;
          b = hi < (double)(p.K - 1) ? (hi > -1.0 ? (int)hi : -1) : p.K - 1;
        }
        if (a <= b) {
          L.x0 = 10 * a + 1;
          L.x1 = 10 * (b + 1) + 1;
        }
      }
      if (a <= b) rc.samples += (unsigned long long)(b - a + 1);
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    L.A[c] = p.M[3 * c] * L.r.o[0] + p.M[3 * c + 1] * L.r.o[1] + p.M[3 * c + 2] * L.r.o[2] +
             p.t[c];
    L.B[c] = p.M[3 * c] * L.r.d[0] + p.M[3 * c + 1] * L.r.d[1] + p.M[3 * c + 2] * L.r.d[2];
    L.b[c] = (float)L.B[c];
    L.ib[c] = line_rcp(L.b[c]);
  }
  L.bb = fmaf(L.b[0], L.b[0], fmaf(L.b[1], L.b[1], L.b[2] * L.b[2]));
  L.bl = __builtin_amdgcn_sqrtf(L.bb);
}

__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ void line_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Root collection (or a single primitive), p.line == LINE_COLL.  The ray's
// index range is walked in segments: a segment computes every listed child's
// runs, and one whose runs do not fit the cap's slots is halved.
template <int INTEG, bool TRY>
__device__ __forceinline__ void line_coll(const MarchParams& p, const LineRay& L,
                                          const LineSlots& S, int cap, const Cull& cl,
                                          LineState& st, LineSum<INTEG>& sum, RayCounts& rc) {
  const double unit = INTEG == INT_SIMPLE ? p.ds : p.ds_fine;
  const float u32 = (float)unit, iu = (float)(1.0 / unit);
  const float reach = INTEG == INT_SIMPLE ? p.skip_inv : 10.0f * p.skip_inv;
  const int lane = threadIdx.x & 63;
  const bool some = L.x0 < L.x1;
  const int wx0 = __builtin_amdgcn_readfirstlane(wave_min_i(some ? L.x0 : 0x7fffffff));
  const int wx1 = __builtin_amdgcn_readfirstlane(wave_max_i(some ? L.x1 : 0));
  const DevNode* __restrict__ N = p.nodes;
  const bool coll = N[0].kind == K_COLL;
  const bool greedy = coll && N[0].greedy;
  const int n_list = cl.n >= 0 ? cl.n : -1;
  int len = kLineSegment;
  for (int s0 = wx0; s0 < wx1;) {
    const int s1 = min(s0 + len, wx1);
    const int la = max(L.x0, s0), lb = max(min(L.x1, s1), la);
    const int xc = s0 + ((s1 - s0) >> 1);
    const double sc = p.smin + (double)xc * unit;
    double Q[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) Q[c] = L.A[c] + L.B[c] * sc;
    int n = 0;
    bool over = false;
    // a segment of one index needs no slots: its density is summed here
    const bool single = s1 - s0 == 1;
    double acc = 0.0;
    bool hit = false;
    auto add = [&](double rho) {
      if (hit) return;
      hit = greedy && rho > 0.0;
      acc = hit ? rho : acc + rho;
    };
    st.wa = 0x7fffffff;
    st.wb = 0;
    int t = 0;
    int c = !coll ? 0
            : n_list < 0 ? N[0].first
                         : (n_list > 0 ? __builtin_amdgcn_readfirstlane((int)cl.idx[0]) : N[0].next);
    const int cend = coll ? N[0].next : 1;
    for (; c < cend && !over;
         c = n_list < 0 ? N[c].next
                        : (++t < n_list ? __builtin_amdgcn_readfirstlane((int)cl.idx[t]) : cend)) {
      const DevNode& k = N[c];
      if (k.kind == K_GYROID) {
        const double rho = k.d[5];
        if (rho == 0.0) continue;
        int x = la, start = 0, got = 0;
        bool cur = false;
        const float q0 = (float)Q[0], q1 = (float)Q[1], q2 = (float)Q[2];
        while (__ballot(x < lb)) {
          if (x < lb) {
            const float sj = (float)(x - xc) * u32;
            PBlock<1> P;
            P.x[0] = fmaf(L.b[0], sj, q0);
            P.y[0] = fmaf(L.b[1], sj, q1);
            P.z[0] = fmaf(L.b[2], sj, q2);
            if (p.vel) {
              P.vx = L.b[0];
              P.vy = L.b[1];
              P.vz = L.b[2];
            }
            double gv[1];
            unsigned amb = 0;
            float dist = INFINITY;
            gyroid_blk<1, true>(k, P, gv, amb, dist);
            bool in = gv[0] != 0.0;
            int m = 0;
            if (amb & 1u) {
              if constexpr (TRY) {
                st.aborted = true;
              } else {
                // FP64: the membership, and the second-order reach without a
                // band (a ray along the level stays in the FP32 band for
                // many indices)
                const double s = line_s<INTEG>(p, x);
                const LineG e = line_gyroid64(
                    p.nodes, p.defs, p.n_defs, c, L.r.o[0] + L.r.d[0] * s,
                    L.r.o[1] + L.r.d[1] * s, L.r.o[2] + L.r.d[2] * s, L.B[0], L.B[1], L.B[2]);
                const double th = k.d[4], ag = fabs(e.g);
                in = ag < th;
                ++st.reeval;
                const double gap = fabs(ag - th) - 1e-12;
                if (!(gap > 0.0)) {
                  st.wa = min(st.wa, x);
                  st.wb = max(st.wb, x + 1);
                } else if (k.g[6] > 0.0f) {
                  // both sides of the level inside, one outside; 1e-6 and
                  // the shrink cover g1 and the FP32 root
                  const float M = k.g[6], g1 = (float)e.g1, g = (float)gap;
                  const float toward = in ? fabsf(g1) : (e.g < 0.0 ? g1 : -g1);
                  const float bq = -toward - 1e-6f * (1.0f + fabsf(g1));
                  const float r1 = quad_reach(g, bq, M, k.g[1]) * (1.0f - 1e-4f);
                  const float f = r1 * iu;
                  m = f >= 1.0f ? min(f < 65536.0f ? (int)f : 65536, lb - x - 1) : 0;
                }
              }
            } else {
              const float f = dist * reach;
              m = f >= 1.0f ? min(f < 65536.0f ? (int)f : 65536, lb - x - 1) : 0;
            }
            if (in && !cur) start = x;
            if (!in && cur) {
              if (n + got < cap)
                S.span[64 * (n + got) + lane] = ((uint32_t)(start - s0) << 16) | (uint32_t)(x - s0);
              ++got;
            }
            cur = in;
            x += m + 1;
          }
        }
        if (single) {
          if (cur) add(rho);
          continue;
        }
        if (cur) {
          if (n + got < cap)
            S.span[64 * (n + got) + lane] = ((uint32_t)(start - s0) << 16) | (uint32_t)(lb - s0);
          ++got;
        }
        const int most = __builtin_amdgcn_readfirstlane(wave_max_i(got));
        if (n + most > cap) {
          over = true;
          break;
        }
        for (int q = got; q < most; ++q) S.span[64 * (n + q) + lane] = 0u;
        if (lane == 0)
          for (int q = 0; q < most; ++q) S.rho[n + q] = rho;
        n += most;
      } else {
        const double rho = k.kind == K_SPHERE ? k.d[4]
                           : k.kind == K_BOX  ? k.d[6]
                           : k.kind == K_PPED ? k.d[12]
                                              : k.d[8];
        if (rho == 0.0) continue;
        const LineSpan q = line_span(k, L, (float)(Q[0] - k.d[0]), (float)(Q[1] - k.d[1]),
                                     (float)(Q[2] - k.d[2]), p.line_eps);
        int lo, he;
        line_run<INTEG, false, TRY>(p, L, q, c, xc, la, lb, iu, st, lo, he);
        if (single) {
          if (he > lo) add(rho);
          continue;
        }
        if (__ballot(he > lo)) {
          if (n == cap) {
            over = true;
            break;
          }
          S.span[64 * n + lane] = he > lo ? ((uint32_t)(lo - s0) << 16) | (uint32_t)(he - s0) : 0u;
          if (lane == 0) S.rho[n] = rho;
          ++n;
        }
      }
    }
    if (over) {  // never on a single index
      len = (s1 - s0 + 1) >> 1;
      continue;
    }
    line_fence();
    int x = la;
    if (single && la < lb && !(TRY && st.aborted) && !(s0 >= st.wa && s0 < st.wb)) {
      if (coll && !hit) acc = acc < 0.0 ? 0.0 : (acc > 1.0 ? 1.0 : acc);
      if (!TRY && p.audit &&
          line_density(p, L.r.o, L.r.d, line_s<INTEG>(p, s0), cl) != acc)
        ++rc.miss;
      ++sum.runs;
      sum.push(p, acc, s1);
      x = lb;
    }
    line_events<INTEG, TRY>(p, L, S, n, s0, x, st.aborted && TRY ? x : lb, greedy, coll, cl, st,
                            sum, rc);
    line_fence();
    s0 = s1;
    len = min(2 * len, kLineSegment);
  }
}

// Root tessellation of a collection of convex primitives, p.line ==
// LINE_TESS.  Each lane walks its ray cell by cell: the cell of the index
// reached is found in FP64 as the reference wraps (objects.go:568-582), the
// indices that stay clear of its faces form one segment, and one within the
// error bound of a face is evaluated in FP64 by itself.
template <int INTEG, bool TRY>
__device__ __forceinline__ void line_tess(const MarchParams& p, const LineRay& L,
                                          const LineSlots& S, LineState& st,
                                          LineSum<INTEG>& sum, RayCounts& rc) {
  const double unit = INTEG == INT_SIMPLE ? p.ds : p.ds_fine;
  const float iu = (float)(1.0 / unit);
  const int lane = threadIdx.x & 63;
  const DevNode* __restrict__ N = p.nodes;
  const DevNode& R = N[0];
  const DevNode& C = N[R.first];
  const Cull all;
  // indices inside the tessellation's closed bounds: one range
  int xa = L.x0, xb = L.x1;
  if (L.x0 < L.x1) {
    double ta = -1e300, tb = 1e300;
    bool hit = true;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double g = L.B[c];
      if (fabs(g) > 1e-9) {
        const double ig = 1.0 / g;
        const double t1 = (R.d[2 * c] - L.A[c]) * ig, t2 = (R.d[2 * c + 1] - L.A[c]) * ig;
        ta = fmax(ta, fmin(t1, t2));
        tb = fmin(tb, fmax(t1, t2));
      } else {
        // parallel to the faces: every index goes to the FP64 evaluator
        // unless the line is clear of them
        const double m = L.A[c] + g * (p.smin + 0.5 * (double)(L.x0 + L.x1) * unit);
        if (m < R.d[2 * c] - 1e-7 || m > R.d[2 * c + 1] + 1e-7)
          hit = false;
        else if (m < R.d[2 * c] + 1e-7 || m > R.d[2 * c + 1] - 1e-7)
          st.wa = L.x0, st.wb = L.x1;
      }
    }
    if (hit && ta <= tb + 1e-9) {
      const double ua = (ta - p.smin) / unit, ub = (tb - p.smin) / unit;
      const double tol = 1e-6 + p.line_seam / ((double)L.bl * unit);
      double ca = ceil(ua - tol), cb = floor(ub + tol);
      const double x0 = (double)L.x0, x1 = (double)L.x1;
      xa = (int)fmin(fmax(ca, x0), x1);
      xb = (int)fmin(fmax(cb + 1.0, x0), x1);
      if (xb < xa) xb = xa;
      // an end that close to an index leaves it to the FP64 evaluator
      const bool ea = xa < xb && (double)xa < ua + tol, eb = xa < xb && (double)(xb - 1) > ub - tol;
      if (ea) {
        st.wa = min(st.wa, xa);
        st.wb = max(st.wb, xa + 1);
      }
      if (eb) {
        st.wa = min(st.wa, xb - 1);
        st.wb = max(st.wb, xb);
      }
      if (TRY && st.wa < st.wb) st.aborted = true;
    } else {
      xa = xb = L.x0;
    }
  }
  const int wa = st.wa, wb = st.wb;  // FP64 indices of the bounds' faces
  int x = xa;
  if (L.x0 < xa) {
    ++sum.runs;
    sum.push(p, 0.0, xa);
  }
  while (__ballot(x < xb)) {
    int m1 = 0;    // indices of this segment
    int seam = 0;  // of them, from x on, within the FP64 tolerance of a face
    float w0 = 0.0f, w1 = 0.0f, w2 = 0.0f;
    st.wa = wa;
    st.wb = wb;
    if (x < xb) {
      const double s = p.smin + (double)x * unit;
      float face = 1e30f;
      float w[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double q = L.A[c] + L.B[c] * s;
        const double lo = R.d[6 + c], dx = R.d[9 + c] - lo;
        const double f = (q - lo) * (double)R.f[12 + c];
        double fl = floor(f);
        // R.f is FP32: settle the floor with the FP64 offset itself
        double l = (q - lo) - dx * fl;
        if (l < 0.0) l += dx;
        if (l >= dx) l -= dx;
        if (l < p.line_seam || l > dx - p.line_seam)
          seam = max(seam, 1 + (int)fminf((float)p.line_seam * fabsf(L.ib[c]) * iu, 4096.0f));
        w[c] = (float)(l + lo);
        const float fdx = (float)dx, wl = (float)l;
        const float e = fmaf(4.0f * kLineU, fdx, p.line_eps);
        const float room = (L.b[c] > 0.0f ? fdx - wl : wl) - e;
        face = fminf(face, room * fabsf(L.ib[c]));
      }
      w0 = w[0];
      w1 = w[1];
      w2 = w[2];
      // indices past x clear of the nearest face (the 1e-5 covers the
      // products' roundings)
      const float fm = fminf(fmaxf(face * iu * (1.0f - 1e-5f), 0.0f), 59990.0f);
      m1 = min(seam ? seam : (int)fm + 1, xb - x);
      if (seam) {
        st.wa = min(st.wa, x);
        st.wb = max(st.wb, x + m1);
        if (TRY) st.aborted = true;
      }
    }
    int n = 0;
    for (int c = C.first; c < C.next; c = N[c].next) {
      const DevNode& k = N[c];
      const double rho = k.kind == K_SPHERE ? k.d[4]
                         : k.kind == K_BOX  ? k.d[6]
                         : k.kind == K_PPED ? k.d[12]
                                            : k.d[8];
      if (rho == 0.0) continue;
      const LineSpan q = line_span(k, L, w0 - k.f[0], w1 - k.f[1], w2 - k.f[2], p.line_eps);
      int lo, he;
      line_run<INTEG, true, TRY>(p, L, q, c, x, x, seam ? x : x + m1, iu, st, lo, he);
      if (__ballot(he > lo)) {
        S.span[64 * n + lane] = he > lo ? ((uint32_t)(lo - x) << 16) | (uint32_t)(he - x) : 0u;
        if (lane == 0) S.rho[n] = rho;
        ++n;
      }
    }
    if (TRY && st.aborted) x = xb, m1 = 0;
    line_fence();
    line_events<INTEG, TRY>(p, L, S, n, x, x, x + m1, C.greedy != 0, true, all, st, sum, rc);
    line_fence();
    x += m1;
  }
  if (L.x0 < L.x1 && xb < L.x1) {
    ++sum.runs;
    sum.push(p, 0.0, L.x1);
  }
}

// Optical depth of pixel (i, j) of view v; every lane of the wave calls it
// together.  TRY: no FP64 evaluator; `aborted` is set for a ray that needs
// one, whose result is not used.  KIND: LINE_COLL, LINE_TESS, or LINE_NONE
// for p.line's (wave-uniform).
template <int INTEG, bool TRY, int KIND>
__device__ __forceinline__ double line_T(const MarchParams& p, int v, int i, int j, bool valid,
                                         const LineSlots& S, int cap, RayCounts& rc,
                                         bool& aborted) {
  LineRay L;
  RayCounts own;
  line_setup<INTEG>(p, v, i, j, valid, L, own);
  LineSum<INTEG> sum;
  sum.start(p.flat_field, L.x0);
  LineState st;
  if (KIND == LINE_TESS || (KIND == LINE_NONE && p.line == LINE_TESS)) {
    line_tess<INTEG, TRY>(p, L, S, st, sum, rc);
  } else {
    const Cull cl = wave_cull<1>(p, v, i, j, valid);
    line_coll<INTEG, TRY>(p, L, S, cap, cl, st, sum, rc);
  }
  sum.flush(p, sum.cur);
  aborted = st.aborted;
  if (!(TRY && st.aborted)) {
    rc.samples += own.samples;
    rc.reeval += st.reeval;
    rc.fine += sum.fine;
    rc.skipped += own.samples > sum.runs ? own.samples - sum.runs : 0u;
  }
  return sum.T;
}

}  // namespace xrp
