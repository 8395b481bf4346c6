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

#include <cstddef>

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
// Error bound of a gyroid's FP32 g whose arguments are FP64 up to their
// reduction to [-0.5, 0.5] revolutions: six factors, each off by pi 2^-24
// from its argument and kHwSinCosErr from the unit, and the products'
// roundings: 6 (1.9e-7 + 1.3e-7) + 5 2^-24 < 2.3e-6.
constexpr float kLineGyroid = 3.0e-6f;
// Longest segment (16-bit relative indices).
constexpr int kLineSegment = 60000;

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
  unsigned runs = 1, fine = 0;  // runs of equal density, fine samples

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
      ++runs;
    }
    b = to;
  }
};

// ---------------------------------------------------------------------------
// Runs of a line in a convex primitive, as parameters along the line (units
// of s from the origin of w): the primitive holds every point of (ia, ib)
// and none outside [oa, ob].  F = float for every child; F = double, on the
// FP64 parameters, where an index lies between the two.
// ---------------------------------------------------------------------------
template <typename F>
struct LineSpan {
  F oa, ob, ia, ib;
};
template <typename F>
struct LineReal;
template <>
struct LineReal<float> {
  static constexpr float U = 1.2e-7f;  // 2^-23 and a little: two roundings
  static constexpr float big = 1e30f, tiny = 1e-12f;
  static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
  static __device__ __forceinline__ float root(float x) { return __builtin_amdgcn_sqrtf(x); }
};
template <>
struct LineReal<double> {
  static constexpr double U = 4.5e-16;
  static constexpr double big = 1e30, tiny = 1e-14;
  static __device__ __forceinline__ double rcp(double x) { return 1.0 / x; }
  static __device__ __forceinline__ double root(double x) { return sqrt(x); }
};
__device__ __forceinline__ float line_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double line_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float line_min(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double line_min(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ float line_max(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double line_max(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ float line_abs(float a) { return fabsf(a); }
__device__ __forceinline__ double line_abs(double a) { return fabs(a); }
template <typename F>
__device__ __forceinline__ F line_dot(F a0, F a1, F a2, F b0, F b1, F b2) {
  return line_fma(a0, b0, line_fma(a1, b1, a2 * b2));
}

template <typename F>
__device__ __forceinline__ F line_rcp(F x) {  // finite, sign kept
  const F r = LineReal<F>::rcp(line_max(line_abs(x), LineReal<F>::tiny));
  return x < F(0) ? -r : r;
}

// Slab lo <= c + g s <= hi (ig = 1/g): each end is off by at most e |1/g|, e
// bounding the errors of c and of g s in c's units.
template <typename F>
__device__ __forceinline__ void line_slab(LineSpan<F>& q, F c, F lo, F hi, F ig, F e) {
  const F t1 = (lo - c) * ig, t2 = (hi - c) * ig;
  const F d = e * line_abs(ig);
  const F a = line_min(t1, t2), b = line_max(t1, t2);
  q.oa = line_max(q.oa, a - d);
  q.ob = line_min(q.ob, b + d);
  q.ia = line_max(q.ia, a + d);
  q.ib = line_min(q.ib, b - d);
}

// |e0 + e1 s| < r.  w bounds |e0|, |e1 s| at every s where the primitive can
// hold the point, and the lengths e0 and e1 were projected from.  There the
// computed e0 + e1 s is within e of the exact vector, so the runs of radius
// r + e and r - e enclose the exact one from outside and inside; E covers
// both squares, d the roundings of the roots themselves.
template <typename F>
__device__ __forceinline__ void line_round(LineSpan<F>& q, const F (&e0)[3], const F (&e1)[3],
                                           F r, F r2, F w, F bl, F eps) {
  using R = LineReal<F>;
  const F a = line_max(line_dot(e1[0], e1[1], e1[2], e1[0], e1[1], e1[2]),
                       F(0.01) * R::U * R::U * bl * bl);
  const F ia = R::rcp(a), ie = R::root(ia);
  const F s0 = -line_dot(e0[0], e0[1], e0[2], e1[0], e1[1], e1[2]) * ia;
  const F m0 = line_fma(e1[0], s0, e0[0]), m1 = line_fma(e1[1], s0, e0[1]),
          m2 = line_fma(e1[2], s0, e0[2]);
  const F h2 = r2 - line_dot(m0, m1, m2, m0, m1, m2);
  const F e = line_fma(F(7) * R::U, w, eps);
  const F E = line_fma(F(2.5) * r + F(2) * e, e, F(4) * R::U * r2);
  const F ho = R::root(line_max(h2 + E, F(0)) * ia);
  const F hi = R::root(line_max(h2 - E, F(0)) * ia);
  const F d = F(4) * R::U * line_fma(w, ie, ho);
  const bool out = h2 + E < F(0), none = !(h2 - E > F(0));
  q.oa = line_max(q.oa, out ? R::big : s0 - ho - d);
  q.ob = line_min(q.ob, out ? -R::big : s0 + ho + d);
  q.ia = line_max(q.ia, none ? R::big : s0 - hi + d);
  q.ib = line_min(q.ib, none ? -R::big : s0 + hi - d);
}

// Node records: through the scalar cache (a cell's children, read again and
// again), or held by the wave, one dword per lane, and read lane by lane (a
// collection's, each read once: the next record's vector load is in flight
// while one is used, where a scalar load's latency was paid per child).
struct LineNodeRef {
  const DevNode& n;
  __device__ __forceinline__ int kind() const { return n.kind; }
  __device__ __forceinline__ float f(int q) const { return n.f[q]; }
  __device__ __forceinline__ float g(int q) const { return n.g[q]; }
  __device__ __forceinline__ double d(int q) const { return n.d[q]; }
};
struct LineNodeRec {
  uint32_t rec;
  __device__ __forceinline__ uint32_t word(size_t byte) const {
    return (uint32_t)__builtin_amdgcn_readlane((int)rec, (int)(byte / 4));
  }
  __device__ __forceinline__ int kind() const { return (int)word(offsetof(DevNode, kind)); }
  __device__ __forceinline__ float f(int q) const {
    return __uint_as_float(word(offsetof(DevNode, f) + 4 * q));
  }
  __device__ __forceinline__ float g(int q) const {
    return __uint_as_float(word(offsetof(DevNode, g) + 4 * q));
  }
  __device__ __forceinline__ double d(int q) const {
    const uint32_t lo = word(offsetof(DevNode, d) + 8 * q),
                   hi = word(offsetof(DevNode, d) + 8 * q + 4);
    return __hiloint2double((int)hi, (int)lo);
  }
};
__device__ __forceinline__ LineNodeRec line_load(const DevNode* __restrict__ N, int c) {
  static_assert(sizeof(DevNode) == 256, "one dword per lane");
  return {((const uint32_t*)(N + c))[threadIdx.x & 63]};
}

// w: the line's origin relative to the node's reference point (f[0..2]), b
// its direction per unit of s, ib its reciprocals, bl its length.  f[13..15]
// hold sizes the error bounds use (flatten in scene.cpp).
template <typename F, class D, class S>
__device__ __forceinline__ F line_pick(D&& d, S&& f) {
  if constexpr (sizeof(F) == 8)
    return d();
  else
    return f();
}
template <typename F, class Node>
__device__ __forceinline__ LineSpan<F> line_span(const Node& n, F w0, F w1, F w2, F b0, F b1,
                                                 F b2, F ib0, F ib1, F ib2, F bl, F eps) {
  using R = LineReal<F>;
  constexpr bool f64 = sizeof(F) == 8;
  LineSpan<F> q = {-R::big, R::big, -R::big, R::big};
  switch (n.kind()) {
    case K_SPHERE: {
      const F e0[3] = {w0, w1, w2}, e1[3] = {b0, b1, b2};
      const F w = R::root(line_dot(w0, w1, w2, w0, w1, w2));
      const F r = line_pick<F>([&] { return n.d(3); }, [&] { return n.f(14); }), r2 = f64 ? r * r : F(n.f(3));
      line_round(q, e0, e1, r, r2, w + r, bl, eps);
      break;
    }
    case K_BOX: {
      const F h0 = line_pick<F>([&] { return n.d(3); }, [&] { return n.f(3); }), h1 = line_pick<F>([&] { return n.d(4); }, [&] { return n.f(4); }),
              h2 = line_pick<F>([&] { return n.d(5); }, [&] { return n.f(5); });
      line_slab(q, w0, -h0, h0, ib0, line_fma(F(4) * R::U, line_abs(w0) + h0, eps));
      line_slab(q, w1, -h1, h1, ib1, line_fma(F(4) * R::U, line_abs(w1) + h1, eps));
      line_slab(q, w2, -h2, h2, ib2, line_fma(F(4) * R::U, line_abs(w2) + h2, eps));
      break;
    }
    case K_PPED: {
      const F w = line_abs(w0) + line_abs(w1) + line_abs(w2) + F(n.f(14));
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const F m0 = line_pick<F>([&] { return n.d(3 + k); }, [&] { return n.f(3 + k); }), m1 = line_pick<F>([&] { return n.d(6 + k); }, [&] { return n.f(6 + k); }),
                m2 = line_pick<F>([&] { return n.d(9 + k); }, [&] { return n.f(9 + k); });
        const F c = line_dot(m0, m1, m2, w0, w1, w2);
        const F g = line_dot(m0, m1, m2, b0, b1, b2);
        // |row of M^-1| <= f[13]
        line_slab(q, c, F(0), F(1), line_rcp(g),
                  line_fma(F(n.f(13)), line_fma(F(5) * R::U, w, eps), F(4) * R::U));
      }
      break;
    }
    default: {  // K_CYL
      const F v0 = line_pick<F>([&] { return n.d(3); }, [&] { return n.f(3); }), v1 = line_pick<F>([&] { return n.d(4); }, [&] { return n.f(4); }),
              v2 = line_pick<F>([&] { return n.d(5); }, [&] { return n.f(5); }), vv = line_pick<F>([&] { return n.d(6); }, [&] { return n.f(6); });
      const F ivv = f64 ? F(1) / vv : F(n.f(7));
      const F r = line_pick<F>([&] { return n.d(7); }, [&] { return n.f(14); }), r2 = f64 ? r * r : F(n.f(8));
      const F t0 = line_dot(w0, w1, w2, v0, v1, v2), t1 = line_dot(b0, b1, b2, v0, v1, v2);
      const F c0 = t0 * ivv, c1 = t1 * ivv;
      const F e0[3] = {line_fma(-c0, v0, w0), line_fma(-c0, v1, w1), line_fma(-c0, v2, w2)};
      const F e1[3] = {line_fma(-c1, v0, b0), line_fma(-c1, v1, b1), line_fma(-c1, v2, b2)};
      const F w = R::root(line_dot(w0, w1, w2, w0, w1, w2)) + F(n.f(13));
      line_round(q, e0, e1, r, r2, w + r, bl, eps);
      line_slab(q, t0, F(0), vv, line_rcp(t1), F(n.f(13)) * line_fma(F(5) * R::U, w, eps));
      break;
    }
  }
  return q;
}

// The full FP64 evaluator, for the rays that ties stop.  The node records
// come through the constant address space: read through plain pointers in a
// called function they were vector loads, one memory latency per field (a
// 36-strut cell: 0.33 ms per call).
typedef const DevNode __attribute__((address_space(4))) * LineNodes;
typedef const DevDeform __attribute__((address_space(4))) * LineDefs;
__device__ __forceinline__ unsigned long long line_uniform(const void* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v),
                 hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}
// One primitive's FP64 density at an object-space (cell-local) point.
// gyroid64's operations (objects.go:1014-1032): inside the sheet.  The three
// sines and cosines take turns in one copy of their code: it runs cold, and
// fetching it costs more than running it.
__device__ __forceinline__ bool line_gyroid64(const double (&k)[14], double X, double Y,
                                              double Z) {
  double q[3] = {(X - k[0]) / k[3], (Y - k[1]) / k[3], (Z - k[2]) / k[3]};
  double s[3] = {0.0, 0.0, 0.0}, c[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
  for (int a = 0; a < 3; ++a) {
    double sa, ca;
    sincos(q[0], &sa, &ca);
    q[0] = q[1], q[1] = q[2];
    s[0] = s[1], s[1] = s[2], s[2] = sa;
    c[0] = c[1], c[1] = c[2], c[2] = ca;
  }
  const double g = s[0] * c[1] + s[1] * c[2] + s[2] * c[0];
  return fabs(g) < k[4];
}
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
  return line_gyroid64(k.d, X, Y, Z) ? k.d[5] : 0.0;
}
// deform64's operations.
__device__ __forceinline__ void line_deform64(LineDefs D, int nd, double& x, double& y,
                                              double& z) {
  for (int k = 0; k < nd; ++k) {
    DevDeform f;
    f.kind = D[k].kind;
    f.axis = D[k].axis;
    f.src = D[k].src;
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
// Density of the whole tree (one of line_plan's forms) at a world point.
__device__ __forceinline__ double line_density64(const DevNode* nodes, const DevDeform* defs,
                                              int n_defs, double x, double y, double z) {
  const LineNodes N = (LineNodes)line_uniform(nodes);
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
  const int end = N[c].next;
  double sum = 0.0;
  bool hit = false;
  for (c = N[c].first; c < end; c = N[c].next) {
    const double rho = line_leaf64(N, c, x, y, z);
    if (!hit) {
      hit = greedy && rho > 0.0;
      sum = hit ? rho : sum + rho;
    }
  }
  if (!hit) sum = sum < 0.0 ? 0.0 : (sum > 1.0 ? 1.0 : sum);
  return in ? sum : 0.0;
}
// sin(2 pi t) and cos(2 pi t) in FP64 (within 1e-15): t reduced exactly to
// an eighth of a revolution, Taylor series there (terms to y^17 and y^18,
// |y| <= pi / 4: the next are below 1e-18), quadrant restored.
__device__ __forceinline__ void line_sincos64(double t, double& s, double& c) {
  const double h = rint(4.0 * t);
  const double y = fma(-0.25, h, t) * 6.283185307179586476925286766559;
  const double z = y * y;
  // 1 / (n (n-1)) steps of the two series, highest first
  double ps = 1.0 / 272.0, pc = 1.0 / 306.0;
  double a = 1.0 - z * ps, b = 1.0 - z * pc;
  constexpr double is[8] = {1.0 / 210, 1.0 / 156, 1.0 / 110, 1.0 / 72,
                            1.0 / 42,  1.0 / 20,  1.0 / 6,   0.0};
  constexpr double ic[8] = {1.0 / 240, 1.0 / 182, 1.0 / 132, 1.0 / 90,
                            1.0 / 56,  1.0 / 30,  1.0 / 12,  1.0 / 2};
#pragma unroll
  for (int q = 0; q < 7; ++q) a = fma(-z * is[q], a, 1.0);
#pragma unroll
  for (int q = 0; q < 8; ++q) b = fma(-z * ic[q], b, 1.0);
  a *= y;
  const int k = (int)(h - 4.0 * floor(0.25 * h));
  const double u = k & 1 ? b : a, v = k & 1 ? a : b;
  s = k & 2 ? -u : u;
  c = (k + 1) & 2 ? -v : v;
}

// FP64 density of the whole tree at parameter s of the ray o + d s.
__device__ __forceinline__ double line_density(const MarchParams& p, const double (&o)[3],
                                               const double (&d)[3], double s) {
  return line_density64(p.nodes, p.defs, p.n_defs, o[0] + d[0] * s, o[1] + d[1] * s,
                        o[2] + d[2] * s);
}

__device__ __forceinline__ void line_fence();

// State of one ray of the interval march beside its sum.
struct LineState {
  unsigned reeval = 0;
  bool stopped = false;  // an index only the full FP64 evaluator decides
};

// Indices of a span about index xc within [la, lb) (iu: indices per unit of
// s): [oa, ob) those it may hold, [lo, he) those it holds.
template <typename F>
__device__ __forceinline__ void line_indices(const LineSpan<F>& q, int xc, int la, int lb, F iu,
                                             int& oa, int& ob, int& lo, int& he) {
  const F fa = (F)(la - xc), fb = (F)(lb - xc);
  // first index at or past the start, one past the last index before the end
  oa = xc + (int)ceil(line_min(line_max(q.oa * iu, fa), fb));
  ob = xc + (int)line_min(line_max(floor(q.ob * iu) + F(1), fa), fb);
  lo = xc + (int)ceil(line_min(line_max(q.ia * iu, fa), fb));
  he = xc + (int)line_min(line_max(floor(q.ib * iu) + F(1), fa), fb);
  if (he < lo) he = lo;
}

// Child run [lo, he) of indices within [la, lb), from its FP32 span about
// index xc; w64() gives the line's FP64 origin relative to the node.  Indices
// between the outer and the inner FP32 span are decided by the FP64 roots;
// one between those (a tie) stops the ray.
template <class W64>
__device__ __forceinline__ void line_run(const MarchParams& p, const LineRay& L, int node, int xc,
                                         int la, int lb, double unit, float iu,
                                         const LineSpan<float>& q, W64&& w64, LineState& st,
                                         int& lo, int& he) {
  int oa, ob;
  line_indices(q, xc, la, lb, iu, oa, ob, lo, he);
  const bool amb = ob > oa && (oa != lo || ob != he);
  if (__builtin_expect(__ballot(amb) != 0ull, 0)) {
    if (__builtin_expect(amb, 0)) {
      double w[3];
      w64(w);
      const LineSpan<double> e =
          line_span(LineNodeRef{p.nodes[node]}, w[0], w[1], w[2], L.B[0], L.B[1], L.B[2], line_rcp(L.B[0]),
                    line_rcp(L.B[1]), line_rcp(L.B[2]), (double)L.bl, p.line_seam);
      line_indices(e, xc, la, lb, 1.0 / unit, oa, ob, lo, he);
      ++st.reeval;
      st.stopped = st.stopped || (ob > oa && (oa != lo || ob != he));
    }
  }
}

// Density at index x (relative to the segment) over the wave's n slots (a
// multiple of kLineUnroll), and the next index at which it changes.  The
// slots of a group are read together: one LDS latency for all.
constexpr int kLineUnroll = 4;
__device__ __forceinline__ double line_scan(const LineSlots& S, int n, unsigned x, bool greedy,
                                            bool clamp, unsigned& next) {
  const uint32_t* sp = S.span + (threadIdx.x & 63);
  double sum = 0.0;
  bool hit = false;
  next = 0xffffffffu;
  for (int t = 0; t < n; t += kLineUnroll) {
    uint32_t u[kLineUnroll];
    double r[kLineUnroll];
#pragma unroll
    for (int q = 0; q < kLineUnroll; ++q) {
      u[q] = sp[64 * (t + q)];
      r[q] = S.rho[t + q];
    }
    if (!greedy) {
#pragma unroll
      for (int q = 0; q < kLineUnroll; ++q) {
        const unsigned lo = u[q] >> 16, he = u[q] & 0xffffu;
        next = min(next, x < lo ? lo : (x < he ? he : 0xffffffffu));
        sum += x >= lo && x < he ? r[q] : 0.0;
      }
    } else {
#pragma unroll
      for (int q = 0; q < kLineUnroll; ++q) {
        const unsigned lo = u[q] >> 16, he = u[q] & 0xffffu;
        next = min(next, x < lo ? lo : (x < he ? he : 0xffffffffu));
        if (x >= lo && x < he && !hit) {
          hit = r[q] > 0.0;
          sum = hit ? r[q] : sum + r[q];
        }
      }
    }
  }
  if (clamp && !hit) sum = sum < 0.0 ? 0.0 : (sum > 1.0 ? 1.0 : sum);
  return sum;
}

// Fills slots n .. with empty runs up to a whole group; returns their number.
__device__ __forceinline__ int line_pad(const LineSlots& S, int n) {
  const int lane = threadIdx.x & 63;
  const int m = (n + kLineUnroll - 1) & ~(kLineUnroll - 1);
  for (int t = n; t < m; ++t) {
    S.span[64 * t + lane] = 0u;
    if (lane == 0) S.rho[t] = 0.0;
  }
  return m;
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

// One lane's ray (`own`) by the full FP64 evaluator, from index x0 on: up to
// 64 indices (hierarchical: coarse indices, then the fine walks of the steps
// that toggle) evaluated one per lane of the wave, the owner adding the runs.
// Returns the index reached.
template <int INTEG>
__device__ __forceinline__ int line_window(const MarchParams& p, const double (&o)[3],
                                           const double (&d)[3], int own, int x0, int end,
                                           unsigned& reeval, LineSum<INTEG>& sum) {
  const int lane = threadIdx.x & 63;
  int evals = 0;
  if (INTEG == INT_SIMPLE) {
    end = min(end, x0 + 64);
    double e = 0.0;
    if (lane < end - x0) e = line_density(p, o, d, line_s<INTEG>(p, x0 + lane));
    line_push_lanes<INTEG>(p, own, 0, end - x0, x0, e, sum);
    evals = end - x0;
  } else {
    // coarse indices xc + 10 lane
    const int xc = ((x0 + 9) / 10) * 10;
    const int cc = min(64, end > xc ? (end - xc + 9) / 10 : 0);
    if (cc == 64) end = min(end, xc + 631);
    if (lane == own) sum.flush(p, sum.cur);
    double e = 0.0;
    if (lane < cc) e = line_density(p, o, d, line_s<INTEG>(p, xc + 10 * lane));
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
          if (need) f = line_density(p, o, d, s);
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
      if (lane < end - xl) g = line_density(p, o, d, line_s<INTEG>(p, xl + lane));
      line_push_lanes<INTEG>(p, own, 0, end - xl, xl, g, sum);
      evals += end - xl;
    }
  }
  if (lane == own) reeval += (unsigned)evals;
  return end;
}

// Walk the runs of [x, xe) (absolute indices, slots relative to base).
// AUDIT: every index of a run is also evaluated in FP64 and compared.
template <int INTEG, bool AUDIT>
__device__ __forceinline__ void line_events(const MarchParams& p, const LineRay& L,
                                            const LineSlots& S, int n, int base, int x, int xe,
                                            bool greedy, bool clamp, LineSum<INTEG>& sum,
                                            RayCounts& rc) {
  while (__ballot(x < xe)) {
    if (x < xe) {
      unsigned nx;
      const double rho = line_scan(S, n, (unsigned)(x - base), greedy, clamp, nx);
      const int to = nx == 0xffffffffu ? xe : min(base + (int)nx, xe);
      if constexpr (AUDIT) {
        for (int k = x; k < to; ++k)
          if (line_density(p, L.r.o, L.r.d, line_s<INTEG>(p, k)) != rho) ++rc.miss;
      }
      sum.push(p, rho, to);
      x = to;
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

// The children of the root collection that the wave's rays can meet, as
// Cull (eval_block.hpp).  All rays leave one eye, so they lie in a cone about
// their mean direction; lane l tests child l of each 64 against it (bounding
// spheres, which the host inflates past rounding; 1e-5 of the distance
// covers the FP32 test's own).  One pass for 64 children where a ray per
// lane tested them one by one (batch of 10 scenes: 3.27 -> 2.75 ms with the
// record loads above).
__device__ __forceinline__ Cull line_cull(const MarchParams& p, const LineRay& L) {
  __shared__ int16_t list[kMaxCull];
  Cull cl;
  const DevNode* __restrict__ N = p.nodes;
  const int first = N[0].first, count = N[0].next - first;
  if (N[0].kind != K_COLL || count < 8) return cl;
  const int lane = threadIdx.x & 63;
  const unsigned long long some = __ballot(L.x0 < L.x1);
  cl.idx = list;
  cl.n = 0;
  if (!some) return cl;
  const int src = (int)__builtin_ctzll(some);
  const float e0 = (float)__shfl(L.A[0], src, 64), e1 = (float)__shfl(L.A[1], src, 64),
              e2 = (float)__shfl(L.A[2], src, 64);
  const float il = L.x0 < L.x1 ? __builtin_amdgcn_rcpf(L.bl) : 0.0f;
  const float n0 = L.b[0] * il, n1 = L.b[1] * il, n2 = L.b[2] * il;
  float c0 = n0, c1 = n1, c2 = n2;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    c0 += __shfl_xor(c0, off, 64);
    c1 += __shfl_xor(c1, off, 64);
    c2 += __shfl_xor(c2, off, 64);
  }
  const float ic = __builtin_amdgcn_rsqf(fmaf(c0, c0, fmaf(c1, c1, c2 * c2)));
  c0 *= ic;
  c1 *= ic;
  c2 *= ic;
  // sine of the cone's half angle: the largest |n x c|
  const float x0 = fmaf(n1, c2, -n2 * c1), x1 = fmaf(n2, c0, -n0 * c2),
              x2 = fmaf(n0, c1, -n1 * c0);
  float sa = L.x0 < L.x1 ? fmaf(x0, x0, fmaf(x1, x1, x2 * x2)) : 0.0f;
  bool back = L.x0 < L.x1 && fmaf(n0, c0, fmaf(n1, c1, n2 * c2)) < 0.5f;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) sa = fmaxf(sa, __shfl_xor(sa, off, 64));
  if (__ballot(back)) {  // a pencil this wide keeps every child
    cl.idx = nullptr;
    cl.n = -1;
    return cl;
  }
  const float s = __builtin_amdgcn_sqrtf(sa) * (1.0f + 1e-5f) + 2e-6f;
  const float co = __builtin_amdgcn_sqrtf(fmaxf(1.0f - s * s, 0.0f));
  int n = 0;
  for (int base = 0; base < count; base += 64) {
    bool keep = base + lane < count;
    if (keep) {
      const DevNode& ch = N[first + base + lane];
      if (ch.kind != K_GYROID) {
        const float w0 = ch.bsph[0] - e0, w1 = ch.bsph[1] - e1, w2 = ch.bsph[2] - e2;
        const float a = fabsf(fmaf(w0, c0, fmaf(w1, c1, w2 * c2)));
        const float y0 = fmaf(w1, c2, -w2 * c1), y1 = fmaf(w2, c0, -w0 * c2),
                    y2 = fmaf(w0, c1, -w1 * c0);
        const float q = __builtin_amdgcn_sqrtf(fmaf(y0, y0, fmaf(y1, y1, y2 * y2)));
        // distance to the cone's surface (both nappes)
        keep = q * co - a * s <= ch.bsph[3] + 1e-5f * (a + q);
      }
    }
    const unsigned long long m = __ballot(keep);
    const int at = n + (int)__popcll(m & __lanemask_lt());
    if (keep && at < kMaxCull) list[at] = (int16_t)(first + base + lane);
    n += (int)__popcll(m);
  }
  if (n > kMaxCull) {
    cl.idx = nullptr;
    n = -1;
  }
  cl.n = n;
  line_fence();
  return cl;
}

// Adds a finished ray's counts: every index but the first of each run of
// equal density is settled.
template <int INTEG>
__device__ __forceinline__ void line_counts(RayCounts& rc, const RayCounts& own, unsigned reeval,
                                            const LineSum<INTEG>& sum) {
  rc.samples += own.samples;
  rc.reeval += reeval;
  rc.fine += sum.fine;
  rc.skipped += own.samples > sum.runs ? own.samples - sum.runs : 0u;
}

// Root collection (or a single primitive), p.line == LINE_COLL.  The ray's
// index range is walked in segments: a segment computes every listed child's
// runs, and one whose runs do not fit the cap's slots is halved.
template <int INTEG, bool AUDIT>
__device__ __forceinline__ void line_coll(const MarchParams& p, const LineRay& L,
                                          const LineSlots& S, int cap, const Cull& cl,
                                          LineState& st, LineSum<INTEG>& sum, RayCounts& rc) {
  const double unit = INTEG == INT_SIMPLE ? p.ds : p.ds_fine;
  const float iu = (float)(1.0 / unit);
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
    const int n_kids = !coll ? 1 : n_list >= 0 ? n_list : N[0].next - N[0].first;
    auto child = [&](int t) {
      return !coll         ? 0
             : n_list >= 0 ? __builtin_amdgcn_readfirstlane((int)cl.idx[t])
                           : N[0].first + t;
    };
    int c = n_kids > 0 ? child(0) : 0;
    LineNodeRec ahead = line_load(N, c);
    for (int t = 0; t < n_kids && !over; ++t) {
      const LineNodeRec k = ahead;
      const int node = c;
      if (t + 1 < n_kids) {
        c = child(t + 1);
        ahead = line_load(N, c);
      }
      const int kind = k.kind();
      if (kind == K_GYROID) {
        const double rho = k.d(5);
        if (rho == 0.0) continue;
        int x = la, start = 0, got = 0;
        bool cur = false;
        // arguments of the sines in revolutions, FP64 up to their reduction:
        // g is then off by at most kLineGyroid beside the positions' share
        // (with FP32 positions the band was 3e-5, and near each crossing
        // some lane of the wave waited on the FP64 sines)
        const double th64 = k.d(4), rv = 0.15915494309189535 / k.d(3);
        const float inv = k.f(3), iso = k.g(4), M = k.g(6), inv_M = k.g(1), e1 = k.g(7),
                    lip = k.g(5);
        double a0[3], a1[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          a0[q] = (Q[q] - k.d(q)) * rv;
          a1[q] = L.B[q] * (unit * rv);
        }
        const float band = kLineGyroid + 10.0f * p.line_eps * inv, th = k.f(4);
        while (__ballot(x < lb)) {
          if (x < lb) {
            float sn[3], cs[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
              const double t = a0[q] + a1[q] * (double)(x - xc);
              const float r = (float)(t - rint(t));
              sn[q] = __builtin_amdgcn_sinf(r);
              cs[q] = __builtin_amdgcn_cosf(r);
            }
            const float gg = fmaf(sn[0], cs[1], fmaf(sn[1], cs[2], sn[2] * cs[0]));
            const float gap = fabsf(gg) - th;
            float dist = (fabsf(gap) - band) * iso;
            if (p.vel) {
              // the second-order reach of gyroid_blk
              const float g1 = fmaf(fmaf(cs[0], cs[1], -sn[2] * sn[0]), L.b[0],
                                    fmaf(fmaf(cs[1], cs[2], -sn[0] * sn[1]), L.b[1],
                                         fmaf(cs[2], cs[0], -sn[1] * sn[2]) * L.b[2])) * inv;
              dist = fmaxf(dist, gyroid_reach(gg, g1, th, band, M, inv_M, e1) * lip);
            }
            const bool amb = fabsf(gap) < band;
            bool in = gap < 0.0f;
            int m = 0;
            if (__builtin_expect(amb, 0)) {
              // FP64: the membership, and the second-order reach without a
              // band (a ray along the level stays in the FP32 band for many
              // indices); within 1e-12 of the level it is a tie
              double s6[3], c6[3];
#pragma unroll
              for (int q = 0; q < 3; ++q)
                line_sincos64(a0[q] + a1[q] * (double)(x - xc), s6[q], c6[q]);
              const double g = s6[0] * c6[1] + s6[1] * c6[2] + s6[2] * c6[0];
              const double g1 = ((c6[0] * c6[1] - s6[2] * s6[0]) * L.B[0] +
                                 (c6[1] * c6[2] - s6[0] * s6[1]) * L.B[1] +
                                 (c6[2] * c6[0] - s6[1] * s6[2]) * L.B[2]) * (double)inv;
              const double away = fabs(fabs(g) - th64) - (1e-12 + 10.0 * p.line_seam * rv);
              in = fabs(g) < th64;
              ++st.reeval;
              if (!(away > 0.0)) {
                st.stopped = true;
              } else if (M > 0.0f) {
                // both sides of the level inside, one outside; 1e-6 and the
                // shrink cover g1 and the FP32 root
                const float s1 = (float)g1;
                const float toward = in ? fabsf(s1) : (g < 0.0 ? s1 : -s1);
                const float bq = -toward - 1e-6f * (1.0f + fabsf(s1));
                const float f = quad_reach((float)away, bq, M, inv_M) * (1.0f - 1e-4f) * iu;
                m = f >= 1.0f ? min(f < 65536.0f ? (int)f : 65536, lb - x - 1) : 0;
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
        const double rho = k.d(kind == K_SPHERE ? 4 : kind == K_BOX ? 6 : kind == K_PPED ? 12 : 8);
        if (rho == 0.0) continue;
        const double r0 = k.d(0), r1 = k.d(1), r2 = k.d(2);
        const LineSpan<float> q =
            line_span(k, (float)(Q[0] - r0), (float)(Q[1] - r1), (float)(Q[2] - r2), L.b[0],
                      L.b[1], L.b[2], L.ib[0], L.ib[1], L.ib[2], L.bl, p.line_eps);
        int lo, he;
        line_run(
            p, L, node, xc, la, lb, unit, iu, q,
            [&](double (&w)[3]) {
              w[0] = Q[0] - r0;
              w[1] = Q[1] - r1;
              w[2] = Q[2] - r2;
            },
            st, lo, he);
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
    n = line_pad(S, n);
    line_fence();
    if (single) {
      if (la < lb && !st.stopped) {
        if (coll && !hit) acc = acc < 0.0 ? 0.0 : (acc > 1.0 ? 1.0 : acc);
        if (AUDIT && line_density(p, L.r.o, L.r.d, line_s<INTEG>(p, s0)) != acc) ++rc.miss;
        sum.push(p, acc, s1);
      }
    } else {
      line_events<INTEG, AUDIT>(p, L, S, n, s0, la, st.stopped ? la : lb, greedy, coll, sum, rc);
    }
    line_fence();
    s0 = s1;
    len = min(2 * len, kLineSegment);
  }
}

// Offset of coordinate q into its cell along axis c, in [0, side): the
// reference's wrap (objects.go:568-582).  f[12..14] are FP32, so the floor
// is settled with the FP64 offset itself.
__device__ __forceinline__ double line_local(const DevNode& R, int c, double q) {
  const double lo = R.d[6 + c], dx = R.d[9 + c] - lo;
  double l = (q - lo) - dx * floor((q - lo) * (double)R.f[12 + c]);
  if (l < 0.0) l += dx;
  if (l >= dx) l -= dx;
  return l;
}

// Root tessellation of a collection of convex primitives, p.line ==
// LINE_TESS.  Each lane walks its ray cell by cell: the cell of the index
// reached is found in FP64 as the reference wraps (objects.go:568-582), the
// indices that stay clear of its faces form one segment; one within the FP64
// tolerance of a face stops the ray.
template <int INTEG, bool AUDIT>
__device__ __forceinline__ void line_tess(const MarchParams& p, const LineRay& L,
                                          const LineSlots& S, LineState& st,
                                          LineSum<INTEG>& sum, RayCounts& rc) {
  const double unit = INTEG == INT_SIMPLE ? p.ds : p.ds_fine;
  const float iu = (float)(1.0 / unit);
  const int lane = threadIdx.x & 63;
  const DevNode* __restrict__ N = p.nodes;
  const DevNode& R = N[0];
  const DevNode& C = N[R.first];
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
        // parallel to the faces: a tie unless the line is clear of them
        const double m = L.A[c] + g * (p.smin + 0.5 * (double)(L.x0 + L.x1) * unit);
        if (m < R.d[2 * c] - 1e-7 || m > R.d[2 * c + 1] + 1e-7)
          hit = false;
        else if (m < R.d[2 * c] + 1e-7 || m > R.d[2 * c + 1] - 1e-7)
          st.stopped = true;
      }
    }
    if (hit && ta <= tb + 1e-9) {
      const double ua = (ta - p.smin) / unit, ub = (tb - p.smin) / unit;
      const double tol = 1e-8 + p.line_seam / ((double)L.bl * unit);
      double ca = ceil(ua - tol), cb = floor(ub + tol);
      const double x0 = (double)L.x0, x1 = (double)L.x1;
      xa = (int)fmin(fmax(ca, x0), x1);
      xb = (int)fmin(fmax(cb + 1.0, x0), x1);
      if (xb < xa) xb = xa;
      // an end that close to an index is a tie
      if (xa < xb && ((double)xa < ua + tol || (double)(xb - 1) > ub - tol)) st.stopped = true;
    } else {
      xa = xb = L.x0;
    }
  }
  if (st.stopped) xa = xb;
  int x = xa;
  if (L.x0 < xa) sum.push(p, 0.0, xa);
  while (__ballot(x < xb)) {
    int m1 = 0;  // indices of this segment
    float w0 = 0.0f, w1 = 0.0f, w2 = 0.0f;
    if (x < xb) {
      const double s = p.smin + (double)x * unit;
      float face = 1e30f;
      float w[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double q = L.A[c] + L.B[c] * s;
        const double lo = R.d[6 + c], dx = R.d[9 + c] - lo, l = line_local(R, c, q);
        if (l < p.line_seam || l > dx - p.line_seam) st.stopped = true;
        w[c] = (float)(l + lo);
        const float fdx = (float)dx, wl = (float)l;
        const float e = fmaf(4.0f * LineReal<float>::U, fdx, p.line_eps);
        const float room = (L.b[c] > 0.0f ? fdx - wl : wl) - e;
        face = fminf(face, room * fabsf(L.ib[c]));
      }
      w0 = w[0];
      w1 = w[1];
      w2 = w[2];
      // indices past x clear of the nearest face (the 1e-5 covers the
      // products' roundings)
      const float fm = fminf(fmaxf(face * iu * (1.0f - 1e-5f), 0.0f), 59990.0f);
      m1 = min((int)fm + 1, xb - x);
      if (st.stopped) {
        m1 = 0;
        x = xb;
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
      const LineSpan<float> q =
          line_span(LineNodeRef{k}, w0 - k.f[0], w1 - k.f[1], w2 - k.f[2], L.b[0], L.b[1], L.b[2], L.ib[0],
                    L.ib[1], L.ib[2], L.bl, p.line_eps);
      int lo, he;
      line_run(
          p, L, c, x, x, x + m1, unit, iu, q,
          [&](double (&w)[3]) {
            const double s = p.smin + (double)x * unit;
#pragma unroll
            for (int a = 0; a < 3; ++a) w[a] = line_local(R, a, L.A[a] + L.B[a] * s) +
                                               (R.d[6 + a] - k.d[a]);
          },
          st, lo, he);
      if (__ballot(he > lo)) {
        S.span[64 * n + lane] = he > lo ? ((uint32_t)(lo - x) << 16) | (uint32_t)(he - x) : 0u;
        if (lane == 0) S.rho[n] = rho;
        ++n;
      }
    }
    if (st.stopped) {
      m1 = 0;
      x = xb;
    }
    n = line_pad(S, n);
    line_fence();
    line_events<INTEG, AUDIT>(p, L, S, n, x, x, x + m1, C.greedy != 0, true, sum, rc);
    line_fence();
    x += m1;
  }
  if (L.x0 < L.x1 && xb < L.x1) sum.push(p, 0.0, L.x1);
}

// Optical depth of pixel (i, j) of view v; every lane of the wave calls it
// together.  A ray that meets a tie is stopped: its result is not used, and
// line_T_exact gives it.  KIND: LINE_COLL, LINE_TESS, or LINE_NONE for
// p.line's (wave-uniform).
template <int INTEG, bool AUDIT, int KIND>
__device__ __forceinline__ double line_T(const MarchParams& p, int v, int i, int j, bool valid,
                                         const LineSlots& S, int cap, RayCounts& rc,
                                         bool& stopped) {
  LineRay L;
  RayCounts own;
  line_setup<INTEG>(p, v, i, j, valid, L, own);
  LineSum<INTEG> sum;
  sum.start(p.flat_field, L.x0);
  LineState st;
  if (KIND == LINE_TESS || (KIND == LINE_NONE && p.line == LINE_TESS)) {
    line_tess<INTEG, AUDIT>(p, L, S, st, sum, rc);
  } else {
    const Cull cl = line_cull(p, L);
    line_coll<INTEG, AUDIT>(p, L, S, cap, cl, st, sum, rc);
  }
  sum.flush(p, sum.cur);
  stopped = st.stopped;
  if (!st.stopped) line_counts(rc, own, st.reeval, sum);
  return sum.T;
}

// Optical depth of one lane's pixel (`own`; wave-uniform) by the full FP64
// evaluator, the indices spread over the wave.  Every lane calls it with the
// owner's pixel; T is meaningful on the owner.
template <int INTEG>
__device__ __forceinline__ double line_T_exact(const MarchParams& p, int v, int i, int j, int own,
                                               RayCounts& rc) {
  LineRay L;
  RayCounts mine;
  line_setup<INTEG>(p, v, i, j, true, L, mine);
  LineSum<INTEG> sum;
  sum.start(p.flat_field, L.x0);
  unsigned reeval = 0;
  const int x1 = __builtin_amdgcn_readfirstlane(L.x1);
  for (int x = __builtin_amdgcn_readfirstlane(L.x0); x < x1;)
    x = line_window<INTEG>(p, L.r.o, L.r.d, own, x, x1, reeval, sum);
  sum.flush(p, sum.cur);
  if ((int)(threadIdx.x & 63) == own) line_counts(rc, mine, reeval, sum);
  return sum.T;
}

}  // namespace xrp
