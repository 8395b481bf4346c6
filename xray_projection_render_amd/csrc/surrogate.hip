// surrogate.hip - training and inference kernels of the learned density
// surrogate (hash encoding + 32-64-64-1 MLP, BF16 MFMA, FP32 accumulation).
//
// Wave layout.  One wave evaluates 16 samples at a time: lane l serves
// sample s = l % 16 and lane group g = l / 16.  The MLP layers are computed
// transposed, H^T = W^T X^T, with v_mfma_f32_16x16x16_bf16: the weights are
// the A operand (A[m][k] in lane m%16... see below) and the activations the
// B operand.  For that instruction lane l holds
//   A[m = l%16][k = 4(l/16) + i],  B[k = 4(l/16) + i][n = l%16],
//   D[m = 4(l/16) + i][n = l%16],  i = 0..3,
// so a layer's output tile (rows = units 4g+i, column = sample s) is, after
// bias, ReLU and BF16 rounding, exactly the B operand of the next layer's
// K block.  The 32 encoding features therefore split over the lane groups
// as features 4g..4g+3 and 16+4g..16+4g+3, i.e. hash levels 2g, 2g+1,
// 8+2g and 9+2g: every lane encodes four levels of its sample.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "eval_device.hpp"
#include "march.hpp"
#include "surrogate.hpp"

namespace xrp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}
// f2bf of four finite values (v_cvt_pk_bf16_f32, round to nearest even)
__device__ __forceinline__ bf16x4 f2bf4(float a, float b, float c, float d) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 h2 __attribute__((ext_vector_type(2)));
  typedef short s2 __attribute__((ext_vector_type(2)));
  const s2 p = __builtin_bit_cast(s2, __builtin_convertvector((f2{a, b}), h2));
  const s2 q = __builtin_bit_cast(s2, __builtin_convertvector((f2{c, d}), h2));
  return bf16x4{p[0], p[1], q[0], q[1]};
}
__device__ __forceinline__ float bf2f(unsigned h) { return __uint_as_float(h << 16); }

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

struct SurOffsets {
  size_t W1, b1, W2, b2, w3, b3;
};
__host__ __device__ inline SurOffsets sur_offsets(int log2_table) {
  const size_t t = sur_table_floats(log2_table);
  SurOffsets o;
  o.W1 = t;
  o.b1 = o.W1 + kSurIn * kSurHidden;
  o.W2 = o.b1 + kSurHidden;
  o.b2 = o.W2 + kSurHidden * kSurHidden;
  o.w3 = o.b2 + kSurHidden;
  o.b3 = o.w3 + kSurHidden;
  return o;
}

// ---------------------------------------------------------------------------
// Hash encoding of one level: corner indices and trilinear weights.
// ---------------------------------------------------------------------------
struct LevelCell {
  uint32_t idx[8];
  float w[8];
};

__device__ __forceinline__ LevelCell level_cell(int N, uint32_t tmask, bool dense, float ux,
                                                float uy, float uz) {
  // inputs outside [0, 1] (and NaN) are clamped, so every index stays in the table
  ux = fminf(fmaxf(ux, 0.0f), 1.0f);
  uy = fminf(fmaxf(uy, 0.0f), 1.0f);
  uz = fminf(fmaxf(uz, 0.0f), 1.0f);
  const float gx = ux * (float)N, gy = uy * (float)N, gz = uz * (float)N;
  const float fx = fminf(floorf(gx), (float)(N - 1)), fy = fminf(floorf(gy), (float)(N - 1)),
              fz = fminf(floorf(gz), (float)(N - 1));
  const float wx = gx - fx, wy = gy - fy, wz = gz - fz;
  const uint32_t bx = (uint32_t)fx, by = (uint32_t)fy, bz = (uint32_t)fz;
  const uint32_t n1 = (uint32_t)N + 1u;
  LevelCell c;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t ox = (k >> 2) & 1, oy = (k >> 1) & 1, oz = k & 1;
    const uint32_t cx = bx + ox, cy = by + oy, cz = bz + oz;
    c.idx[k] = dense ? cx + n1 * (cy + n1 * cz)
                     : ((cx * 1u) ^ (cy * 2654435761u) ^ (cz * 805459861u)) & tmask;
    c.w[k] = (ox ? wx : 1.0f - wx) * (oy ? wy : 1.0f - wy) * (oz ? wz : 1.0f - wz);
  }
  return c;
}

__device__ __forceinline__ bool level_dense(int N, int log2_table) {
  const double n1 = (double)N + 1.0;
  return n1 * n1 * n1 <= (double)(1u << log2_table);
}

// Levels of lane group g, in feature order: features 4g..4g+3 are levels
// 2g, 2g+1; features 16+4g..16+4g+3 are levels 8+2g, 9+2g.
__device__ __forceinline__ int lane_level(int g, int q) {
  return (q < 2 ? 2 * g : 8 + 2 * g) + (q & 1);
}

// Features of the lane's four levels from the FP32 tables.
__device__ __forceinline__ void encode_f32(const SurNet& net, int g, float ux, float uy,
                                           float uz, float (&feat)[8]) {
  const uint32_t T = 1u << net.log2_table, tmask = T - 1u;
  const float2* tab = reinterpret_cast<const float2*>(net.params);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int l = lane_level(g, q);
    const int N = net.res[l];
    const LevelCell c = level_cell(N, tmask, level_dense(N, net.log2_table), ux, uy, uz);
    // corners along x, mostly of one line, one after the other
    float2 e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = (j >> 1) | ((j & 1) << 2);
      e[k] = tab[(size_t)l * T + c.idx[k]];
    }
    float f0 = 0.0f, f1 = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      f0 = fmaf(c.w[k], e[k].x, f0);
      f1 = fmaf(c.w[k], e[k].y, f1);
    }
    feat[2 * q] = f0;
    feat[2 * q + 1] = f1;
  }
}

// ---------------------------------------------------------------------------
// Weight operands staged in LDS, pre-arranged per lane (one 8-byte read).
// ---------------------------------------------------------------------------
struct SurFwdLds {
  bf16x4 a1[4][2][64];  // layer 1: A = W1^T  [mt][k step][lane]
  bf16x4 a2[4][4][64];  // layer 2: A = W2^T  [mt][k block][lane]
};
struct SurBwdLds {
  bf16x4 bw2[4][4][64];  // dH1^T = W2 dH2^T:  A = W2  [in tile][out block][lane]
  bf16x4 bw1[2][4][64];  // dX^T  = W1 dH1^T:  A = W1  [feat tile][hidden block][lane]
};

__device__ __forceinline__ void stage_fwd(SurFwdLds& L, const float* W1, const float* W2) {
  for (int e = threadIdx.x; e < 4 * 2 * 64; e += blockDim.x) {
    const int lane = e & 63, ks = (e >> 6) & 1, mt = e >> 7;
    const int s = lane & 15, g = lane >> 4;
    bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = f2bf(W1[(size_t)(16 * ks + 4 * g + i) * kSurHidden + 16 * mt + s]);
    L.a1[mt][ks][lane] = v;
  }
  for (int e = threadIdx.x; e < 4 * 4 * 64; e += blockDim.x) {
    const int lane = e & 63, kb = (e >> 6) & 3, mt = e >> 8;
    const int s = lane & 15, g = lane >> 4;
    bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = f2bf(W2[(size_t)(16 * kb + 4 * g + i) * kSurHidden + 16 * mt + s]);
    L.a2[mt][kb][lane] = v;
  }
}

__device__ __forceinline__ void stage_bwd(SurBwdLds& L, const float* W1, const float* W2) {
  for (int e = threadIdx.x; e < 4 * 4 * 64; e += blockDim.x) {
    const int lane = e & 63, kb = (e >> 6) & 3, mt = e >> 8;
    const int s = lane & 15, g = lane >> 4;
    bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = f2bf(W2[(size_t)(16 * mt + s) * kSurHidden + 16 * kb + 4 * g + i]);
    L.bw2[mt][kb][lane] = v;
  }
  for (int e = threadIdx.x; e < 2 * 4 * 64; e += blockDim.x) {
    const int lane = e & 63, kb = (e >> 6) & 3, mt = e >> 8;
    const int s = lane & 15, g = lane >> 4;
    bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = f2bf(W1[(size_t)(16 * mt + s) * kSurHidden + 16 * kb + 4 * g + i]);
    L.bw1[mt][kb][lane] = v;
  }
}

// Forward pass of one 16-sample group.  Returns sigmoid(z) on every lane of
// the sample; h1/h2 receive the post-bias pre-activations.
struct SurAct {
  f32x4 h1[4], h2[4];
};

__device__ __forceinline__ float mlp_forward(const SurFwdLds& L, const float* b1,
                                             const float* b2, const float* w3, float b3,
                                             int lane, const float (&feat)[8], SurAct& a) {
  const int g = lane >> 4;
  bf16x4 x0, x1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x0[i] = f2bf(feat[i]);
    x1[i] = f2bf(feat[4 + i]);
  }
  bf16x4 h1b[4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    acc = mfma16(L.a1[mt][0][lane], x0, acc);
    acc = mfma16(L.a1[mt][1][lane], x1, acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i] += b1[16 * mt + 4 * g + i];
      h1b[mt][i] = f2bf(fmaxf(acc[i], 0.0f));
    }
    a.h1[mt] = acc;
  }
  float part = 0.0f;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc = mfma16(L.a2[mt][kb][lane], h1b[kb], acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i] += b2[16 * mt + 4 * g + i];
      part = fmaf(w3[16 * mt + 4 * g + i], fmaxf(acc[i], 0.0f), part);
    }
    a.h2[mt] = acc;
  }
  part += __shfl_xor(part, 16, 64);
  part += __shfl_xor(part, 32, 64);
  const float z = part + b3;
  return 1.0f / (1.0f + expf(-z));
}

// ---------------------------------------------------------------------------
// Training data.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {  // splitmix64 finalizer
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ float unit_float(uint64_t h) {
  return (float)(h >> 40) * (1.0f / 16777216.0f);  // 24 bits -> [0, 1)
}

__global__ void sur_labels_kernel(SurNet net, MarchParams scene, uint64_t seed, int64_t n,
                                  float* pts, float* labels) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint64_t base = seed * 0x9E3779B97F4A7C15ull + (uint64_t)k * 3ull;
  const float u0 = unit_float(mix64(base + 1)), u1 = unit_float(mix64(base + 2)),
              u2 = unit_float(mix64(base + 3));
  const double x = (double)net.lo[0] + (double)u0 * (double)net.ext[0];
  const double y = (double)net.lo[1] + (double)u1 * (double)net.ext[1];
  const double z = (double)net.lo[2] + (double)u2 * (double)net.ext[2];
  const double rho = node64<0>(scene.nodes, 0, x, y, z);
  pts[3 * k] = u0;
  pts[3 * k + 1] = u1;
  pts[3 * k + 2] = u2;
  labels[k] = (float)(rho / (double)net.rho_scale);
}

// ---------------------------------------------------------------------------
// Training step: forward, backward, gradient accumulation, in three kernels.
// Global memory takes 18 G FP32 adds/s wherever they land, and a step of n
// samples makes 256 n for the tables, and one kernel made 6337 per wave for the
// MLP.  So the first kernel only writes the gradients of the features, and each
// workgroup its own sum of the MLP's gradients, which the second adds up; in the
// third every slice of a table has a workgroup that owns it, meets all samples
// and adds in LDS (three cycles a lane: small levels, all of whose corners are
// in one slice, are shared out over parts of the samples as well).  65536
// samples, 2^17-entry tables: 940 us -> 82 + 7 + 188 us; a whole training step
// with 2^14, 2^17, 2^19 and 2^21 entries 0.96, 0.97, 1.02, 1.37 -> 0.24, 0.30,
// 0.40, 0.84 ms, of 1000 samples 0.33, 0.35, 0.40, 0.79 -> 0.07, 0.09, 0.15,
// 0.48.  Every workgroup meets all samples, so the gain goes with the number of
// slices: beyond kSurSlicesMost (2^22 entries and up) the tables' adds stay in
// global memory.
// ---------------------------------------------------------------------------
constexpr int kSurTrainWaves = 4;
constexpr int kSurTrainGroups = 256;         // workgroups of a launch, at most
constexpr uint32_t kSurSlice = 8192;         // entries of a slice: 64 KiB of LDS
constexpr int kSurScatterWaves = 16;
constexpr uint32_t kSurParts = 16;           // workgroups of a level, at least
constexpr uint32_t kSurSlicesMost = 4096;
constexpr int64_t kSurTrainChunk = 1 << 17;  // samples of a launch, at most

// Entries that level l's cells reach.
__host__ __device__ inline uint32_t sur_entries(const SurNet& net, int l) {
  const uint64_t n1 = (uint64_t)net.res[l] + 1u, t = 1ull << net.log2_table;
  // n1^3 <= t: the level is dense
  return (uint32_t)(n1 <= 4096u && n1 * n1 * n1 <= t ? n1 * n1 * n1 : t);
}
// Slices of a level, and workgroups of each (each with a part of the samples).
struct SurSlices {
  uint32_t n, parts;
};
__host__ __device__ inline SurSlices sur_slices(const SurNet& net, int l) {
  const uint32_t n = (sur_entries(net, l) + kSurSlice - 1) / kSurSlice;
  return {n, n < kSurParts ? (kSurParts + n - 1) / n : 1u};
}
inline uint32_t sur_slices(const SurNet& net) {
  uint32_t n = 0;
  for (int l = 0; l < kSurLevels; ++l) n += sur_slices(net, l).n * sur_slices(net, l).parts;
  return n;
}

struct SurWaveLds {
  short t1[64][16];  // h1 (post ReLU, bf16) [unit][sample]
  short t2[64][16];  // dH2 pre-activation gradient
  short tx[32][16];  // encoding features
  short t3[64][16];  // dH1 pre-activation gradient
};

__device__ __forceinline__ bf16x4 lds_row4(const short (*t)[16], int unit, int s0) {
  bf16x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = t[unit][s0 + i];
  return v;
}

// dx: the samples' feature gradients, [level][sample], or null (adds to the
// tables' gradients in `grads`).  sums: kSurMlpParams of each workgroup.
__global__ __launch_bounds__(256) void sur_train_kernel(SurNet net, const float* pts,
                                                        const float* labels, int64_t n,
                                                        float inv_n, float* grads, float2* dx_out,
                                                        float* sums, double* loss_sum) {
  __shared__ SurFwdLds F;
  __shared__ SurBwdLds B;
  __shared__ SurWaveLds WL[kSurTrainWaves];
  const SurOffsets off = sur_offsets(net.log2_table);
  const float* P = net.params;
  stage_fwd(F, P + off.W1, P + off.W2);
  stage_bwd(B, P + off.W1, P + off.W2);
  __shared__ float sum[kSurMlpParams];
  for (int e = threadIdx.x; e < kSurMlpParams; e += blockDim.x) sum[e] = 0.0f;
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = lane & 15, g = lane >> 4;
  SurWaveLds& W = WL[wave];
  const float* b1 = P + off.b1;
  const float* b2 = P + off.b2;
  const float* w3 = P + off.w3;
  const float b3 = P[off.b3];
  const uint32_t T = 1u << net.log2_table, tmask = T - 1u;
  float* gtab = grads;

  f32x4 accW2[4][4], accW1[2][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) accW2[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) accW1[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float db1[16], db2[16], dw3[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) db1[q] = db2[q] = dw3[q] = 0.0f;
  float db3 = 0.0f, sq = 0.0f;

  const int64_t step = (int64_t)gridDim.x * kSurTrainWaves * 16;
  for (int64_t first = ((int64_t)blockIdx.x * kSurTrainWaves + wave) * 16; first < n;
       first += step) {
    const int64_t k = first + s;
    const bool ok = k < n;
    const float ux = ok ? pts[3 * k] : 0.5f, uy = ok ? pts[3 * k + 1] : 0.5f,
                uz = ok ? pts[3 * k + 2] : 0.5f;
    const float t = ok ? labels[k] : 0.0f;
    float feat[8];
    encode_f32(net, g, ux, uy, uz, feat);
    SurAct a;
    const float y = mlp_forward(F, b1, b2, w3, b3, lane, feat, a);
    const float err = ok ? y - t : 0.0f;
    if (g == 0) sq = fmaf(err, err, sq);
    const float dz = 2.0f * err * inv_n * y * (1.0f - y);
    if (g == 0) db3 += dz;
    // layer 3 and the H2 ReLU
    bf16x4 dh2b[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int u = 16 * mt + 4 * g + i;
        const float h2 = fmaxf(a.h2[mt][i], 0.0f);
        dw3[4 * mt + i] = fmaf(dz, h2, dw3[4 * mt + i]);
        const float d = a.h2[mt][i] > 0.0f ? dz * w3[u] : 0.0f;
        db2[4 * mt + i] += d;
        dh2b[mt][i] = f2bf(d);
        W.t2[u][s] = dh2b[mt][i];
        W.t1[u][s] = f2bf(fmaxf(a.h1[mt][i], 0.0f));
      }
    // dH1^T = W2 dH2^T, then the H1 ReLU
    bf16x4 dh1b[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) acc = mfma16(B.bw2[mt][kb][lane], dh2b[kb], acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float d = a.h1[mt][i] > 0.0f ? acc[i] : 0.0f;
        db1[4 * mt + i] += d;
        dh1b[mt][i] = f2bf(d);
        W.t3[16 * mt + 4 * g + i][s] = dh1b[mt][i];
      }
    }
    // dX^T = W1 dH1^T: the lane's own features
    float dx[8];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) acc = mfma16(B.bw1[mt][kb][lane], dh1b[kb], acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dx[4 * mt + i] = acc[i];
        W.tx[16 * mt + 4 * g + i][s] = f2bf(feat[4 * mt + i]);
      }
    }
    // hash table gradients (only real samples)
    if (ok && dx_out) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        dx_out[(int64_t)lane_level(g, q) * n + k] = make_float2(dx[2 * q], dx[2 * q + 1]);
    } else if (ok) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int l = lane_level(g, q);
        const int N = net.res[l];
        const LevelCell c = level_cell(N, tmask, level_dense(N, net.log2_table), ux, uy, uz);
        float* gl = gtab + (size_t)l * T * 2;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          atomicAdd(gl + 2 * (size_t)c.idx[kk], c.w[kk] * dx[2 * q]);
          atomicAdd(gl + 2 * (size_t)c.idx[kk] + 1, c.w[kk] * dx[2 * q + 1]);
        }
      }
    }
    // weight gradients over the group's 16 samples, from the transposes in
    // LDS (this wave's own region; DS operations of one wave complete in
    // order, the fence keeps the compiler from reordering them)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const bf16x4 av = lds_row4(W.t1, 16 * mt + s, 4 * g);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        accW2[mt][nt] = mfma16(av, lds_row4(W.t2, 16 * nt + s, 4 * g), accW2[mt][nt]);
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const bf16x4 av = lds_row4(W.tx, 16 * mt + s, 4 * g);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        accW1[mt][nt] = mfma16(av, lds_row4(W.t3, 16 * nt + s, 4 * g), accW1[mt][nt]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // per-unit sums over the 16 samples (lanes of one group)
#pragma unroll
  for (int q = 0; q < 16; ++q)
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      db1[q] += __shfl_xor(db1[q], o, 64);
      db2[q] += __shfl_xor(db2[q], o, 64);
      dw3[q] += __shfl_xor(dw3[q], o, 64);
    }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    db3 += __shfl_xor(db3, o, 64);
    sq += __shfl_xor(sq, o, 64);
  }
  if (lane == 0) atomicAdd(loss_sum, (double)sq);
  // the workgroup's sum, a wave after the other (adds in LDS by atomics take
  // three cycles a lane); weight tiles hold D[m = 4g+i][n = s] of each (mt, nt)
  float* gW2 = sum + (off.W2 - off.W1);
  for (int w = 0; w < kSurTrainWaves; ++w) {
    __syncthreads();
    if (wave != w) continue;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          gW2[(16 * mt + 4 * g + i) * kSurHidden + 16 * nt + s] += accW2[mt][nt][i];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          sum[(16 * mt + 4 * g + i) * kSurHidden + 16 * nt + s] += accW1[mt][nt][i];
      }
    if (s == 0) {
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int u = 16 * (q >> 2) + 4 * g + (q & 3);
        sum[off.b1 - off.W1 + u] += db1[q];
        sum[off.b2 - off.W1 + u] += db2[q];
        sum[off.w3 - off.W1 + u] += dw3[q];
      }
    }
    if (lane == 0) sum[off.b3 - off.W1] += db3;
  }
  __syncthreads();
  float* out = sums + (size_t)blockIdx.x * kSurMlpParams;
  for (int e = threadIdx.x; e < kSurMlpParams; e += blockDim.x) out[e] = sum[e];
}

// grads[e] += the workgroups' sums: 64 parameters a workgroup, a wave per 16th
// of the sums.
__global__ __launch_bounds__(1024) void sur_sum_kernel(const float* sums, int groups,
                                                       float* grads) {
  __shared__ float part[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = blockIdx.x * 64 + lane;
  float a = 0.0f;
  if (e < kSurMlpParams)
    for (int q = wave; q < groups; q += 16) a += sums[(size_t)q * kSurMlpParams + e];
  part[wave][lane] = a;
  __syncthreads();
  if (wave == 0 && e < kSurMlpParams) {
    for (int q = 1; q < 16; ++q) a += part[q][lane];
    grads[e] += a;
  }
}

// The tables' gradients: a slice of kSurSlice entries of a level per workgroup,
// over all samples or a part of them.
__global__ __launch_bounds__(64 * kSurScatterWaves) void sur_scatter_kernel(
    SurNet net, const float* __restrict__ pts, const float2* __restrict__ dx, int64_t n,
    float* grads) {
  __shared__ float acc0[kSurSlice], acc1[kSurSlice];
  // the workgroup's level, part and slice
  int l = 0;
  uint32_t b = blockIdx.x;
  SurSlices sl = sur_slices(net, 0);
  while (b >= sl.n * sl.parts) {
    b -= sl.n * sl.parts;
    sl = sur_slices(net, ++l);
  }
  const uint32_t part = b / sl.n, first = (b - part * sl.n) * kSurSlice;
  const uint32_t count = min(sur_entries(net, l) - first, kSurSlice);
  for (uint32_t e = threadIdx.x; e < count; e += blockDim.x) acc0[e] = acc1[e] = 0.0f;
  __syncthreads();
  const uint32_t tmask = (1u << net.log2_table) - 1u;
  const int N = net.res[l];
  const bool dense = level_dense(N, net.log2_table);
  const float2* d = dx + (int64_t)l * n;
  for (int64_t k = (int64_t)part * blockDim.x + threadIdx.x; k < n;
       k += (int64_t)sl.parts * blockDim.x) {
    const float2 t = d[k];
    const LevelCell c =
        level_cell(N, tmask, dense, pts[3 * k], pts[3 * k + 1], pts[3 * k + 2]);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const uint32_t at = c.idx[q] - first;
      if (at < count) {
        atomicAdd(acc0 + at, c.w[q] * t.x);
        atomicAdd(acc1 + at, c.w[q] * t.y);
      }
    }
  }
  __syncthreads();
  float2* g = (float2*)grads + (((size_t)l << net.log2_table) + first);
  for (uint32_t e = threadIdx.x; e < count; e += blockDim.x) {
    const float2 a = make_float2(acc0[e], acc1[e]);
    if (a.x == 0.0f && a.y == 0.0f) continue;
    if (sl.parts == 1) {
      float2 v = g[e];
      v.x += a.x;
      v.y += a.y;
      g[e] = v;
    } else {
      atomicAdd(&g[e].x, a.x);
      atomicAdd(&g[e].y, a.y);
    }
  }
}

__global__ void sur_adam_kernel(float* params, const float* grads, float* m, float* v,
                                int64_t count, int64_t table_count, float lr_table,
                                float lr_mlp, float beta1, float beta2, float eps, float c1,
                                float c2) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  const float gk = grads[k];
  const float mk = beta1 * m[k] + (1.0f - beta1) * gk;
  const float vk = beta2 * v[k] + (1.0f - beta2) * gk * gk;
  m[k] = mk;
  v[k] = vk;
  const float lr = k < table_count ? lr_table : lr_mlp;
  params[k] -= lr * (mk * c1) / (sqrtf(vk * c2) + eps);
}

__global__ void sur_pack_kernel(const float* tables, uint32_t* out, int64_t entries) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= entries) return;
  const uint32_t lo = (uint16_t)f2bf(tables[2 * k]), hi = (uint16_t)f2bf(tables[2 * k + 1]);
  out[k] = lo | (hi << 16);
}

__global__ __launch_bounds__(256) void sur_predict_kernel(SurNet net, const float* pts,
                                                          int64_t n, float* out) {
  __shared__ SurFwdLds F;
  const SurOffsets off = sur_offsets(net.log2_table);
  const float* P = net.params;
  stage_fwd(F, P + off.W1, P + off.W2);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = lane & 15, g = lane >> 4;
  const int64_t k = ((int64_t)blockIdx.x * 4 + wave) * 16 + s;
  const bool ok = k < n;
  const float ux = ok ? pts[3 * k] : 0.5f, uy = ok ? pts[3 * k + 1] : 0.5f,
              uz = ok ? pts[3 * k + 2] : 0.5f;
  float feat[8];
  encode_f32(net, g, ux, uy, uz, feat);
  SurAct a;
  const float y = mlp_forward(F, P + off.b1, P + off.b2, P + off.w3, P[off.b3], lane, feat, a);
  if (ok && g == 0) out[k] = y;
}

// ---------------------------------------------------------------------------
// Surrogate march.  One wave = 16 rays (a 4x4 pixel block), one sample of
// each per step, midpoint rule with step ds_sur; the four lanes of a ray
// encode four levels each.  FP64 ray set-up and clipping, FP32 positions
// re-anchored in FP64 every kChunk steps, Kahan-compensated FP32 sum.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool sur_domain(const SurNet& net, float x, float y, float z,
                                           float& ux, float& uy, float& uz) {
  if (net.wrap) {
    if (x < net.bounds[0] || x > net.bounds[1] || y < net.bounds[2] || y > net.bounds[3] ||
        z < net.bounds[4] || z > net.bounds[5])
      return false;
    ux = (x - net.lo[0]) * net.inv_ext[0];
    uy = (y - net.lo[1]) * net.inv_ext[1];
    uz = (z - net.lo[2]) * net.inv_ext[2];
    ux -= floorf(ux);
    uy -= floorf(uy);
    uz -= floorf(uz);
    return true;
  }
  ux = (x - net.lo[0]) * net.inv_ext[0];
  uy = (y - net.lo[1]) * net.inv_ext[1];
  uz = (z - net.lo[2]) * net.inv_ext[2];
  return ux >= 0.0f && ux <= 1.0f && uy >= 0.0f && uy <= 1.0f && uz >= 0.0f && uz <= 1.0f;
}

// The march's operands in LDS: the weights' and, per unit tile and lane group,
// the four biases (of both layers) and output weights that group's lanes use.
constexpr uint32_t kSurLdsEntries = 37600;  // 147 KiB
struct SurMlpLds {
  SurFwdLds F;
  f32x4 b1[4][4], b2[4][4], w3[4][4];
};
struct SurMarchLds : SurMlpLds {
  uint32_t tab[kSurLdsEntries];  // tables of the first levels, as many as fit
};
static_assert(sizeof(SurMarchLds) <= 160 * 1024, "one workgroup a CU");

// A lane's four hash levels: cells per axis, the strides of y and z (of a
// dense level's grid, or the hash's factors) and the first table entry, in
// LDS or in the level's global table.
struct SurLevels {
  float n[4];
  uint32_t y[4], z[4], first[4];
  bool dense[4], lds[4];
};

__device__ __forceinline__ SurLevels sur_levels(const SurNet& net, int g, int n_lds) {
  SurLevels L;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int l = lane_level(g, q), N = net.res[l];
    L.dense[q] = level_dense(N, net.log2_table);
    L.n[q] = (float)N;
    L.y[q] = L.dense[q] ? (uint32_t)N + 1u : 2654435761u;
    L.z[q] = L.dense[q] ? ((uint32_t)N + 1u) * ((uint32_t)N + 1u) : 805459861u;
    L.lds[q] = l < n_lds;
    L.first[q] = (uint32_t)l << net.log2_table;
    if (L.lds[q]) {
      L.first[q] = 0;
      for (int k = 0; k < l; ++k) L.first[q] += sur_entries(net, k);
    }
  }
  return L;
}

// The lane's features at u in [0, 1]^3 from the packed BF16 tables: all 32
// gathers first, then the sums, whose terms and order are encode_f32's.
template <bool LDS>
__device__ __forceinline__ void encode_bf16(const uint32_t* __restrict__ tab,
                                            const uint32_t* lds_tab, uint32_t tmask,
                                            const SurLevels& L, float ux, float uy, float uz,
                                            float (&feat)[8]) {
  uint32_t e[4][8];
  float w[4][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float gx = ux * L.n[q], gy = uy * L.n[q], gz = uz * L.n[q];
    const float top = L.n[q] - 1.0f;
    const float fx = fminf(floorf(gx), top), fy = fminf(floorf(gy), top),
                fz = fminf(floorf(gz), top);
    w[q][0] = gx - fx, w[q][1] = gy - fy, w[q][2] = gz - fz;
    const uint32_t x = (uint32_t)fx, y = (uint32_t)fy * L.y[q], z = (uint32_t)fz * L.z[q];
    uint32_t at[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t cx = x + ((k >> 2) & 1), cy = y + ((k >> 1) & 1) * L.y[q],
                     cz = z + (k & 1) * L.z[q];
      at[k] = L.first[q] + (L.dense[q] ? cx + cy + cz : (cx ^ cy ^ cz) & tmask);
    }
    if (LDS && L.lds[q]) {
#pragma unroll
      for (int k = 0; k < 8; ++k) e[q][k] = lds_tab[at[k]];
    } else {
      // 32-bit byte offsets (16 levels of at most 2^24 entries); the two
      // corners along x, mostly of one line, one after the other
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = (j >> 1) | ((j & 1) << 2);
        e[q][k] = *(const uint32_t*)((const char*)tab + (at[k] << 2));
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float f0 = 0.0f, f1 = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float c = ((k & 4) ? w[q][0] : 1.0f - w[q][0]) *
                      ((k & 2) ? w[q][1] : 1.0f - w[q][1]) *
                      ((k & 1) ? w[q][2] : 1.0f - w[q][2]);
      f0 = fmaf(c, bf2f(e[q][k] & 0xffffu), f0);
      f1 = fmaf(c, bf2f(e[q][k] >> 16), f1);
    }
    feat[2 * q] = f0;
    feat[2 * q + 1] = f1;
  }
}

// mlp_forward with its constants in LDS and no activations kept.
__device__ __forceinline__ float mlp_density(const SurMlpLds& L, float b3, int lane,
                                             const float (&feat)[8]) {
  const int g = lane >> 4;
  const bf16x4 x0 = f2bf4(feat[0], feat[1], feat[2], feat[3]);
  const bf16x4 x1 = f2bf4(feat[4], feat[5], feat[6], feat[7]);
  bf16x4 h[4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    acc = mfma16(L.F.a1[mt][0][lane], x0, acc);
    acc = mfma16(L.F.a1[mt][1][lane], x1, acc);
    const f32x4 b = L.b1[mt][g];
    h[mt] = f2bf4(fmaxf(acc[0] + b[0], 0.0f), fmaxf(acc[1] + b[1], 0.0f),
                  fmaxf(acc[2] + b[2], 0.0f), fmaxf(acc[3] + b[3], 0.0f));
  }
  float part = 0.0f;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc = mfma16(L.F.a2[mt][kb][lane], h[kb], acc);
    const f32x4 b = L.b2[mt][g], w = L.w3[mt][g];
#pragma unroll
    for (int i = 0; i < 4; ++i) part = fmaf(w[i], fmaxf(acc[i] + b[i], 0.0f), part);
  }
  part += __shfl_xor(part, 16, 64);
  part += __shfl_xor(part, 32, 64);
  return 1.0f / (1.0f + expf(-(part + b3)));
}

// RESIDENT: one workgroup a CU, which stays for the launch: it stages the weights and
// tables once, and its waves take tiles (16 rays, 4x4 pixels) from the counter
// p.counts until none is left (kStatStride words after it, kBatchSinkBytes that
// the adds of a wave's other lanes go to).
//
// The gathers bound it: 64 lines of a step's 128 corners are distinct for each
// sample (fine cells are smaller than the pixel spacing), and L1 and L2 are
// smaller than what the waves have in flight and the tables.  Of 2^17-entry
// tables (8 MiB), 4 x 256^2 rays at step 0.008: 3.18 ms with one wave per
// workgroup and the corners in index order; 3.3 with this workgroup's operands
// in LDS; 2.57 with the first levels' tables in LDS as well (three of 16 levels'
// requests gone, 2 waves a SIMD); 2.1 with the corners along x, mostly of one
// line, loaded one after the other (L2 requests 340 -> 212 M).  2 waves a SIMD:
// 2.11 ms; 2.31 at 1, 2.48 at 3 and 2.57 at 4, which evict each other's lines.
// One 8-byte load for an aligned pair of corners: 2.58 ms.
constexpr int kSurMarchWaves = 8;
constexpr int kSurGroups = 256;
// RESIDENT = false, for launches of fewer tiles than kSurResidentLeast: a
// one-wave workgroup per tile, which keeps the operands in registers.  Such a
// launch lasts as long as one wave's chain of steps, which the LDS reads
// lengthen: 2^17-entry tables, 400, 2025, 3249, 4096 (one view, four views) and
// 16384 tiles 0.45, 0.48, 0.69, 1.28, 1.55 and 2.51 ms, resident 0.93, 0.92,
// 1.20, 1.26, 1.12 and 2.05 ms.
constexpr unsigned kSurResidentLeast = 4096;

template <bool RESIDENT>
__global__ __launch_bounds__(RESIDENT ? 64 * kSurMarchWaves : 64)
    __attribute__((amdgpu_waves_per_eu(2))) void sur_render_kernel(SurNet net, MarchParams p,
                                                                   double ds_sur, long K,
                                                                   unsigned n_tiles) {
  __shared__ std::conditional_t<RESIDENT, SurMarchLds, SurMlpLds> L;
  const uint32_t* lds_tab = nullptr;
  const SurOffsets off = sur_offsets(net.log2_table);
  const float* P = net.params;
  stage_fwd(L.F, P + off.W1, P + off.W2);
  if (threadIdx.x < 64) {
    ((float*)L.b1)[threadIdx.x] = P[off.b1 + threadIdx.x];
    ((float*)L.b2)[threadIdx.x] = P[off.b2 + threadIdx.x];
    ((float*)L.w3)[threadIdx.x] = P[off.w3 + threadIdx.x];
  }
  int n_lds = 0;
  if constexpr (RESIDENT) {
    lds_tab = L.tab;
    for (uint32_t at = 0; n_lds < kSurLevels; ++n_lds) {
      const uint32_t n = sur_entries(net, n_lds);
      if (n > kSurLdsEntries - at) break;
      const uint32_t* t = net.table_bf16 + ((size_t)n_lds << net.log2_table);
      for (uint32_t e = threadIdx.x; e < n; e += blockDim.x) L.tab[at + e] = t[e];
      at += n;
    }
  }
  __syncthreads();
  const float b3 = P[off.b3];
  const int lane = threadIdx.x & 63;
  const int s = lane & 15, g = lane >> 4;
  const SurLevels levels = sur_levels(net, g, n_lds);
  const uint32_t tmask = (1u << net.log2_table) - 1u;
  const int tiles_j = (p.res + 3) >> 2;
  const unsigned per_view = (unsigned)tiles_j * (unsigned)tiles_j;
  const float dsf = (float)ds_sur;
  unsigned long long n_samples = 0;

  // the next tile, by an atomic of every lane (eval_device.hpp lane_slot)
  auto next = [&]() -> unsigned {
    if constexpr (!RESIDENT) return n_tiles;
    unsigned long long* sink = (unsigned long long*)p.counts + kStatStride;
    return __builtin_amdgcn_readfirstlane(
        atomicAdd(lane_slot(p.counts, sink), first_lane() ? 1u : 0u));
  };
  for (unsigned tile = RESIDENT ? next() : blockIdx.x; tile < n_tiles; tile = next()) {
    const int v = (int)(tile / per_view);
    const int in_view = (int)(tile - (unsigned)v * per_view);
    const int ti = in_view / tiles_j, tj = in_view - ti * tiles_j;
    const int i = ti * 4 + (s >> 2);
    const int j = tj * 4 + (s & 3);
    const bool valid = i < p.res && j < p.res;

    long k_lo = 1, k_hi = 0;
    Ray r;
    r.o[0] = r.o[1] = r.o[2] = 0.0;
    r.d[0] = r.d[1] = r.d[2] = 0.0;
    if (valid) {
      r = make_ray(p, p.views[p.view_offset + v], i, j);
      double t_in, t_out;
      if (clip_ray(p, r, t_in, t_out)) {
        double a = floor((t_in - p.smin) / ds_sur - 0.5) - 1.0;
        double b = ceil((t_out - p.smin) / ds_sur - 0.5) + 1.0;
        k_lo = a > 0.0 ? (long)a : 0;
        k_hi = b < (double)(K - 1) ? (long)b : K - 1;
      }
    }
    long wlo = k_lo, whi = k_hi;
    // the union of the wave's sample ranges (empty ranges have lo > hi)
    if (k_lo > k_hi) {
      wlo = 0x7fffffffffffL;
      whi = -1;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      wlo = min(wlo, (long)__shfl_xor(wlo, o, 64));
      whi = max(whi, (long)__shfl_xor(whi, o, 64));
    }
    if (whi >= wlo) n_samples += (unsigned long long)(whi - wlo + 1) * 16ull;
    float acc = 0.0f, comp = 0.0f;
    const float d0 = (float)r.d[0], d1 = (float)r.d[1], d2 = (float)r.d[2];
    for (long k0 = wlo; k0 <= whi; k0 += kChunk) {
      const double sa = p.smin + ((double)k0 + 0.5) * ds_sur;
      const float a0 = (float)(r.o[0] + r.d[0] * sa), a1 = (float)(r.o[1] + r.d[1] * sa),
                  a2 = (float)(r.o[2] + r.d[2] * sa);
      const int n = (int)min((long)kChunk, whi - k0 + 1);
      // the ray's own samples of the chunk
      const int lo = (int)max(min(k_lo - k0, (long)kChunk), 0l),
                hi = (int)max(min(k_hi - k0, (long)kChunk), -1l);
      for (int jj = 0; jj < n; ++jj) {
        const float sj = (float)jj * dsf;
        float x = fmaf(d0, sj, a0), y = fmaf(d1, sj, a1), z = fmaf(d2, sj, a2);
        deform32(p.defs, p.n_defs, x, y, z);
        float ux = 0.5f, uy = 0.5f, uz = 0.5f;
        const bool in = sur_domain(net, x, y, z, ux, uy, uz) && jj >= lo && jj <= hi;
        float feat[8];
        encode_bf16<RESIDENT>(net.table_bf16, lds_tab, tmask, levels, in ? ux : 0.5f, in ? uy : 0.5f,
                    in ? uz : 0.5f, feat);
        // an index the compiler takes as new in every step: it would otherwise
        // keep the operands in 144 registers
        int operand_lane = lane;
        if constexpr (RESIDENT) asm volatile("" : "+v"(operand_lane));
        const float dens = mlp_density(L, b3, operand_lane, feat);
        const float rho = in ? dens * net.rho_scale : 0.0f;
        const float yk = rho - comp;
        const float tt = acc + yk;
        comp = (tt - acc) - yk;
        acc = tt;
      }
    }
    if (valid && g == 0) {
      const double T = p.flat_field + ((double)acc * p.dm) * ds_sur;
      store_pixel(p, v, i, j, T);
    }
  }
  if (p.stats && lane == 0 && n_samples) atomicAdd(p.stats + ST_SAMPLES, n_samples);
}

// ---------------------------------------------------------------------------
// MFMA operand layout probe: a, b, d are 16x16 row-major float matrices.
// ---------------------------------------------------------------------------
__global__ void mfma_probe_kernel(const float* a, const float* b, float* d) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  bf16x4 av, bv;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    av[i] = f2bf(a[r * 16 + 4 * g + i]);   // A[m = lane%16][k = 4g+i]
    bv[i] = f2bf(b[(4 * g + i) * 16 + r]);  // B[k = 4g+i][n = lane%16]
  }
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  acc = mfma16(av, bv, acc);
#pragma unroll
  for (int i = 0; i < 4; ++i) d[(4 * g + i) * 16 + r] = acc[i];  // D[m = 4g+i][n = lane%16]
}

// Image values at listed pixels (view, i, j) of a [view][i][j] image.
__global__ void gather_pixels_kernel(const float* img, const int* items, int n, int res,
                                     float* out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const size_t off =
      ((size_t)items[3 * k] * res + (size_t)items[3 * k + 1]) * res + (size_t)items[3 * k + 2];
  out[k] = img[off];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sur_certify_kernel(float* img, const float* exact,
                                                          int res, float tol,
                                                          unsigned* counters) {
  __shared__ float wave_max[4];
  const int tiles_side = (res + 15) / 16;
  const int ti = blockIdx.x / tiles_side, tj = blockIdx.x - ti * tiles_side;
  const int i = ti * 16 + (threadIdx.x >> 4), j = tj * 16 + (threadIdx.x & 15);
  const bool in = i < res && j < res;
  const size_t at = ((size_t)blockIdx.y * res + (in ? i : 0)) * res + (in ? j : 0);
  const float e = in ? exact[at] : 0.0f;
  float d = in ? fabsf(img[at] - e) : 0.0f;
  if (!(d == d)) d = INFINITY;  // a NaN never passes
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) d = fmaxf(d, __shfl_xor(d, off, 64));
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = d;
  __syncthreads();
  const float m = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
  if (m > tol && in) img[at] = e;
  if (threadIdx.x == 0) {
    if (m > tol) atomicAdd(counters, 1u);
    atomicMax(counters + 1, __float_as_uint(m));  // non-negative: bits order like values
  }
}

int launch_sur_certify(float* img, const float* exact, int n_views, int res, float tol,
                       unsigned* counters, void* stream) {
  if (n_views <= 0 || res <= 0) return 0;
  const int tiles_side = (res + 15) / 16;
  hipLaunchKernelGGL(sur_certify_kernel, dim3(tiles_side * tiles_side, n_views), dim3(256), 0,
                     (hipStream_t)stream, img, exact, res, tol, counters);
  return (int)hipGetLastError();
}

int launch_gather_pixels(const float* img, const int* items, int n, int res, float* out,
                         void* stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(gather_pixels_kernel, dim3((n + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, img, items, n, res, out);
  return (int)hipGetLastError();
}

int launch_sur_labels(const SurNet& net, const MarchParams& scene, uint64_t seed, int64_t n,
                      float* pts, float* labels, void* stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(sur_labels_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, net, scene, seed, n, pts, labels);
  return (int)hipGetLastError();
}

static int64_t sur_train_chunk(int64_t n) { return std::min(n, kSurTrainChunk); }

// Whether the tables' gradients are added by slices ($XRP_SUR_SLICES: fewer
// slices at most, for tests; read per batch).
static bool sur_sliced(const SurNet& net) {
  uint32_t most = kSurSlicesMost;
  if (const char* e = std::getenv("XRP_SUR_SLICES"))
    most = (uint32_t)std::min<long>(most, std::max(0L, std::atol(e)));
  return sur_slices(net) <= most;
}

size_t sur_train_bytes(const SurNet& net, int64_t n) {
  const size_t sums = (size_t)kSurTrainGroups * kSurMlpParams * sizeof(float);
  return sums + (sur_sliced(net) ? (size_t)sur_train_chunk(n) * kSurLevels * sizeof(float2) : 0);
}

int launch_sur_train(const SurNet& net, const float* pts, const float* labels, int64_t n,
                     float inv_n, float* grads, double* loss_sum, void* work, void* stream) {
  const uint32_t slices = sur_slices(net);
  float2* dx = sur_sliced(net) ? (float2*)work : nullptr;
  float* sums = (float*)work + (dx ? (size_t)sur_train_chunk(n) * kSurLevels * 2 : 0);
  hipStream_t s = (hipStream_t)stream;
  for (int64_t at = 0; at < n; at += kSurTrainChunk) {
    const int64_t c = std::min(n - at, kSurTrainChunk);
    const int64_t waves = (c + 15) / 16;
    const int groups =
        (int)std::min<int64_t>((waves + kSurTrainWaves - 1) / kSurTrainWaves, kSurTrainGroups);
    hipLaunchKernelGGL(sur_train_kernel, dim3(groups), dim3(64 * kSurTrainWaves), 0, s, net,
                       pts + 3 * at, labels + at, c, inv_n, grads, dx, sums, loss_sum);
    hipLaunchKernelGGL(sur_sum_kernel, dim3((kSurMlpParams + 63) / 64), dim3(1024), 0, s, sums,
                       groups, grads + sur_table_floats(net.log2_table));
    if (dx)
      hipLaunchKernelGGL(sur_scatter_kernel, dim3(slices), dim3(64 * kSurScatterWaves), 0, s,
                         net, pts + 3 * at, dx, c, grads);
  }
  return (int)hipGetLastError();
}

int launch_sur_adam(float* params, const float* grads, float* m, float* v, int64_t count,
                    int64_t table_count, float lr_table, float lr_mlp, float beta1,
                    float beta2, float eps, int step, void* stream) {
  const float c1 = 1.0f / (1.0f - powf(beta1, (float)step));
  const float c2 = 1.0f / (1.0f - powf(beta2, (float)step));
  hipLaunchKernelGGL(sur_adam_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, params, grads, m, v, count, table_count, lr_table,
                     lr_mlp, beta1, beta2, eps, c1, c2);
  return (int)hipGetLastError();
}

int launch_sur_pack_tables(const SurNet& net, void* stream) {
  const int64_t entries = (int64_t)kSurLevels << net.log2_table;
  hipLaunchKernelGGL(sur_pack_kernel, dim3((unsigned)((entries + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, net.params, net.table_bf16, entries);
  return (int)hipGetLastError();
}

int launch_sur_predict(const SurNet& net, const float* pts, int64_t n, float* out,
                       void* stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(sur_predict_kernel, dim3((unsigned)((n + 63) / 64)), dim3(256), 0,
                     (hipStream_t)stream, net, pts, n, out);
  return (int)hipGetLastError();
}

int launch_sur_render(const SurNet& net, const MarchParams& p, double ds_sur, void* stream) {
  const long K = (long)std::ceil((p.smax - p.smin) / ds_sur);
  const int64_t tiles = (int64_t)((p.res + 3) / 4) * ((p.res + 3) / 4) * p.n_views;
  // tile numbers go past the last by one per wave
  if (tiles > 0xf0000000ll || !p.counts) return (int)hipErrorInvalidValue;
  if (tiles < kSurResidentLeast)
    hipLaunchKernelGGL((sur_render_kernel<false>), dim3((unsigned)tiles), dim3(64), 0,
                       (hipStream_t)stream, net, p, ds_sur, K, (unsigned)tiles);
  else
    hipLaunchKernelGGL((sur_render_kernel<true>), dim3(kSurGroups), dim3(64 * kSurMarchWaves), 0,
                       (hipStream_t)stream, net, p, ds_sur, K, (unsigned)tiles);
  return (int)hipGetLastError();
}

int launch_mfma_probe(const float* a, const float* b, float* d, void* stream) {
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, a, b, d);
  return (int)hipGetLastError();
}

}  // namespace xrp
