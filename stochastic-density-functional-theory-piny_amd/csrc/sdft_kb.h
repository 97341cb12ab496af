// sdft_kb.h -- tiles of the Kleinman-Bylander products (sdft_gemm.hip) on the
// matrix cores: the projection over a slice of coefficients and the force
// product.
#pragma once
#include "sdft_internal.h"

namespace sdft {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <typename TI>
struct Mfma;

// Operand layout of both 16x16x4 instructions: lane l holds A[l%16][l/16]
// and B[l/16][l%16].  Accumulator register r of lane l holds column l%16 and
// row `row(l, r)`: rows 4(l/16)+r for the FP32 form, rows l/16+4r for FP64.
template <>
struct Mfma<double> {
  typedef d4_t acc_t;
  __device__ static inline acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};

template <>
struct Mfma<float> {
  typedef f4_t acc_t;
  __device__ static inline acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

constexpr int KS = 32;   // K per step: 4 lane groups x 8 consecutive k
constexpr int KPL = 8;   // k per lane per step

// 8 consecutive values src[0..7] in 16-byte vector loads (src is 32-byte
// aligned for float, 64-byte for double: row strides and run starts are
// multiples of 8 elements of 256-byte aligned buffers)
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
  typedef float type __attribute__((ext_vector_type(4)));
  static constexpr int n = 4;
};
template <>
struct Vec16<double> {
  typedef double type __attribute__((ext_vector_type(2)));
  static constexpr int n = 2;
};

template <typename T>
__device__ inline void load_run(const T* __restrict__ src, T (&dst)[KPL]) {
  typedef typename Vec16<T>::type V;
  constexpr int NV = Vec16<T>::n;
  const V* s = reinterpret_cast<const V*>(src);
#pragma unroll
  for (int v = 0; v < KPL / NV; ++v) {
    const V x = s[v];
#pragma unroll
    for (int e = 0; e < NV; ++e) dst[v * NV + e] = x[e];
  }
}

// ---- Z partials: zpart[z][p][s] = sum_{k in split z} A[p][k] X[s][k] -------
// Tiles (ceil(P/32), ceil(ns/32), nsplit); the NWV waves of a workgroup share
// the 32x32 output tile and interleave the split's K steps; their partial
// tiles are summed through LDS (`red`, NWV tiles).  AHEAD: the next step's
// operands are loaded before the current step's products (twice the operand
// registers).  Both operands must have their row count
// padded to a multiple of 32 with readable rows (zeros, or values whose
// products land only in the rows / columns the epilogue does not store):
// the K loop loads without bounds tests.
template <typename TA, typename TX, typename TI, int NWV = 4, bool AHEAD = true>
__device__ __forceinline__ void kb_project_tile(const TA* __restrict__ A,
                                                const TX* __restrict__ X, int P, int ns,
                                                int K, int ksteps_per_split,
                                                double* __restrict__ zpart, int bx, int by, int bz,
                                                double* __restrict__ red) {
  typedef typename Mfma<TI>::acc_t acc_t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar K loop
  const int p0 = bx * 32, s0 = by * 32;
  const int g = lane >> 4, r16 = lane & 15;
  acc_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = TI(0);
  // Without AHEAD a split is many steps long (few splits, so that there are few
  // partials to read again), and each step's sums go to FP64 sums of their own:
  // one chain over the split rounded worse than the short chains of many splits
  // (H psi of 8 orbitals at 64^3, error of its norm: FP32 3.8e-8, with these sums
  // 2.4e-8, short chains 2.8e-8; FP64 8.9e-17, 6.7e-17, 7.0e-17).
  constexpr int NS = AHEAD ? 1 : 2;
  double sum[NS][NS][2 * NS] = {};
  const int step0 = bz * ksteps_per_split;
  const int nsteps_total = K / KS;
  const int step1 = min(nsteps_total, step0 + ksteps_per_split);
  const TA* arow[2];
  const TX* xrow[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    arow[i] = A + (size_t)(p0 + 16 * i + r16) * K + KPL * g;
    xrow[i] = X + (size_t)(s0 + 16 * i + r16) * K + KPL * g;
  }
  // Operands are loaded in their storage types and converted to TI only at
  // the MFMAs.  The next step's loads are issued under a condition, and the
  // compiler's wait before the current step's MFMAs then covers them too, so
  // a wave does not overlap its loads with its MFMAs.  A counted, branch-free
  // form that does (correct waits, rings of 2-6 steps in flight) ran the
  // products 6 % faster alone at 2 steps and slower at more; beside the
  // plane kernel on the other stream it left the Si64 step unchanged and
  // the fragment batch 1 % slower.  These products are bound by how the
  // memory system serves their operand stream, shared with the plane kernel.
  TA ra0[2][KPL], ra1[2][KPL];
  TX rb0[2][KPL], rb1[2][KPL];
  auto load_raw = [&](int st, TA (&a)[2][KPL], TX (&b)[2][KPL]) {
    const int k0 = st * KS;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      load_run<TA>(arow[i] + k0, a[i]);
      load_run<TX>(xrow[i] + k0, b[i]);
    }
  };
  auto mma_raw = [&](TA (&a)[2][KPL], TX (&b)[2][KPL]) {
#pragma unroll
    for (int t = 0; t < KPL; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = Mfma<TI>::run(TI(a[i][t]), TI(b[j][t]), acc[i][j]);
  };
  int st = step0 + wave;
  if constexpr (AHEAD) {
    if (st < step1) load_raw(st, ra0, rb0);
    while (st < step1) {
      const int nx = st + NWV;
      if (nx < step1) load_raw(nx, ra1, rb1);
      mma_raw(ra0, rb0);
      st = nx;
      if (st >= step1) break;
      const int nx2 = st + NWV;
      if (nx2 < step1) load_raw(nx2, ra0, rb0);
      mma_raw(ra1, rb1);
      st = nx2;
    }
  } else {
    for (; st < step1; st += NWV) {
      load_raw(st, ra0, rb0);
      mma_raw(ra0, rb0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            sum[i][j][r] += double(acc[i][j][r]);
            acc[i][j][r] = TI(0);
          }
    }
  }
  // sum the waves' tiles
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + Mfma<TI>::row(lane, r);
        const int col = 16 * j + r16;
        if constexpr (AHEAD)
          red[wave * 1024 + row * 32 + col] = double(acc[i][j][r]);
        else
          red[wave * 1024 + row * 32 + col] = sum[i][j][r];
      }
  __syncthreads();
  double* zp = zpart + (size_t)bz * P * ns;
  for (int e = tid; e < 32 * 32; e += 64 * NWV) {
    const int row = e >> 5, col = e & 31;
    const int p = p0 + row, s = s0 + col;
    if (p < P && s < ns) {
      double z = red[e];
#pragma unroll
      for (int w = 1; w < NWV; ++w) z += red[w * 1024 + e];
      zp[(size_t)p * ns + s] = z;
    }
  }
}

// ---- F[s][k] = sum_p Y[s][p] At[k][p] ----------------------------------------
// The reduction (over the padded projector index, ppad) is short, so it is
// not split across waves: a workgroup covers 32 rows s x 64 NJ columns k,
// wave w owns columns 16 NJ w .. 16 NJ (w + 1) - 1 of that block (2 x NJ MFMA
// blocks) and runs the whole reduction (two-stage pipeline as above), and the
// accumulators are stored directly -- no LDS, no barrier.  K2 is a multiple
// of 128, so a wave's columns lie either all below K2 or all above (that
// wave returns at once).  NJ = 2 keeps the kernel's registers low enough for
// it to run beside the plane kernel on the other stream (NJ = 4 reuses each
// Y run twice as often but needs about twice the registers).  Y has its rows padded
// to a multiple of 32 with readable memory.  All operands and F are in the
// form's type T (float for FP32: the MFMA's own operand and accumulator type).
constexpr int kForceNJ = kForceCols / 64;

template <typename T>
__device__ __forceinline__ void kb_force_block(const T* __restrict__ Y, const T* __restrict__ At,
                                               int ns, int K2, int ppad, T* __restrict__ F,
                                               int bx, int by) {
  constexpr int NJ = kForceNJ;
  typedef typename Mfma<T>::acc_t acc_t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s0 = bx * 32, k0 = by * (64 * NJ) + wave * (16 * NJ);
  if (k0 >= K2) return;
  const int g = lane >> 4, r16 = lane & 15;
  acc_t acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = T(0);
  const T* arow[2];
  const T* xrow[NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i) arow[i] = Y + (size_t)(s0 + 16 * i + r16) * ppad + KPL * g;
#pragma unroll
  for (int j = 0; j < NJ; ++j) xrow[j] = At + (size_t)(k0 + 16 * j + r16) * ppad + KPL * g;
  T ra0[2][KPL], ra1[2][KPL];
  T rb0[NJ][KPL], rb1[NJ][KPL];
  auto load_raw = [&](int st, T (&a)[2][KPL], T (&b)[NJ][KPL]) {
    const int kk = st * KS;
#pragma unroll
    for (int i = 0; i < 2; ++i) load_run<T>(arow[i] + kk, a[i]);
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_run<T>(xrow[j] + kk, b[j]);
  };
  auto mma_raw = [&](T (&a)[2][KPL], T (&b)[NJ][KPL]) {
#pragma unroll
    for (int t = 0; t < KPL; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = Mfma<T>::run(a[i][t], b[j][t], acc[i][j]);
  };
  const int nsteps = ppad / KS;
  if constexpr (sizeof(T) == 4) {
    int st = 0;
    load_raw(0, ra0, rb0);
    while (st < nsteps) {
      if (st + 1 < nsteps) load_raw(st + 1, ra1, rb1);
      mma_raw(ra0, rb0);
      if (++st >= nsteps) break;
      if (st + 1 < nsteps) load_raw(st + 1, ra0, rb0);
      mma_raw(ra1, rb1);
      ++st;
    }
  } else {
    // FP64: one operand set in flight (64 fewer VGPRs: 4 waves per SIMD
    // instead of 2 hide the load latency)
    for (int st = 0; st < nsteps; ++st) {
      load_raw(st, ra0, rb0);
      mma_raw(ra0, rb0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = s0 + 16 * i + Mfma<T>::row(lane, r);
      if (s < ns) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) F[(size_t)s * K2 + k0 + 16 * j + r16] = acc[i][j][r];
      }
    }
}

// The two products of a system too small for a launch each: the split's
// partials are summed while they are brought into LDS as Y (one tile of up to
// 32 states, a row each, row stride kb_small_ldy), and the force product reads Y from there.
// Workgroup (bx, by): states 32 bx .., columns 64 by .. 64 by + 63 (16 per
// wave).  Every workgroup sums its tile's partials again: they come from L2
// (at most kKbFusedPartials of them a tile).
__host__ __device__ constexpr int kb_small_ldy(int ppad) { return ppad + 4; }

template <typename T>
__device__ __forceinline__ void kb_reduce_force(const double* __restrict__ zpart, int nsplit, int P,
                                                int ns, int ppad, const double* __restrict__ E,
                                                const T* __restrict__ At, int K2,
                                                T* __restrict__ F, int bx, int by,
                                                T* __restrict__ Y) {
  typedef typename Mfma<T>::acc_t acc_t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int s0 = bx * 32, k0 = by * 64 + wave * 16;
  const int ldy = kb_small_ldy(ppad), w = min(32, ns - s0);
  // K2 is a multiple of 128: the 64 columns exist
  const T* __restrict__ arow = At + (size_t)(k0 + r16) * ppad + KPL * g;
  T b[KPL];
  load_run<T>(arow, b);  // in flight while the partials are summed
  for (int e = tid; e < w * ppad; e += 256) {
    const int p = e / w, s = e - p * w;
    double z = 0.0;
    if (p < P) {
      const double* __restrict__ zp = zpart + (size_t)p * ns + s0 + s;
#pragma unroll 4
      for (int q = 0; q < nsplit; ++q) z += zp[(size_t)q * P * ns];
      z *= -2.0 * E[p];
    }
    Y[s * ldy + p] = T(z);
  }
  __syncthreads();
  acc_t acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[i][r] = T(0);
  for (int st = 0; st < ppad / KS; ++st) {
    if (st) load_run<T>(arow + st * KS, b);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      // rows of states past the block's are never stored: their products stay
      // in their own rows, so any row of Y may stand in for them
      const T* __restrict__ y = Y + min(16 * i + r16, w - 1) * ldy + st * KS + KPL * g;
#pragma unroll
      for (int t = 0; t < KPL; ++t) acc[i] = Mfma<T>::run(y[t], b[t], acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = 16 * i + Mfma<T>::row(lane, r);
      if (s < w) F[(size_t)(s0 + s) * K2 + k0 + r16] = acc[i][r];
    }
}

}  // namespace sdft
