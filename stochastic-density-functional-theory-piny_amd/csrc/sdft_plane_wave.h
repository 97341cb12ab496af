// sdft_plane_wave.h -- the a-plane stage with every line's transform inside
// one wave.
//
// plane_body (sdft_plane.h) deals the butterflies of a group of lines to all
// threads of the workgroup, so each pass ends at a workgroup barrier: 11 per
// plane.  Here a wave owns whole lines -- L b-lines (columns) or LC c-lines
// (rows) at a time -- keeps a pass's outputs in registers and hands them to
// the next pass through its own part of LDS.  LDS operations of one wave
// complete in order, so that exchange needs no barrier; the workgroup meets
// only between the c- and b-stages (two barriers per plane).  In FP64 the
// exchange goes through 8-byte slots twice (real parts, then imaginary
// parts): half the exchange memory, and the same conflict-free pattern as the
// 8-byte complex values of FP32.
// At 64^3 (FP64, 128 pairs) the stage issues 2.94e7 vector instructions (48
// us at one per SIMD and 4 cycles) and keeps the LDS busy for 2.84e7 cycles
// over 256 CUs (46 us; bank conflicts 0.9 % of them): the two together are its
// 103 us, at the 4 workgroups of 3 waves per CU that its plane rows leave room
// for.  In FP32 2.80e7 (46 us) and 1.47e7 (24 us; none), of 60 us.
#pragma once
#include <type_traits>

#include "sdft_plane.h"

namespace sdft {

// Two-pass factorisation N = R0 R1 (the inverse transform runs R0 then R1, the
// forward one R1 then R0), waves per workgroup, b-lines and c-lines per wave
// and trip.  Two passes for every size, so one exchange per line transform.
// The splits are the fastest of those measured per size (us per launch,
// 256 orbitals at 64^3 and 48^3, 512 below, 128 / 64 at 96^3 / 128^3; FP32 /
// FP64, in brackets the workgroup-wide stage of sdft_plane.h):
//   24  14.5 /  23.2 (18.5 /  34.3)     64   60.3 / 103 (66.3 / 139)
//   32  20.5 /  34.3 (23.8 /  42.2)     96  168   / 352 (184  / 377)
//   36  36.0 /  59.4 (51.4 /  78.5)    128  258   / 410 (280  / 621)
//   48  38.7 /  63.0 (53.5 /  80.3)
// Few waves with full lanes win: at 36, 9 c-rows per wave (54 of 64 lanes) on 2
// waves 59.4 us, 5 rows on 4 waves 72.4 us; at 24 and 32 one wave per plane.
template <int N> struct WaveCfg;
template <> struct WaveCfg<24> { static constexpr int R0 = 4, R1 = 6, NW = 1, L = 8, LC = 11; };
template <> struct WaveCfg<32> { static constexpr int R0 = 8, R1 = 4, NW = 1, L = 16, LC = 16; };
template <> struct WaveCfg<36> { static constexpr int R0 = 6, R1 = 6, NW = 2, L = 9, LC = 9; };
template <> struct WaveCfg<48> { static constexpr int R0 = 8, R1 = 6, NW = 3, L = 8, LC = 8; };
template <> struct WaveCfg<64> { static constexpr int R0 = 8, R1 = 8, NW = 3, L = 8, LC = 8; };
template <> struct WaveCfg<96> { static constexpr int R0 = 8, R1 = 12, NW = 4, L = 8, LC = 9; };
template <> struct WaveCfg<128> { static constexpr int R0 = 8, R1 = 16, NW = 8, L = 4, LC = 6; };

// ---- small DFTs beyond radix 8 (fft_lds.h) --------------------------------
// Input r of a first pass lies in [N/4, 3N/4), where the sphere's spectrum is
// zero, for all of its butterflies (and output r of a last forward pass).
template <int R>
SDFT_HD constexpr bool wmid(int r) {
  return 4 * r >= R && 4 * (r + 1) <= 3 * R;
}

template <typename T, int R, int DIR>
struct WDft {
  SDFT_HD static inline void run(Cx<T>* v) { Dft<T, R, DIR>::run(v); }
  SDFT_HD static inline void run_zin(Cx<T>* v) { Dft<T, R, DIR>::run_zin(v); }
};

// 6 = 2 x 3 without twiddles: inputs n = 3 n1 + 2 n2, outputs k = 3 k1 + 4 k2
// (mod 6)
template <typename T, int DIR>
struct WDft<T, 6, DIR> {
  SDFT_HD static inline void tail(Cx<T>* v, Cx<T>* s, Cx<T>* d) {
    Dft<T, 3, DIR>::run(s);
    Dft<T, 3, DIR>::run(d);
    v[0] = s[0];
    v[4] = s[1];
    v[2] = s[2];
    v[3] = d[0];
    v[1] = d[1];
    v[5] = d[2];
  }
  SDFT_HD static inline void run(Cx<T>* v) {
    Cx<T> s[3] = {v[0] + v[3], v[2] + v[5], v[4] + v[1]};
    Cx<T> d[3] = {v[0] - v[3], v[2] - v[5], v[4] - v[1]};
    tail(v, s, d);
  }
  // v[2] = v[3] = 0 (not read)
  SDFT_HD static inline void run_zin(Cx<T>* v) {
    Cx<T> s[3] = {v[0], v[5], v[4] + v[1]};
    Cx<T> d[3] = {v[0], cx(-v[5].x, -v[5].y), v[4] - v[1]};
    tail(v, s, d);
  }
};

// 12 = 3 x 4 without twiddles: inputs n = 4 n1 + 3 n2, outputs k = 4 k1 + 9 k2
// (mod 12), n1, k1 < 3, n2, k2 < 4
template <typename T, int DIR>
struct WDft<T, 12, DIR> {
  SDFT_HD static inline void run(Cx<T>* v) {
    Cx<T> t[3][4];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
      for (int b = 0; b < 4; ++b) t[a][b] = v[(4 * a + 3 * b) % 12];
      Dft<T, 4, DIR>::run(t[a]);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      Cx<T> u[3] = {t[0][b], t[1][b], t[2][b]};
      Dft<T, 3, DIR>::run(u);
#pragma unroll
      for (int a = 0; a < 3; ++a) v[(4 * a + 9 * b) % 12] = u[a];
    }
  }
};

// 16 = 4 x 4 with twiddles: inputs n = n1 + 4 n2, outputs k = 4 k1 + k2
template <typename T, int DIR>
struct WDft<T, 16, DIR> {
  SDFT_HD static inline void run(Cx<T>* v) {
    const T c1 = T(0.92387953251128675613), s1 = T(0.38268343236508977173);
    const T h = T(0.70710678118654752440);
    Cx<T> t[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int b = 0; b < 4; ++b) t[a][b] = v[a + 4 * b];
      Dft<T, 4, DIR>::run(t[a]);
    }
    auto w = [](Cx<T> x, T c, T s) {
      return cx(c * x.x - T(DIR) * s * x.y, c * x.y + T(DIR) * s * x.x);
    };
    t[1][1] = w(t[1][1], c1, s1);
    t[1][2] = w(t[1][2], h, h);
    t[1][3] = w(t[1][3], s1, c1);
    t[2][1] = w(t[2][1], h, h);
    t[2][2] = mul_di<T, DIR>(t[2][2]);
    t[2][3] = w(t[2][3], -h, h);
    t[3][1] = w(t[3][1], s1, c1);
    t[3][2] = w(t[3][2], -h, h);
    t[3][3] = w(t[3][3], -c1, -s1);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      Cx<T> u[4] = {t[0][b], t[1][b], t[2][b], t[3][b]};
      Dft<T, 4, DIR>::run(u);
#pragma unroll
      for (int a = 0; a < 4; ++a) v[4 * a + b] = u[a];
    }
  }
};

// One pass over LN lines in one wave.  SECOND: the second pass of its
// transform, REV: the forward transform.  Radix R, NB butterflies per line,
// butterfly j's inputs at j + r NB; its outputs at j R + r (first pass) or j +
// r NB (second, after the twiddle e^{+-2 pi i r j / N}).  LINE_FAST:
// consecutive lanes on consecutive lines.
template <int N, bool SECOND, bool REV, int LN, bool LINE_FAST>
struct WPass {
  using C = WaveCfg<N>;
  static constexpr int R = SECOND != REV ? C::R1 : C::R0, NB = N / R;
  static constexpr int TOT = LN * NB, MAXB = (TOT + 63) / 64;
  SDFT_DEVI static bool live(int idx) { return TOT % 64 == 0 || idx < TOT; }
  SDFT_DEVI static int line(int idx) { return LINE_FAST ? idx % LN : idx / NB; }
  SDFT_DEVI static int bfly(int idx) { return LINE_FAST ? idx / LN : idx % NB; }
};

template <typename T, int N>
struct WPlane {
  using C = WaveCfg<N>;
  static constexpr int NW = C::NW, L = C::L, LC = C::LC, NT = 64 * NW;
  static constexpr int LDP = N + (24 - N % 16) % 16;  // plane rows: 8 mod 16
  // Exchange between two passes: element j R + r of a line (R the radix of
  // the writing pass) in slot j S + r, S = R or R + 1, odd.  The reading pass
  // takes element j + r R from slot r S + j.
  // Measured bank rules: 8-byte writes and paired reads (ds_read2_b64) of 16
  // consecutive lanes must fall on distinct slots modulo 16 (single 8-byte
  // reads: 32 lanes modulo 32; 16-byte writes / reads: 8 / 16 lanes modulo 8 /
  // 16 elements).  With S odd and b-lines 2 mod 4 slots apart, 8 of them on
  // neighbouring lanes, both sides obey them; so do c-lines of 64 points 8
  // mod 16 slots apart and plane rows 8 mod 16 elements apart.
  static constexpr int S0 = C::R0 | 1, S1 = C::R1 | 1;
  static constexpr int SLOTS = (N / C::R0) * S0 > (N / C::R1) * S1 ? (N / C::R0) * S0
                                                                   : (N / C::R1) * S1;
  static constexpr int LDB = SLOTS + (6 - SLOTS % 4) % 4;
  static constexpr int LDC = SLOTS + (24 - SLOTS % 16) % 16;
  static constexpr int QW = L * LDB > LC * LDC ? L * LDB : LC * LDC;  // 8-byte slots per wave
};

template <typename T, int N>
size_t wplane_lds_bytes(int M) {
  using S = WPlane<T, N>;
  return sizeof(Cx<T>) * (size_t)M * S::LDP + (size_t)8 * S::NW * S::QW;
}

// orders this wave's LDS accesses for the compiler (the hardware runs them
// in order)
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Twiddles of a second pass: a lane's butterflies are the same for every
// group of lines, so their factors stay in registers (read from LDS they were
// a third of the LDS cycles).
template <typename T, class W>
struct WTwiddle {
  Cx<T> w[W::MAXB][W::R];
  SDFT_DEVI void load(const Cx<T>* __restrict__ tw, int lane) {
#pragma unroll
    for (int b = 0; b < W::MAXB; ++b) {
      const int idx = lane + 64 * b;
      const int j = W::live(idx) ? W::bfly(idx) : 0;
#pragma unroll
      for (int r = 1; r < W::R; ++r) w[b][r] = tw[mul24(r, j)];
    }
  }
};

template <typename T, class W, int DIR>
SDFT_DEVI void wsecond(const WTwiddle<T, W>& t, Cx<T> (&v)[W::MAXB][W::R]) {
#pragma unroll
  for (int b = 0; b < W::MAXB; ++b) {
#pragma unroll
    for (int r = 1; r < W::R; ++r)
      v[b][r] = DIR > 0 ? cmul(v[b][r], t.w[b][r]) : cmulc(v[b][r], t.w[b][r]);
    WDft<T, W::R, DIR>::run(v[b]);
  }
}

template <typename T, class W, int DIR, bool ZIN>
SDFT_DEVI void wfirst(Cx<T> (&v)[W::MAXB][W::R]) {
#pragma unroll
  for (int b = 0; b < W::MAXB; ++b) {
    if constexpr (ZIN)
      WDft<T, W::R, DIR>::run_zin(v[b]);
    else
      WDft<T, W::R, DIR>::run(v[b]);
  }
}

// outputs of pass A (registers) -> inputs of pass B (registers)
template <typename T, class A, class B, int LDQ>
SDFT_DEVI void wexchange(void* qv, int lane, const Cx<T> (&v)[A::MAXB][A::R],
                         Cx<T> (&u)[B::MAXB][B::R]) {
  using E = typename std::conditional<sizeof(T) == 8, T, Cx<T>>::type;
  E* q = reinterpret_cast<E*>(qv);
  constexpr int PH = sizeof(T) == 8 ? 2 : 1, S = A::R | 1;
  static_assert(B::NB == A::R, "two-pass exchange");
#pragma unroll
  for (int ph = 0; ph < PH; ++ph) {
    wave_order();
#pragma unroll
    for (int b = 0; b < A::MAXB; ++b) {
      const int idx = lane + 64 * b;
      if (A::live(idx)) {
        E* dst = q + mul24(A::line(idx), LDQ) + mul24(A::bfly(idx), S);
#pragma unroll
        for (int r = 0; r < A::R; ++r) {
          if constexpr (PH == 1)
            dst[r] = v[b][r];
          else
            dst[r] = ph == 0 ? v[b][r].x : v[b][r].y;
        }
      }
    }
    wave_order();
#pragma unroll
    for (int b = 0; b < B::MAXB; ++b) {
      const int idx = lane + 64 * b;
      if (B::live(idx)) {
        const E* src = q + mul24(B::line(idx), LDQ) + B::bfly(idx);
#pragma unroll
        for (int r = 0; r < B::R; ++r) {
          if constexpr (PH == 1)
            u[b][r] = src[r * S];
          else if (ph == 0)
            u[b][r].x = src[r * S];
          else
            u[b][r].y = src[r * S];
        }
      }
    }
  }
}

// MODE as in plane_body.  Spheres inside |k| < n/4 only (pruned first and
// last passes).
template <typename T, int N, int MODE>
__device__ __forceinline__ void wplane_body(const PlaneArgs& a, int ra, int q) {
  using S = WPlane<T, N>;
  constexpr int NW = S::NW, L = S::L, LC = S::LC, LDP = S::LDP;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int ncolp = a.ncolp, M = a.M, K = (M - 1) / 2;
  const int* __restrict__ rowcol = a.rowcol;
  Cx<T>* Pl = reinterpret_cast<Cx<T>*>(smem_raw);  // M rows, stride LDP
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* Q = reinterpret_cast<double*>(Pl + M * LDP) + wave * S::QW;
  const Cx<T>* __restrict__ tw = reinterpret_cast<const Cx<T>*>(a.tw);
  Cx<T>* Wp = reinterpret_cast<Cx<T>*>(a.W) + ((size_t)q * N + ra) * ncolp;
  Cx<T>* __restrict__ F = reinterpret_cast<Cx<T>*>(a.field) + ((size_t)q * N + ra) * N * N;

  // inverse along c: W -> rows of the plane
  if constexpr (MODE != 2) {
    using A = WPass<N, false, false, LC, false>;
    using B = WPass<N, true, false, LC, false>;
    WTwiddle<T, B> tl;
    tl.load(tw, lane);
    for (int r0 = wave * LC; r0 < M; r0 += NW * LC) {
      Cx<T> v[A::MAXB][A::R], u[B::MAXB][B::R];
#pragma unroll
      for (int b = 0; b < A::MAXB; ++b) {
        const int idx = lane + 64 * b;
        const int row = r0 + A::line(idx);
        const int* rc = rowcol + mul24(row < M ? row : M - 1, N) + A::bfly(idx);
#pragma unroll
        for (int r = 0; r < A::R; ++r)
          if (!wmid<A::R>(r)) {
            const int d = rc[r * A::NB];
            const Cx<T> x = Wp[d >= 0 ? d : 0];
            const T m = d >= 0 ? T(1) : T(0);
            v[b][r] = cx(x.x * m, x.y * m);
          }
      }
      wfirst<T, A, +1, true>(v);
      wexchange<T, A, B, S::LDC>(Q, lane, v, u);
      wsecond<T, B, +1>(tl, u);
#pragma unroll
      for (int b = 0; b < B::MAXB; ++b) {
        const int idx = lane + 64 * b;
        const int row = r0 + B::line(idx);
        if (B::live(idx) && row < M) {
          Cx<T>* dst = Pl + mul24(row, LDP) + B::bfly(idx);
#pragma unroll
          for (int r = 0; r < B::R; ++r) dst[r * B::NB] = u[b][r];
        }
      }
    }
    __syncthreads();
  }

  // along b: columns c0 .. c0 + L - 1 of this wave
  {
    using A = WPass<N, false, false, L, true>;
    using B = WPass<N, true, false, L, true>;
    using FA = WPass<N, false, true, L, true>;  // B's butterflies
    using FB = WPass<N, true, true, L, true>;
    static_assert(N % L == 0, "whole groups of b-lines");
    WTwiddle<T, B> ti;
    WTwiddle<T, FB> tf;
    if constexpr (MODE != 2) ti.load(tw, lane);
    if constexpr (MODE == 0 || MODE == 2) tf.load(tw, lane);
    const T* vplane = reinterpret_cast<const T*>(a.v) + (size_t)ra * N * N;
    const unsigned short* skip = a.skip + (MODE == 3 ? ra * (N / 16) : 0);
    for (int c0 = wave * L; c0 < N; c0 += NW * L) {
      Cx<T> u[B::MAXB][B::R];
      if constexpr (MODE == 2) {
#pragma unroll
        for (int b = 0; b < B::MAXB; ++b) {
          const int ii = B::live(lane + 64 * b) ? lane + 64 * b : 0;
          const Cx<T>* src = F + (size_t)B::bfly(ii) * N + c0 + B::line(ii);
#pragma unroll
          for (int r = 0; r < B::R; ++r) u[b][r] = src[(size_t)r * B::NB * N];
        }
      } else {
        // v_KS of this lane's points, in flight during the transform
        T sv[B::MAXB][B::R];
        if constexpr (MODE == 0 || MODE == 3) {
#pragma unroll
          for (int b = 0; b < B::MAXB; ++b) {
            const int ii = B::live(lane + 64 * b) ? lane + 64 * b : 0;
            const T* src = vplane + mul24(B::bfly(ii), N) + c0 + B::line(ii);
#pragma unroll
            for (int r = 0; r < B::R; ++r) sv[b][r] = src[r * B::NB * N];
          }
        }
        Cx<T> v[A::MAXB][A::R];
#pragma unroll
        for (int b = 0; b < A::MAXB; ++b) {
          const int ii = A::live(lane + 64 * b) ? lane + 64 * b : 0;
          const int c = c0 + A::line(ii), j = A::bfly(ii);
#pragma unroll
          for (int r = 0; r < A::R; ++r)
            if (!wmid<A::R>(r)) {
              const int pos = j + r * A::NB;
              const int kb = pos <= N / 2 ? pos : pos - N;
              const bool in = kb >= -K && kb <= K;
              const Cx<T> x = Pl[mul24(in ? kb + K : 0, LDP) + c];
              v[b][r] = cx(in ? x.x : T(0), in ? x.y : T(0));
            }
        }
        wfirst<T, A, +1, true>(v);
        wexchange<T, A, B, S::LDB>(Q, lane, v, u);
        wsecond<T, B, +1>(ti, u);
        if constexpr (MODE == 1 || MODE == 3) {
#pragma unroll
          for (int b = 0; b < B::MAXB; ++b) {
            const int idx = lane + 64 * b;
            if (B::live(idx)) {
              if constexpr (MODE == 3) {  // v_KS where its tile is marked (plane_body)
                const int marks = skip[(c0 + B::line(idx)) >> 4];
#pragma unroll
                for (int r = 0; r < B::R; ++r) {
                  const int rb = B::bfly(idx) + r * B::NB;
                  const T m = (marks >> (rb >> 4)) & 1 ? sv[b][r] : T(1);
                  u[b][r] = cx(m * u[b][r].x, m * u[b][r].y);
                }
              }
              Cx<T>* dst = F + (size_t)B::bfly(idx) * N + c0 + B::line(idx);
#pragma unroll
              for (int r = 0; r < B::R; ++r) dst[(size_t)r * B::NB * N] = u[b][r];
            }
          }
        } else {
#pragma unroll
          for (int b = 0; b < B::MAXB; ++b)
#pragma unroll
            for (int r = 0; r < B::R; ++r)
              u[b][r] = cx(u[b][r].x * sv[b][r], u[b][r].y * sv[b][r]);
        }
      }
      if constexpr (MODE == 0 || MODE == 2) {
        Cx<T> w[FB::MAXB][FB::R];
        wfirst<T, FA, -1, false>(u);
        wexchange<T, FA, FB, S::LDB>(Q, lane, u, w);
        wsecond<T, FB, -1>(tf, w);
#pragma unroll
        for (int b = 0; b < FB::MAXB; ++b) {
          const int idx = lane + 64 * b;
          if (FB::live(idx)) {
            const int c = c0 + FB::line(idx), j = FB::bfly(idx);
#pragma unroll
            for (int r = 0; r < FB::R; ++r)
              if (!wmid<FB::R>(r)) {
                const int pos = j + r * FB::NB;
                const int kb = pos <= N / 2 ? pos : pos - N;
                if (kb >= -K && kb <= K) Pl[mul24(kb + K, LDP) + c] = w[b][r];
              }
          }
        }
      }
    }
  }

  // forward along c: rows of the plane -> W
  if constexpr (MODE == 0 || MODE == 2) {
    __syncthreads();
    using A = WPass<N, false, true, LC, false>;
    using B = WPass<N, true, true, LC, false>;
    WTwiddle<T, B> tl;
    tl.load(tw, lane);
    for (int r0 = wave * LC; r0 < M; r0 += NW * LC) {
      Cx<T> v[A::MAXB][A::R], u[B::MAXB][B::R];
#pragma unroll
      for (int b = 0; b < A::MAXB; ++b) {
        const int idx = lane + 64 * b;
        const int row = r0 + A::line(idx);
        const Cx<T>* src = Pl + mul24(row < M ? row : M - 1, LDP) + A::bfly(idx);
#pragma unroll
        for (int r = 0; r < A::R; ++r) v[b][r] = src[r * A::NB];
      }
      wfirst<T, A, -1, false>(v);
      wexchange<T, A, B, S::LDC>(Q, lane, v, u);
      wsecond<T, B, -1>(tl, u);
#pragma unroll
      for (int b = 0; b < B::MAXB; ++b) {
        const int idx = lane + 64 * b;
        const int row = r0 + B::line(idx);
        if (B::live(idx) && row < M) {
          const int j = B::bfly(idx);
          const int* rc = rowcol + mul24(row, N) + j;
#pragma unroll
          for (int r = 0; r < B::R; ++r)
            if (!wmid<B::R>(r)) {
              const int d = rc[r * B::NB];
              if (d >= 0) Wp[d] = u[b][r];
            }
        }
      }
    }
  }
}

#define SDFT_WPLANE_SWITCH(n, ...)                                  \
  switch (n) {                                                      \
    case 24: { constexpr int NN = 24; __VA_ARGS__; } break;         \
    case 32: { constexpr int NN = 32; __VA_ARGS__; } break;         \
    case 36: { constexpr int NN = 36; __VA_ARGS__; } break;         \
    case 48: { constexpr int NN = 48; __VA_ARGS__; } break;         \
    case 64: { constexpr int NN = 64; __VA_ARGS__; } break;         \
    case 96: { constexpr int NN = 96; __VA_ARGS__; } break;         \
    case 128: { constexpr int NN = 128; __VA_ARGS__; } break;       \
    default: set_error("unsupported grid size"); return SDFT_EINVAL_CODE; \
  }

}  // namespace sdft
