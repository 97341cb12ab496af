// sdft_cheby.hip -- FP64 scalar side of the Chebyshev path, on the device.
//
//  * expansion coefficients of f_FD or sqrt(f_FD) (calcChebyCoeff,
//    stodft/coeff.c:1093-1223): c_k = (2/M) sum_j g(x_j) cos(2 pi jk/M),
//    c_0 = (1/M) sum_j g(x_j), x_j = (dE/2) cos(2 pi j/M) + E_mean,
//    M = roundFFT(32 L) (coeff.c:1556-1600).  The reference takes the real
//    part of an M-point complex DFT; here the L kept outputs come from a
//    two-step decimated DFT (k_dft_inner, k_dft_outer).
//  * electron count and chemical potential (calcNumElecCheby /
//    calcChemPotCheby, stodft/calc-chempot-chebyshev.c:30-315,918-972):
//    N(mu) = occ sum_{k<L} c_k(mu) m_k = (occ/M) sum_j f(x_j; mu) h_j with
//    h_j = m_0 + 2 sum_{k=1}^{L-1} m_k cos(2 pi jk/M) computed once (the same
//    two-step DFT; x_j and h_j are even in j, so only j <= M/2 is kept), so
//    each N(mu) is one reduction over M/2 points; the bracket /
//    interpolation / bisection sequence of the reference runs as rounds that
//    evaluate all mu values the sequence can reach in its next steps.
//  * per-step moment partial reduction and the kinetic / nonlocal energy
//    sums (stodft/calc-energy.c:133-191).
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/sdft_hip.h"
#include "sdft_internal.h"

namespace sdft {

int round_fft(int n_in);

__device__ inline double fermi_dev(double x, double mu, double beta) {
  return 1.0 / (1.0 + exp(beta * (x - mu)));
}

// tw[m] = exp(+2 pi i m / M)
__global__ void k_unit_roots(double2* __restrict__ tw, int M) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < M) {
    double sn, cs;
    sincospi(2.0 * (double)j / (double)M, &sn, &cs);
    tw[j] = make_double2(cs, sn);
  }
}

__global__ void k_cheby_fvals(const double2* __restrict__ tw, int M, double dE, double em,
                              double mu, double beta, int fun_flag, double* __restrict__ g) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= M) return;
  const double x = dE * tw[j].x + em;
  double f = fermi_dev(x, mu, beta);
  if (fun_flag == 2) f = sqrt(f);
  g[j] = f;
}

// X_k = Re sum_{j<nx} w_j x_j e^{2 pi i jk/M} in two steps with M = P Q, j =
// j1 + P j2:
//   A[j1][k'] = sum_{j2} w_j x_j e^{2 pi i j2 k'/Q}   (k' < Q)
//   X_k       = Re sum_{j1<P} A[j1][k mod Q] e^{2 pi i j1 k/M}
// nx/P + P terms per output instead of nx.  One sum per output over the whole
// table took 200 us (h_j) and 150 us (the coefficients) at L = 1024 (M =
// 34992); the two steps take 18 and 27 us.
// twice: w_j = 2 for j > 0 (the moments), else 1.
__global__ __launch_bounds__(256) void k_dft_inner(const double* __restrict__ x, int nx, int twice,
                                                   const double2* __restrict__ tw, int P, int Q,
                                                   double2* __restrict__ A) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  const int j1 = t / Q, k = t - j1 * Q;
  if (j1 >= P) return;
  double re = 0.0, im = 0.0;
  int i = 0;
#pragma unroll 4
  for (int j = j1; j < nx; j += P) {
    const double xv = (twice && j > 0) ? 2.0 * x[j] : x[j];
    const double2 w = tw[(size_t)P * i];
    re += xv * w.x;
    im += xv * w.y;
    i += k;
    if (i >= Q) i -= Q;
  }
  A[t] = make_double2(re, im);
}

// 16 outputs per workgroup, their terms j1 dealt to 64 threads each (the
// gathers of tw are all cache misses: few of them in a row per thread).
// out[k] = a1 X_k, or a0 X_k at k = 0 and (ends) at 2 k = M.
__global__ __launch_bounds__(1024) void k_dft_outer(const double2* __restrict__ A, int P, int Q,
                                                    const double2* __restrict__ tw, int M,
                                                    int nout, double a0, double a1, int ends,
                                                    double* __restrict__ out) {
  __shared__ double sh[64][17];
  const int o = threadIdx.x & 15, grp = threadIdx.x >> 4;
  const int k = blockIdx.x * 16 + o;
  double s = 0.0;
  if (k < nout) {
    const int kq = k % Q;
    int i = (int)((long long)grp * k % M);
    const int step = (int)(64LL * k % M);
#pragma unroll 4
    for (int j1 = grp; j1 < P; j1 += 64) {
      const double2 a = A[(size_t)j1 * Q + kq];
      const double2 w = tw[i];
      s += a.x * w.x - a.y * w.y;
      i += step;
      if (i >= M) i -= M;
    }
  }
  sh[grp][o] = s;
  __syncthreads();
  if (grp < 4) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) t += sh[grp * 16 + w][o];
    t += __shfl_xor(t, 16, 64);
    t += __shfl_xor(t, 32, 64);
    if (grp == 0 && k < nout)
      out[k] = t * ((k == 0 || (ends && 2 * (long long)k == M)) ? a0 : a1);
  }
}

__device__ inline double block_sum(double v, double* sh) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  double s = 0.0;
  const int nw = blockDim.x >> 6;
  for (int w = 0; w < nw; ++w) s += sh[w];
  return s;
}

// ---- chemical potential: bracket, interpolation, bisection ------------------
// The search's state between rounds.  phase 0: (lo, hi) is a bracket to be
// evaluated; phase 1: mu is the next trial point of the bisection between lo
// and hi; phase 2: done.
struct MuState {
  double lo, hi, mu, nn;
  int phase, it, ib;
};

constexpr int kMuDepth = 5;                    // bisection steps per round
constexpr int kMuCand = (1 << kMuDepth) - 1;   // trial points per round
constexpr int kMuSlices = 8;                   // workgroups per trial point
constexpr int kMuUp = 16;                      // phase 0: last candidate upwards

// Trial point c of a round from state s.  Phase 0: 0 = lo, 1 = hi, then hi
// widened upwards (2 .. kMuUp) and lo widened downwards, each by repeated
// addition as the reference steps.  Phase 1: node c + 1 of the bisection
// tree whose root is mu (a right child where N(mu) fell short).
__device__ inline double mu_candidate(const MuState& s, int c, double gap) {
  if (s.phase == 0) {
    if (c == 0) return s.lo;
    double m = s.hi;
    if (c <= kMuUp) {
      for (int i = 1; i < c; ++i) m += gap;
      return m;
    }
    m = s.lo;
    for (int i = kMuUp; i < c; ++i) m -= gap;
    return m;
  }
  double lo = s.lo, hi = s.hi, mu = s.mu;
  const int node = c + 1;
  for (int b = 30 - __clz(node); b >= 0; --b) {
    if ((node >> b) & 1)
      lo = mu;
    else
      hi = mu;
    mu = 0.5 * (lo + hi);
  }
  return mu;
}

// The sequence of calcChemPotCheby continued with the N values of a round's
// trial points, until it needs a point the round did not evaluate.
__device__ inline void mu_advance(MuState& s, const double* N, double gap, double ne, double tol,
                                  int max_iter) {
  if (s.phase == 0) {
    double nlo = N[0], nhi = N[1];
    int up = 1, down = kMuUp;
    while (nhi < ne && s.it < max_iter) {
      s.lo = s.hi;
      s.hi += gap;
      ++s.it;
      if (++up > kMuUp) return;
      nlo = nhi;
      nhi = N[up];
    }
    while (nlo > ne && s.it < max_iter) {
      s.hi = s.lo;
      s.lo -= gap;
      ++s.it;
      if (++down >= kMuCand) return;
      nhi = nlo;
      nlo = N[down];
    }
    s.mu = (ne - nlo) * (s.hi - s.lo) / (nhi - nlo) + s.lo;
    s.phase = 1;
    return;
  }
  for (int node = 1; node <= kMuCand;) {
    s.nn = N[node - 1];
    if (!(fabs(s.nn - ne) > tol) || s.ib >= max_iter) {
      s.phase = 2;
      return;
    }
    int right = 0;
    if (s.nn > ne) s.hi = s.mu;
    if (s.nn < ne) {
      s.lo = s.mu;
      right = 1;
    }
    s.mu = 0.5 * (s.lo + s.hi);
    ++s.ib;
    node = 2 * node + right;
  }
}

// One round: every workgroup continues the sequence with the previous
// round's partial sums (all of them the same way), then sums its slice of
// its trial point's N.  st[0/1] and part[0/1] alternate between rounds, so a
// round reads what the previous launch wrote and writes the other half.  A
// search that took one workgroup 35 dependent reductions (546 us at L =
// 1024) takes 8 rounds of about 5 us.
__global__ __launch_bounds__(256) void k_mu_round(const double2* __restrict__ tw,
                                                  const double* __restrict__ h, int npt, int M,
                                                  double dE, double em, double beta, double occ,
                                                  double ne, double gap, double tol, int max_iter,
                                                  int round, MuState s0, MuState* __restrict__ st,
                                                  double* __restrict__ part) {
  __shared__ double N[kMuCand + 1];
  __shared__ MuState sh_s;
  __shared__ double sh_mu;
  __shared__ double sh[4];
  const int c = blockIdx.x % kMuCand, slice = blockIdx.x / kMuCand;
  const int cur = round & 1;
  const double* pin = part + cur * kMuCand * kMuSlices;
  double* pout = part + (1 - cur) * kMuCand * kMuSlices;
  if (round > 0 && threadIdx.x < kMuCand) {
    double v = 0.0;
    for (int i = 0; i < kMuSlices; ++i) v += pin[i * kMuCand + threadIdx.x];
    N[threadIdx.x] = occ * v / (double)M;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    MuState s = round > 0 ? st[cur] : s0;
    if (round > 0 && s.phase < 2) mu_advance(s, N, gap, ne, tol, max_iter);
    if (blockIdx.x == 0) st[1 - cur] = s;
    sh_s = s;
    if (s.phase < 2) sh_mu = mu_candidate(s, c, gap);
  }
  __syncthreads();
  if (sh_s.phase == 2) return;
  const double mu = sh_mu;
  double v = 0.0;
  for (int j = slice * 256 + threadIdx.x; j < npt; j += kMuSlices * 256)
    v += fermi_dev(dE * tw[j].x + em, mu, beta) * h[j];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) pout[slice * kMuCand + c] = sh[0] + sh[1] + sh[2] + sh[3];
}

// out[step*3 + i] = sum_w part[(step*nwg + w)*3 + i]
__global__ void k_mom_reduce(const double* __restrict__ part, int nwg, double* __restrict__ out) {
  __shared__ double sh[16];
  const int step = blockIdx.x;
  for (int i = 0; i < 3; ++i) {
    double s = 0.0;
    for (int w = threadIdx.x; w < nwg; w += blockDim.x) s += part[((size_t)step * nwg + w) * 3 + i];
    s = block_sum(s, sh);
    if (threadIdx.x == 0) out[step * 3 + i] = s;
  }
}

// per state: sum_{j < ncoef-1} 2 ak2 (re^2 + im^2)
__global__ void k_eke(const double* __restrict__ X, int ldx, int ncp, int ncoef,
                      const double* __restrict__ ak2, double* __restrict__ out) {
  __shared__ double sh[16];
  const int s = blockIdx.x;
  const double* x = X + (size_t)s * ldx;
  double acc = 0.0;
  for (int j = threadIdx.x; j < ncoef - 1; j += blockDim.x)
    acc += 2.0 * ak2[j] * (x[j] * x[j] + x[ncp + j] * x[ncp + j]);
  acc = block_sum(acc, sh);
  if (threadIdx.x == 0) out[s] = acc;
}

// sum_{p, s < nstate} E_p Z[p][s]^2
__global__ void k_enl(const double* __restrict__ Z, const double* __restrict__ E, int P, int ns,
                      int nstate, double* __restrict__ out) {
  __shared__ double sh[16];
  double acc = 0.0;
  for (int i = threadIdx.x; i < P * ns; i += blockDim.x) {
    const int p = i / ns, s = i - p * ns;
    if (s < nstate) acc += E[p] * Z[i] * Z[i];
  }
  acc = block_sum(acc, sh);
  if (threadIdx.x == 0) out[0] = acc;
}

// One power-iteration update of genEnergyMax / genEnergyMin
// (stodft/calc-spectral-range.c:180-221 / :380-420) on orbital 0 of X with
// raw force F: h = -f/4 (G != 0), -f/2 (G = 0); E = 2 sum_{G!=0} (h.re v.re +
// h.im v.im) + h.re(0) v.re(0); w = h (mode 0) or emax v - h (mode 1);
// v = w / sqrt(2 sum_{G!=0} |w|^2 + w.re(0)^2).  One workgroup.
// The loop's state lives here, so that the next iteration is in the queue
// before the host has seen this one: st = {E of the iteration before, E,
// iterations}; an update after |st[0] - st[1]| <= conv changes nothing.
// `seen` (pinned host memory) receives a copy of st.
__global__ void k_power_update(double* __restrict__ X, const double* __restrict__ F, int ncp,
                               int ncoef, int mode, double emax, double conv,
                               double* __restrict__ st, double* __restrict__ seen) {
  __shared__ double sh[16];
  __shared__ double len_sh;
  const double e1 = st[1];
  if (!(fabs(st[0] - e1) > conv)) {
    if (threadIdx.x < 3) seen[threadIdx.x] = st[threadIdx.x];
    return;
  }
  double e = 0.0, l2 = 0.0;
  const int g0 = ncoef - 1;
  for (int j = threadIdx.x; j < ncoef; j += blockDim.x) {
    const double s = (j == g0) ? -0.5 : -0.25;
    const double hr = s * F[j], hi = s * F[ncp + j];
    const double vr = X[j], vi = X[ncp + j];
    const double wr = mode ? emax * vr - hr : hr;
    const double wi = mode ? emax * vi - hi : hi;
    if (j == g0) {
      e += hr * vr;
      l2 += wr * wr;
    } else {
      e += 2.0 * (hr * vr + hi * vi);
      l2 += 2.0 * (wr * wr + wi * wi);
    }
    X[j] = wr;
    X[ncp + j] = wi;
  }
  e = block_sum(e, sh);
  l2 = block_sum(l2, sh);
  if (threadIdx.x == 0) {
    seen[0] = st[0] = e1;
    seen[1] = st[1] = e;
    seen[2] = st[2] = st[2] + 1.0;
    len_sh = sqrt(l2);
  }
  __syncthreads();
  const double inv = 1.0 / len_sh;
  for (int j = threadIdx.x; j < ncoef; j += blockDim.x) {
    X[j] *= inv;
    X[ncp + j] *= inv;
  }
}

// v /= sqrt(<v|v>) (Gamma norm) for orbital 0 of X; the power iteration's state
// starts from energyOld = 1e7, energy = 1e5 (calc-spectral-range.c:168-170)
__global__ void k_normalize0(double* __restrict__ X, int ncp, int ncoef, double* __restrict__ st) {
  __shared__ double sh[16];
  __shared__ double len_sh;
  double l2 = 0.0;
  for (int j = threadIdx.x; j < ncoef; j += blockDim.x)
    l2 += (j == ncoef - 1) ? X[j] * X[j] : 2.0 * (X[j] * X[j] + X[ncp + j] * X[ncp + j]);
  l2 = block_sum(l2, sh);
  if (threadIdx.x == 0) {
    len_sh = sqrt(l2);
    st[0] = 1.0e7;
    st[1] = 1.0e5;
    st[2] = 0.0;
  }
  __syncthreads();
  const double inv = 1.0 / len_sh;
  for (int j = threadIdx.x; j < ncoef; j += blockDim.x) {
    X[j] *= inv;
    X[ncp + j] *= inv;
  }
}

// ==========================================================================

static int ensure_red(Ctx& c, size_t need) {
  if (c.red_bytes >= need) return 0;
  if (c.red) SDFT_HIP_CHECK(hipFree(c.red));
  c.red = nullptr;
  c.red_bytes = 0;
  if (hipMalloc(&c.red, need) != hipSuccess) {
    set_error("device allocation failed (reduction scratch)");
    return -3;
  }
  c.red_bytes = need;
  return 0;
}

// P of the two-step DFT: the divisor of M = 2^a 3^b nearest to sqrt(8 nx) from
// above (M itself if none).  A thread runs nx / P dependent terms in the first
// step and P / 64 in the second.
static int dft_split(int M, int nx) {
  int best = M;
  for (int p = 1; p <= M && p > 0; p *= 2) {
    if (M % p) break;
    for (int q = p; q <= M && q > 0 && M % q == 0; q *= 3)
      if ((long long)q * q >= 8LL * nx && q < best) best = q;
  }
  return best;
}

// X_k (k < nout) of x (nx values); A: scratch of M complex values
static void launch_dft(Ctx& c, const double* x, int nx, bool twice, const double2* tw, int M,
                       int nout, double a0, double a1, bool ends, double2* A, double* out) {
  const int P = dft_split(M, nx), Q = M / P;
  hipLaunchKernelGGL(k_dft_inner, dim3((M + 255) / 256), dim3(256), 0, c.stream, x, nx,
                     twice ? 1 : 0, tw, P, Q, A);
  hipLaunchKernelGGL(k_dft_outer, dim3((nout + 15) / 16), dim3(1024), 0, c.stream, A, P, Q, tw, M,
                     nout, a0, a1, ends ? 1 : 0, out);
}

int cheby_coeffs_device(Ctx& c, int L, double emin, double emax, double mu, double beta,
                        int fun_flag, double* coeffs_host) {
  const int M = round_fft(32 * L);
  int rc = ensure_red(c, sizeof(double) * ((size_t)5 * M + L));
  if (rc) return rc;
  double2* tw = reinterpret_cast<double2*>(c.red);
  double2* A = tw + M;
  double* g = reinterpret_cast<double*>(A + M);
  double* cdev = g + M;
  const double dE = (emax - emin) * 0.5, em = 0.5 * (emax + emin);
  const int nb = (M + 255) / 256;
  hipLaunchKernelGGL(k_unit_roots, dim3(nb), dim3(256), 0, c.stream, tw, M);
  hipLaunchKernelGGL(k_cheby_fvals, dim3(nb), dim3(256), 0, c.stream, tw, M, dE, em, mu, beta,
                     fun_flag, g);
  launch_dft(c, g, M, false, tw, M, L, 1.0 / (double)M, 2.0 / (double)M, false, A, cdev);
  SDFT_HIP_CHECK(hipGetLastError());
  SDFT_HIP_CHECK(hipMemcpyAsync(coeffs_host, cdev, sizeof(double) * L, hipMemcpyDeviceToHost,
                                c.stream));
  SDFT_HIP_CHECK(hipStreamSynchronize(c.stream));
  return 0;
}

// The chemical-potential search on a device buffer `buf` of at least
// chem_pot_scratch_doubles(L) doubles: unit roots and the DFT's inner sums (M
// complex each), h_j (j <= M/2), the raw moments (L), the rounds' partial
// sums and states.  The moments are copied in unnormalised; the 1/nsto
// factor is folded into h_j.
constexpr size_t kMuPart = (size_t)2 * kMuCand * kMuSlices;
constexpr size_t kMuStateDoubles = 2 * sizeof(MuState) / sizeof(double);
static size_t chem_pot_scratch_doubles(int L) {
  const size_t M = (size_t)round_fft(32 * L);
  return 4 * M + (M / 2 + 1) + L + kMuPart + kMuStateDoubles + 4;
}

static int chem_pot_on(Ctx& c, double* buf, int L, double emin, double emax, double beta,
                       const double* moments, double nsto, double ne_true, double mu_init,
                       double gap, double occ, double tol, double* mu_out, double* ne_out) {
  constexpr int kMaxIter = 400;
  const int M = round_fft(32 * L), npt = M / 2 + 1;
  double2* tw = reinterpret_cast<double2*>(buf);
  double2* A = tw + M;
  double* h = reinterpret_cast<double*>(A + M);
  double* m = h + npt;
  double* part = m + L;
  MuState* st = reinterpret_cast<MuState*>(part + kMuPart);
  SDFT_HIP_CHECK(hipMemcpyAsync(m, moments, sizeof(double) * L, hipMemcpyHostToDevice, c.stream));
  const int nb = (M + 255) / 256;
  hipLaunchKernelGGL(k_unit_roots, dim3(nb), dim3(256), 0, c.stream, tw, M);
  // h_j carries the count of j and M - j
  launch_dft(c, m, L, true, tw, M, npt, 1.0 / nsto, 2.0 / nsto, true, A, h);
  const double dE = (emax - emin) * 0.5, em = 0.5 * (emax + emin);
  MuState s0{};
  s0.lo = mu_init - 0.5 * gap;
  s0.hi = mu_init + 0.5 * gap;
  // rounds are queued in batches: one for the bracket, one per kMuDepth
  // bisection steps (about 35 from the interpolated point to 1e-11 N_e) and
  // one that reads the last values; a finished search makes the rest return
  // at once
  MuState s = s0;
  int round = 0;
  const int most = 2 * (kMaxIter / (kMuCand - kMuUp) + kMaxIter / kMuDepth + 8);
  while (s.phase != 2 && round < most) {
    const int batch = round == 0 ? 9 : 4;
    for (int i = 0; i < batch; ++i, ++round)
      hipLaunchKernelGGL(k_mu_round, dim3(kMuCand * kMuSlices), dim3(256), 0, c.stream, tw, h, npt,
                         M, dE, em, beta, occ, ne_true, gap, tol, kMaxIter, round, s0, st, part);
    SDFT_HIP_CHECK(hipGetLastError());
    SDFT_HIP_CHECK(hipMemcpyAsync(&s, st + (round & 1), sizeof(s), hipMemcpyDeviceToHost,
                                  c.stream));
    SDFT_HIP_CHECK(hipStreamSynchronize(c.stream));
  }
  *mu_out = s.mu;
  *ne_out = s.nn;
  return 0;
}

int chem_pot_device(Ctx& c, int L, double emin, double emax, double beta, const double* moments,
                    double nsto, double ne_true, double mu_init, double gap, double occ,
                    double tol, double* mu_out, double* ne_out) {
  int rc = ensure_red(c, sizeof(double) * chem_pot_scratch_doubles(L));
  if (rc) return rc;
  return chem_pot_on(c, c.red, L, emin, emax, beta, moments, nsto, ne_true, mu_init, gap, occ,
                     tol, mu_out, ne_out);
}

// ---- chemical-potential search without device allocation ----------------
// A fixed per-device array holds the search's scratch for every L up to
// kNoAllocMaxL: the largest roundFFT(32 L) there is 279936 (2^7 3^7), so
// 4.5 * 279936 + 8192 and the rounds' partial sums (10.2 MB).  Each device that loads the
// library holds its own copy until the process ends.  The host never uses
// the array's name as an address: at context creation the device address
// is read once per device with hipGetSymbolAddress and kept in
// g_scratch_dev[device].  Every no-allocation call on a device shares that
// device's array, so such calls that overlap on one device (two host
// threads, or two contexts' streams) race; nothing in it has to start at
// zero (every element a search reads is written first by the same call).
constexpr int kNoAllocMaxL = 8192;
constexpr size_t kNoAllocDoubles =
    (size_t)4 * 279936 + (279936 / 2 + 1) + kNoAllocMaxL + kMuPart + kMuStateDoubles + 4;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) double scratch[kNoAllocDoubles];

static std::mutex g_scratch_mu;
static double* g_scratch_dev[kMaxDevices] = {nullptr};

int noalloc_scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices) {
    set_error("device ordinal out of range for the no-allocation scratch table");
    return SDFT_EINVAL;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_dev[device]) return 0;
  void* p = nullptr;
  SDFT_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_dev[device] = static_cast<double*>(p);
  return 0;
}

int chem_pot_device_noalloc(Ctx& c, int L, double emin, double emax, double beta,
                            const double* moments, double nsto, double ne_true, double mu_init,
                            double gap, double occ, double tol, double* mu_out, double* ne_out) {
  if (L > kNoAllocMaxL || chem_pot_scratch_doubles(L) > kNoAllocDoubles) {
    set_error("sdft_hip_chem_pot_noalloc: L = " + std::to_string(L) +
              " exceeds the fixed scratch (L <= " + std::to_string(kNoAllocMaxL) + ")");
    return SDFT_EINVAL;
  }
  double* buf = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (c.device >= 0 && c.device < kMaxDevices) buf = g_scratch_dev[c.device];
  }
  if (!buf) {
    set_error("sdft_hip_chem_pot_noalloc: no scratch address for this device");
    return SDFT_ESTATE;
  }
  return chem_pot_on(c, buf, L, emin, emax, beta, moments, nsto, ne_true, mu_init, gap, occ, tol,
                     mu_out, ne_out);
}

int moments_reduce(Ctx& c, const double* mom_part, int nsteps, int nwg, double* out3) {
  int rc = ensure_red(c, sizeof(double) * (size_t)3 * nsteps);
  if (rc) return rc;
  hipLaunchKernelGGL(k_mom_reduce, dim3(nsteps), dim3(256), 0, c.stream, mom_part, nwg, c.red);
  SDFT_HIP_CHECK(hipGetLastError());
  SDFT_HIP_CHECK(hipMemcpyAsync(out3, c.red, sizeof(double) * 3 * nsteps, hipMemcpyDeviceToHost,
                                c.stream));
  SDFT_HIP_CHECK(hipStreamSynchronize(c.stream));
  return 0;
}

int energy_ke_device(Ctx& c, const double* X, int nstate, double* out) {
  int rc = ensure_red(c, sizeof(double) * (size_t)nstate);
  if (rc) return rc;
  hipLaunchKernelGGL(k_eke, dim3(nstate), dim3(256), 0, c.stream, X, 2 * c.g.ncp, c.g.ncp,
                     c.g.ncoef, c.t.ak2, c.red);
  SDFT_HIP_CHECK(hipGetLastError());
  std::vector<double> h(nstate);
  SDFT_HIP_CHECK(hipMemcpyAsync(h.data(), c.red, sizeof(double) * nstate, hipMemcpyDeviceToHost,
                                c.stream));
  SDFT_HIP_CHECK(hipStreamSynchronize(c.stream));
  double s = 0.0;
  for (int i = 0; i < nstate; ++i) s += h[i];
  *out = s;
  return 0;
}

int power_start_device(Ctx& c, double* X) {
  int rc = ensure_red(c, 3 * sizeof(double));
  if (rc) return rc;
  hipLaunchKernelGGL(k_normalize0, dim3(1), dim3(1024), 0, c.stream, X, c.g.ncp, c.g.ncoef, c.red);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

int power_update_device(Ctx& c, double* X, const double* F, int mode, double emax, double conv,
                        double* seen) {
  hipLaunchKernelGGL(k_power_update, dim3(1), dim3(1024), 0, c.stream, X, F, c.g.ncp, c.g.ncoef,
                     mode, emax, conv, c.red, seen);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

int energy_nl_device(Ctx& c, int ns, int nstate, double* out) {
  int rc = ensure_red(c, sizeof(double));
  if (rc) return rc;
  hipLaunchKernelGGL(k_enl, dim3(1), dim3(1024), 0, c.stream, c.Z, c.E, c.nproj, ns, nstate, c.red);
  SDFT_HIP_CHECK(hipGetLastError());
  SDFT_HIP_CHECK(hipMemcpyAsync(out, c.red, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  SDFT_HIP_CHECK(hipStreamSynchronize(c.stream));
  return 0;
}

}  // namespace sdft
