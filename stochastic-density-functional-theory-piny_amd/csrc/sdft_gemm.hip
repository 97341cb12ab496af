// sdft_gemm.hip -- Kleinman-Bylander projector contraction as MFMA GEMMs.
//
// The G-space KB path of the reference loops over G x atoms x (l,m) x states
// with scalar arithmetic (controlEwdNonlocFilter / getNlmatFilter,
// stodft/reduced-energy/cp-energy-eext-stodft.c:865-946,1105-1168, and
// getnl_fcoef, energy/cp/cp_energy_eext_nonloc.c:1669+).  With the projector
// table folded into A[p][2 ncp] (Gamma weights included) the same arithmetic
// is two dense products over the orbital block X (2 ncp x nstate):
//   Z  = A X                      (projections, split-K, reduced in FP64)
//   Y  = -2 diag(E) Z
//   F  = A^T Y                    (raw NL force, -4/-2 scaling included)
//
// Both products run on the 16x16x4 MFMA (v_mfma_f64_16x16x4f64 for the FP64
// form, v_mfma_f32_16x16x4f32 for the FP32 form).  The K order of an MFMA
// accumulation is free, so lane l (row or column l%16, group g = l/16) owns
// the 8 consecutive k = k0 + 8g .. k0 + 8g + 7 of a 32-wide K step and loads
// them with vector loads straight into registers: no LDS staging and no
// barriers inside the K loop.  Each wave accumulates a 32x32 tile (2x2 MFMA
// blocks).
#include <algorithm>

#include "sdft_kb.h"

namespace sdft {

// 1-D launch over ts * ceil(K2 / kForceCols) blocks, XCD-swizzled, s fastest:
// the blocks sharing one slab of At sit on one XCD.
template <typename T>
__global__ __launch_bounds__(256) void k_kb_force(const T* __restrict__ Y, const T* __restrict__ At,
                                                  int ns, int K2, int ppad, T* __restrict__ F,
                                                  int ts, int total) {
  const int L = xcd_swizzle(blockIdx.x, total);
  kb_force_block<T>(Y, At, ns, K2, ppad, F, L % ts, L / ts);
}

// 1-D launch over tp * ts * nsplit tiles.  Logical tile L (XCD-swizzled) is
// split-major, then column tile, then row tile: the tiles of one K slice sit
// on one XCD, whose L2 then holds that slice of both operands.
template <typename TA, typename TX, typename TI>
__global__ __launch_bounds__(256) void k_kb_project(const TA* __restrict__ A,
                                                    const TX* __restrict__ X, int P, int ns,
                                                    int K, int ksteps_per_split,
                                                    double* __restrict__ zpart, int tp, int ts,
                                                    int total) {
  __shared__ double red[4 * 32 * 32];
  const int L = xcd_swizzle(blockIdx.x, total);
  const int bx = L % tp, r = L / tp;
  kb_project_tile<TA, TX, TI>(A, X, P, ns, K, ksteps_per_split, zpart, bx, r % ts, r / ts, red);
}

// One launch over the fragments of a batch: workgroup w belongs to fragment
// f with prefix[f] <= w < prefix[f+1]; its tile is (local % tp, local / tp %
// ts, local / (tp ts)).
template <typename TA, typename TI>
__global__ __launch_bounds__(256) void k_kb_project_batch(const KbProjectArgs* __restrict__ args,
                                                          const int* __restrict__ prefix,
                                                          int nfrag) {
  __shared__ double red[4 * 32 * 32];
  const int L = xcd_swizzle(blockIdx.x, prefix[nfrag]);
  const int f = find_frag(prefix, nfrag, L);
  const KbProjectArgs a = args[f];
  const int local = L - prefix[f];
  const int bx = local % a.tp, r = local / a.tp;
  kb_project_tile<TA, TA, TI>(reinterpret_cast<const TA*>(a.A), reinterpret_cast<const TA*>(a.X),
                              a.P, a.ns, a.K, a.per, a.zpart, bx, r % a.ts, r / a.ts, red);
}

// Z[p][s] = sum_z part[z][p][s];  Y[s][p] = -2 E_p Z[p][s] (transposed, row
// stride ppad, in the form's type TY; the padding columns p >= P are never
// written and stay zero)
template <typename TY>
__device__ __forceinline__ void nl_reduce_elem(const double* __restrict__ part, int nsplit, int P,
                                               int ns, int ppad, const double* __restrict__ E,
                                               double* __restrict__ Z, TY* __restrict__ Y, int i) {
  if (i >= P * ns) return;
  double s = 0.0;
  for (int z = 0; z < nsplit; ++z) s += part[(size_t)z * P * ns + i];
  const int p = i / ns, st = i - p * ns;
  Z[i] = s;
  if (Y) Y[(size_t)st * ppad + p] = TY(-2.0 * E[p] * s);
}

template <typename TY>
__global__ void k_nl_reduce(const double* __restrict__ part, int nsplit, int P, int ns, int ppad,
                            const double* __restrict__ E, double* __restrict__ Z,
                            TY* __restrict__ Y) {
  nl_reduce_elem<TY>(part, nsplit, P, ns, ppad, E, Z, Y, blockIdx.x * blockDim.x + threadIdx.x);
}

template <typename TY>
__global__ __launch_bounds__(256) void k_nl_reduce_batch(const KbReduceArgs* __restrict__ args,
                                                         const int* __restrict__ prefix,
                                                         int nfrag) {
  const int f = find_frag(prefix, nfrag, blockIdx.x);
  const KbReduceArgs a = args[f];
  nl_reduce_elem<TY>(a.zpart, a.nsplit, a.P, a.ns, a.ppad, a.E, a.Z, reinterpret_cast<TY*>(a.Y),
                     (blockIdx.x - prefix[f]) * 256 + threadIdx.x);
}

// ---- batched F[s][k] = sum_p Y[s][p] At[k][p] ------------------------------
// kb_force_block per fragment: ts x tk blocks of 32 states x kForceCols columns.
template <typename T>
__global__ __launch_bounds__(256) void k_kb_force_batch(const KbForceArgs* __restrict__ args,
                                                        const int* __restrict__ prefix,
                                                        int nfrag) {
  const int L = xcd_swizzle(blockIdx.x, prefix[nfrag]);
  const int f = find_frag(prefix, nfrag, L);
  const KbForceArgs a = args[f];
  const int local = L - prefix[f];
  kb_force_block<T>(reinterpret_cast<const T*>(a.Y), reinterpret_cast<const T*>(a.At), a.ns, a.K2,
                    a.ppad, reinterpret_cast<T*>(a.F), local % a.ts, local / a.ts);
}

static int ensure(void** p, size_t* have, size_t need) {
  if (*have >= need) return 0;
  if (*p) SDFT_HIP_CHECK(hipFree(*p));
  *p = nullptr;
  *have = 0;
  hipError_t e = hipMalloc(p, need);
  if (e != hipSuccess) {
    set_error("device allocation failed (KB scratch)");
    return -3;
  }
  *have = need;
  return 0;
}

// K split of the projection GEMM: about c.kb_wg_target workgroups (512 unless
// tuned), at least 16 K steps (four per wave) per split.  Returns the split
// count, *per = steps per split.
int kb_project_split(const Ctx& c, int ns, int* per) {
  const int P = c.nproj;
  const int K = 2 * c.g.ncp;  // multiple of 128
  const int tiles = ((P + 31) / 32) * ((ns + 31) / 32);
  const int nsteps = K / KS;
  int nsplit = (c.kb_wg_target + tiles - 1) / tiles;
  if (nsplit > nsteps / 16) nsplit = nsteps / 16;
  if (nsplit < 1) nsplit = 1;
  *per = (nsteps + nsplit - 1) / nsplit;
  return (nsteps + *per - 1) / *per;
}

int ensure_zpart(Ctx& c, size_t n) {
  return ensure(reinterpret_cast<void**>(&c.zpart), &c.zpart_bytes, sizeof(double) * n);
}

// Y is [ns][ppad] with zero padding columns: (re)allocated and cleared
// whenever it grows or the padded projector count changes.  Z ([P][ns],
// written by the reduction for every state) is allocated with the same padded
// row count, so it holds P * ns doubles whenever Y needs no reallocation.
static int ensure_Y(Ctx& c, int ns) {
  const int ns_pad = (ns + 31) / 32 * 32;
  const size_t ybytes = sizeof(double) * (size_t)c.ppad * ns_pad;
  if (c.Y_bytes >= ybytes && c.Y_ppad == c.ppad) return 0;
  if (c.Y) SDFT_HIP_CHECK(hipFree(c.Y));
  if (c.Y32) SDFT_HIP_CHECK(hipFree(c.Y32));
  if (c.Z) SDFT_HIP_CHECK(hipFree(c.Z));
  c.Y = c.Z = nullptr;
  c.Y32 = nullptr;
  c.Y_bytes = 0;
  if (hipMalloc(&c.Y, ybytes) != hipSuccess || hipMalloc(&c.Y32, ybytes / 2) != hipSuccess ||
      hipMalloc(&c.Z, sizeof(double) * (size_t)c.ppad * ns_pad) != hipSuccess) {
    set_error("device allocation failed (KB projections)");
    return -3;
  }
  SDFT_HIP_CHECK(hipMemsetAsync(c.Y, 0, ybytes, c.stream));
  SDFT_HIP_CHECK(hipMemsetAsync(c.Y32, 0, ybytes / 2, c.stream));
  c.Y_bytes = ybytes;
  c.Y_ppad = c.ppad;
  return 0;
}

// Z and Y from the nsplit partials in c.zpart
int launch_nl_reduce(Ctx& c, int prec, int ns, int nsplit) {
  const int P = c.nproj, nel = P * ns;
  int rc = ensure_Y(c, ns);
  if (rc) return rc;
  if (prec == 0)
    hipLaunchKernelGGL(k_nl_reduce<double>, dim3((nel + 255) / 256), dim3(256), 0, c.stream,
                       c.zpart, nsplit, P, ns, c.ppad, c.E, c.Z, c.Y);
  else
    hipLaunchKernelGGL(k_nl_reduce<float>, dim3((nel + 255) / 256), dim3(256), 0, c.stream,
                       c.zpart, nsplit, P, ns, c.ppad, c.E, c.Z, c.Y32);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_nl_project(Ctx& c, int prec, const void* X, int ns) {
  const int P = c.nproj;
  const int K = 2 * c.g.ncp;
  int per = 0;
  const int nsplit = kb_project_split(c, ns, &per);
  int rc = ensure_zpart(c, (size_t)nsplit * P * ns);
  if (rc) return rc;
  const int tp = (P + 31) / 32, ts = (ns + 31) / 32, tot = tp * ts * nsplit;
  if (prec == 0)
    hipLaunchKernelGGL((k_kb_project<double, double, double>), dim3(tot), dim3(256), 0, c.stream,
                       c.A64, static_cast<const double*>(X), P, ns, K, per, c.zpart, tp, ts, tot);
  else
    hipLaunchKernelGGL((k_kb_project<float, float, float>), dim3(tot), dim3(256), 0, c.stream,
                       c.A32, static_cast<const float*>(X), P, ns, K, per, c.zpart, tp, ts, tot);
  SDFT_HIP_CHECK(hipGetLastError());
  return launch_nl_reduce(c, prec, ns, nsplit);
}

// Ad[p][j] = G_d(j) A[p][ncp + j], Ad[p][ncp + j] = -G_d(j) A[p][j]: the table
// of dQ_p/dR_a = i G Q_p in the same Gamma packing (G = 0 gives zero).
__global__ void k_kb_deriv_table(const double* __restrict__ A, const double* __restrict__ gd,
                                 int P, int ncp, double* __restrict__ Ad) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)P * ncp) return;
  const size_t p = i / ncp, j = i - p * ncp;
  const double g = gd[j];
  Ad[p * 2 * ncp + j] = g * A[p * 2 * ncp + ncp + j];
  Ad[p * 2 * ncp + ncp + j] = -g * A[p * 2 * ncp + j];
}

// S[p*3 + d] = sum_{s < nstate} Z[p][s] Zd[d][p][s]
__global__ void k_force_sums(const double* __restrict__ Z, const double* __restrict__ Zd, int P,
                             int ns, int nstate, double* __restrict__ S) {
  __shared__ double sh[3][256];
  const int p = blockIdx.x;
  double a[3] = {0, 0, 0};
  for (int s = threadIdx.x; s < nstate; s += blockDim.x) {
    const double z = Z[(size_t)p * ns + s];
#pragma unroll
    for (int d = 0; d < 3; ++d) a[d] += z * Zd[((size_t)d * P + p) * ns + s];
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) sh[d][threadIdx.x] = a[d];
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int d = 0; d < 3; ++d) sh[d][threadIdx.x] += sh[d][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int d = 0; d < 3; ++d) S[p * 3 + d] = sh[d][0];
}

// dZ/dR for the three directions (FP64) and the per-projector sums; gint is
// G in internal coefficient order [3][ncp].
int nl_force_sums(Ctx& c, const double* X, int ns, int nstate, const double* gint,
                  double* Ad, double* Zd, double* part, double* S) {
  const int P = c.nproj;
  const int K = 2 * c.g.ncp;
  int rc = launch_nl_project(c, 0, X, ns);  // c.Z = A X
  if (rc) return rc;
  int per = 0;
  const int nsplit = kb_project_split(c, ns, &per);
  for (int d = 0; d < 3; ++d) {
    const size_t tot = (size_t)P * c.g.ncp;
    hipLaunchKernelGGL(k_kb_deriv_table, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0,
                       c.stream, c.A64, gint + (size_t)d * c.g.ncp, P, c.g.ncp, Ad);
    const int tp = (P + 31) / 32, ts = (ns + 31) / 32, ntile = tp * ts * nsplit;
    hipLaunchKernelGGL((k_kb_project<double, double, double>), dim3(ntile), dim3(256), 0,
                       c.stream, Ad, X, P, ns, K, per, part, tp, ts, ntile);
    // reduce the split partials into Zd[d] (the E factor is applied later)
    const int n2 = P * ns;
    hipLaunchKernelGGL(k_nl_reduce<double>, dim3((n2 + 255) / 256), dim3(256), 0, c.stream, part,
                       nsplit, P, ns, c.ppad, c.E, Zd + (size_t)d * n2, (double*)nullptr);
    SDFT_HIP_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(k_force_sums, dim3(P), dim3(256), 0, c.stream, c.Z, Zd, P, ns, nstate, S);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

// F[s][k] = sum_p Y[s][p] At[k][p] (K2 = 2 ncp is a multiple of 128), F in
// the form's type
int launch_nl_force(Ctx& c, int prec, int ns, void* fnl) {
  const int K2 = 2 * c.g.ncp;
  const int ts = (ns + 31) / 32, tot = ts * ((K2 + kForceCols - 1) / kForceCols);
  if (prec == 0)
    hipLaunchKernelGGL((k_kb_force<double>), dim3(tot), dim3(256), 0, c.stream, c.Y, c.At64, ns,
                       K2, c.ppad, static_cast<double*>(fnl), ts, tot);
  else
    hipLaunchKernelGGL((k_kb_force<float>), dim3(tot), dim3(256), 0, c.stream, c.Y32, c.At32, ns,
                       K2, c.ppad, static_cast<float*>(fnl), ts, tot);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename T>
__global__ __launch_bounds__(256) void k_kb_reduce_force(const double* __restrict__ zpart,
                                                         int nsplit, int P, int ns, int ppad,
                                                         const double* __restrict__ E,
                                                         const T* __restrict__ At, int K2,
                                                         T* __restrict__ F, int ts) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  kb_reduce_force<T>(zpart, nsplit, P, ns, ppad, E, At, K2, F, blockIdx.x % ts, blockIdx.x / ts,
                     reinterpret_cast<T*>(smem_raw));
}

int launch_kb_reduce_force(Ctx& c, int prec, int ns, int nsplit, void* fnl) {
  const int K2 = 2 * c.g.ncp, ts = (ns + 31) / 32, tot = ts * (K2 / 64);
  // as many rows as a tile has states: at most kKbFusedTile projections
  const size_t lds = (size_t)std::min(ns, 32) * kb_small_ldy(c.ppad) * (prec == 0 ? 8 : 4);
  if (prec == 0) {
    auto kern = &k_kb_reduce_force<double>;
    SDFT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(tot), dim3(256), lds, c.stream, c.zpart, nsplit, c.nproj, ns,
                       c.ppad, c.E, c.At64, K2, static_cast<double*>(fnl), ts);
  } else {
    auto kern = &k_kb_reduce_force<float>;
    SDFT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(tot), dim3(256), lds, c.stream, c.zpart, nsplit, c.nproj, ns,
                       c.ppad, c.E, c.At32, K2, static_cast<float*>(fnl), ts);
  }
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

// kind 0: projection partials, 1: split reduction + Y, 2: force product
int launch_kb_batch(int kind, int prec, const void* args, const int* prefix, int nfrag,
                    int total, hipStream_t s) {
  if (total <= 0) return 0;
  if (kind == 0) {
    if (prec == 0)
      hipLaunchKernelGGL((k_kb_project_batch<double, double>), dim3(total), dim3(256), 0, s,
                         reinterpret_cast<const KbProjectArgs*>(args), prefix, nfrag);
    else
      hipLaunchKernelGGL((k_kb_project_batch<float, float>), dim3(total), dim3(256), 0, s,
                         reinterpret_cast<const KbProjectArgs*>(args), prefix, nfrag);
  } else if (kind == 1) {
    if (prec == 0)
      hipLaunchKernelGGL(k_nl_reduce_batch<double>, dim3(total), dim3(256), 0, s,
                         reinterpret_cast<const KbReduceArgs*>(args), prefix, nfrag);
    else
      hipLaunchKernelGGL(k_nl_reduce_batch<float>, dim3(total), dim3(256), 0, s,
                         reinterpret_cast<const KbReduceArgs*>(args), prefix, nfrag);
  } else {
    if (prec == 0)
      hipLaunchKernelGGL((k_kb_force_batch<double>), dim3(total), dim3(256), 0, s,
                         reinterpret_cast<const KbForceArgs*>(args), prefix, nfrag);
    else
      hipLaunchKernelGGL((k_kb_force_batch<float>), dim3(total), dim3(256), 0, s,
                         reinterpret_cast<const KbForceArgs*>(args), prefix, nfrag);
  }
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace sdft
