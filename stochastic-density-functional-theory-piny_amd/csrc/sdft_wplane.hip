// sdft_wplane.hip -- kernels and launchers of the wave-private plane stage
// (sdft_plane_wave.h).
#include <algorithm>
#include <type_traits>

#include "sdft_kb.h"
#include "sdft_plane_wave.h"

namespace sdft {

template <typename T, int N, int MODE>
__global__ __launch_bounds__((WPlane<T, N>::NT)) void k_wplane(PlaneArgs a) {
  wplane_body<T, N, MODE>(a, blockIdx.x, blockIdx.y);
}

template <typename T, int N>
__global__ __launch_bounds__((WPlane<T, N>::NT)) void k_wplane_batch(
    const PlaneArgs* __restrict__ args, const int* __restrict__ prefix, int nfrag) {
  const int f = find_frag(prefix, nfrag, blockIdx.x);
  const PlaneArgs a = args[f];
  const int local = blockIdx.x - prefix[f];
  wplane_body<T, N, 0>(a, local % N, local / N);
}

// The plane stage and the KB projection of the same orbitals, which need
// nothing from each other, in one launch: workgroups below nkb are tiles of the
// projection, the rest (plane, pair).
template <typename T, int N>
__global__ __launch_bounds__((WPlane<T, N>::NT)) void k_wplane_project(PlaneArgs a, KbProjectArgs p,
                                                                       int nkb) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int L = blockIdx.x;
  if (L < nkb) {
    const int r = L / p.tp;
    kb_project_tile<T, T, T, WPlane<T, N>::NW, false>(
        reinterpret_cast<const T*>(p.A), reinterpret_cast<const T*>(p.X), p.P, p.ns, p.K, p.per,
        p.zpart, L - r * p.tp, r % p.ts, r / p.ts, reinterpret_cast<double*>(smem_raw));
  } else {
    wplane_body<T, N, 0>(a, (L - nkb) % N, (L - nkb) / N);
  }
}

template <typename T>
static size_t wplane_lds_t(int n, int M) {
  switch (n) {
    case 24: return wplane_lds_bytes<T, 24>(M);
    case 32: return wplane_lds_bytes<T, 32>(M);
    case 36: return wplane_lds_bytes<T, 36>(M);
    case 48: return wplane_lds_bytes<T, 48>(M);
    case 64: return wplane_lds_bytes<T, 64>(M);
    case 96: return wplane_lds_bytes<T, 96>(M);
    case 128: return wplane_lds_bytes<T, 128>(M);
    default: return 0;
  }
}

size_t wplane_lds_for(int n, int prec, int M) {
  const size_t b = prec == 0 ? wplane_lds_t<double>(n, M) : wplane_lds_t<float>(n, M);
  return b <= 160 * 1024 ? b : 0;
}

template <typename T, int N, int MODE>
static int wplane_run(Ctx& c, const PlaneArgs& a, int npairs) {
  auto kern = &k_wplane<T, N, MODE>;
  const size_t lds = wplane_lds_bytes<T, N>(c.g.M);
  SDFT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(N, npairs), dim3(WPlane<T, N>::NT), lds, c.stream, a);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename T, int MODE>
static int wplane_launch(Ctx& c, const PlaneArgs& a, int npairs) {
  SDFT_WPLANE_SWITCH(c.g.n, return (wplane_run<T, NN, MODE>(c, a, npairs)));
  return 0;
}

int launch_wplane(Ctx& c, int prec, const PlaneArgs& a, int npairs, int mode) {
  if (mode == 1)
    return prec == 0 ? wplane_launch<double, 1>(c, a, npairs) : wplane_launch<float, 1>(c, a, npairs);
  if (mode == 3) {
    // runs of 256 points instead of tiles at 24 and 36: never marked
    if (c.g.n % 16 != 0) {
      set_error("internal error: tile marks at a grid without tiles");
      return SDFT_EINVAL_CODE;
    }
    return prec == 0 ? wplane_launch<double, 3>(c, a, npairs) : wplane_launch<float, 3>(c, a, npairs);
  }
  if (mode == 2)
    return prec == 0 ? wplane_launch<double, 2>(c, a, npairs) : wplane_launch<float, 2>(c, a, npairs);
  return prec == 0 ? wplane_launch<double, 0>(c, a, npairs) : wplane_launch<float, 0>(c, a, npairs);
}

template <typename T, int N>
static int wplane_batch_run(const void* args, const int* prefix, int nfrag, int total, size_t lds,
                            hipStream_t s) {
  auto kern = &k_wplane_batch<T, N>;
  SDFT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(total), dim3(WPlane<T, N>::NT), lds, s,
                     reinterpret_cast<const PlaneArgs*>(args), prefix, nfrag);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename T>
static int wplane_batch_t(int n, const void* args, const int* prefix, int nfrag, int total,
                          size_t lds, hipStream_t s) {
  SDFT_WPLANE_SWITCH(n, return (wplane_batch_run<T, NN>(args, prefix, nfrag, total, lds, s)));
  return 0;
}

int launch_wplane_batch(int n, int prec, const void* args, const int* prefix, int nfrag, int total,
                        size_t lds, hipStream_t s) {
  if (total <= 0) return 0;
  return prec == 0 ? wplane_batch_t<double>(n, args, prefix, nfrag, total, lds, s)
                   : wplane_batch_t<float>(n, args, prefix, nfrag, total, lds, s);
}

template <typename T, int N>
static int wplane_project_run(Ctx& c, const PlaneArgs& a, const KbProjectArgs& p, int npairs) {
  auto kern = &k_wplane_project<T, N>;
  const size_t lds = std::max(wplane_lds_bytes<T, N>(c.g.M),
                              sizeof(double) * 1024 * (size_t)WPlane<T, N>::NW);
  const int nkb = p.tp * p.ts * p.nsplit;
  SDFT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(nkb + N * npairs), dim3(WPlane<T, N>::NT), lds, c.stream, a, p,
                     nkb);
  SDFT_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename T>
static int wplane_project_t(Ctx& c, const PlaneArgs& a, const KbProjectArgs& p, int npairs) {
  switch (c.g.n) {
    case 24: return wplane_project_run<T, 24>(c, a, p, npairs);
    case 32: return wplane_project_run<T, 32>(c, a, p, npairs);
    case 36: return wplane_project_run<T, 36>(c, a, p, npairs);
    case 48: return wplane_project_run<T, 48>(c, a, p, npairs);
    case 64: return wplane_project_run<T, 64>(c, a, p, npairs);
    default: set_error("unsupported grid size"); return SDFT_EINVAL_CODE;
  }
}

bool wave_beside_kb(int n, int prec, int npairs) {
  if (n == 128) return npairs > 16;
  return prec == 0 ? n != 48 : n != 64;
}

bool kb_chain_first(int n, int prec, int npairs, bool wave, bool split) {
  const size_t bytes = (prec == 0 ? sizeof(Cx<double>) : sizeof(Cx<float>)) * (size_t)npairs *
                       (size_t)n * n * n;
  return wave || (n < 192 && !split && bytes < kKbBehindBytes);
}

bool kb_small_applies(const Ctx& c, int prec, int ns) {
  const double force = 2.0 * ((ns + 31) / 32 * 32) * c.ppad * 2.0 * c.g.ncp;
  return c.g.n <= 64 && c.plane_variant == 0 && wplane_applies(c, prec, 0) &&
         force <= (prec == 0 ? 1.0 : 3.0) * kKbSmallFlops;
}

bool kb_small_fused(const Ctx& c, int ns) {
  return c.ppad * std::min(ns, 32) <= kKbFusedTile;
}

// waves of a workgroup, which share a tile of the projection
static int wplane_waves(int n) {
  SDFT_WPLANE_SWITCH(n, return WaveCfg<NN>::NW);
  return SDFT_EINVAL_CODE;
}

int launch_plane_project(Ctx& c, int prec, void* W, int npairs, const void* X, int ns,
                         int* nsplit) {
  const int P = c.nproj, K = 2 * c.g.ncp, nsteps = K / 32;
  KbProjectArgs p{};
  p.A = prec == 0 ? (const void*)c.A64 : (const void*)c.A32;
  p.X = X;
  p.P = P;
  p.ns = ns;
  p.K = K;
  p.tp = (P + 31) / 32;
  p.ts = (ns + 31) / 32;
  const int tiles = p.tp * p.ts;
  const int waves = wplane_waves(c.g.n);
  if (waves < 0) return waves;
  const bool fused = kb_small_fused(c, ns);
  int s = (nsteps + waves - 1) / waves;  // one step of the sum per wave
  s = std::min(s, ((fused ? 256 : 128) + tiles - 1) / tiles);
  if (fused) s = std::min(s, std::max(1, kKbFusedPartials / (c.ppad * std::min(ns, 32))));
  p.per = (nsteps + s - 1) / s;
  p.nsplit = (nsteps + p.per - 1) / p.per;
  *nsplit = p.nsplit;
  int rc = ensure_zpart(c, (size_t)p.nsplit * P * ns);
  if (rc) return rc;
  p.zpart = c.zpart;
  const PlaneArgs a = make_plane_args(c, prec, W);
  return prec == 0 ? wplane_project_t<double>(c, a, p, npairs)
                   : wplane_project_t<float>(c, a, p, npairs);
}

}  // namespace sdft
