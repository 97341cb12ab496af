// sdft_wplane.hip -- kernels and launchers of the wave-private plane stage
// (sdft_plane_wave.h).
#include <type_traits>

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

}  // namespace sdft
