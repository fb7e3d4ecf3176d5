// Launchers and instance lists of the plane kernel, one translation unit per
// node count so that they compile in parallel.
#pragma once

#include "gd_plane.hpp"
#include "gd_plane_api.hpp"
#include "gd_sizing.hpp"

namespace gd {
namespace pl {

template <typename T, int N, int Q, bool ADV, bool GLL, int FIELD>
int launch_kind(Args<T>& a, const T* x, T* y, hipStream_t s)
{
  using G = Geo<N, Q, ADV>;
  a.spitch = ADV ? ((a.row1 - a.row0) * (Q + 2)) | 1 : 0;
  const size_t per = (size_t)(G::PL * G::PITCH + a.spitch) * sizeof(T);
  // full blocks, unless the coefficients' samples leave too little LDS for two
  // blocks a CU or the mesh is too small for two blocks a CU
  auto kern = plane_kernel<T, N, Q, ADV, GLL, FIELD>;
  static const int resident = blocks_per_cu(kern, G::NT);
  int most = G::EPB;
  while (most > 4 && (size_t)most * per > 80 * 1024) most = (most + 1) / 2;
  a.epb = elements_per_block(a.E, 4, most, per, resident);
  a.num_blocks = (int)((a.E + a.epb - 1) / a.epb);
  const size_t lds = a.epb * per;
  if (lds > 160 * 1024) return GD_ERR_UNSUPPORTED;
  if (lds > 64 * 1024) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    GD_HIP(attr);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)a.num_blocks), dim3(G::NT), lds, s, a, x, y);
  GD_HIP(hipGetLastError());
  return GD_OK;
}

template <typename T, int N, int Q, bool ADV>
int launch(Args<T>& a, const T* x, T* y, hipStream_t s)
{
  if constexpr (!ADV) return launch_kind<T, N, Q, false, true, kSeparable>(a, x, y, s);  // no traces, no beta
  else {
    if constexpr (sizeof(T) == 8)
      if (a.field == kPointwise) return a.gll ? launch_kind<T, N, Q, true, true, kPointwise>(a, x, y, s)
                                              : launch_kind<T, N, Q, true, false, kPointwise>(a, x, y, s);
    if (a.field == kAffine) return a.gll ? launch_kind<T, N, Q, true, true, kAffine>(a, x, y, s)
                                         : launch_kind<T, N, Q, true, false, kAffine>(a, x, y, s);
    return a.gll ? launch_kind<T, N, Q, true, true, kSeparable>(a, x, y, s)
                 : launch_kind<T, N, Q, true, false, kSeparable>(a, x, y, s);
  }
}

#define GD_PLANE(N, Q)                                                                                  \
  Entry                                                                                                 \
  {                                                                                                     \
    N, Q, &launch<double, N, Q, true>, &launch<double, N, Q, false>, &launch<float, N, Q, true>,        \
        &launch<float, N, Q, false>                                                                     \
  }

}  // namespace pl
}  // namespace gd
