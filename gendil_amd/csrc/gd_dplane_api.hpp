// Registry and launch of the diffusion plane kernel (gd_dplane.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "gd_internal.hpp"

namespace gd {
namespace pl {

template <typename T>
struct DArgs;

struct DEntry {
  int N, Q;
  int (*f64)(DArgs<double>&, const double*, double*, hipStream_t);
  int (*f32)(DArgs<float>&, const float*, float*, hipStream_t);
};

struct DList {
  const DEntry* e;
  int n;
};

DList diff_instances_n2();
DList diff_instances_n3();
DList diff_instances_n4();

// y = the SIPDG diffusion apply of a 3D plan; GD_ERR_UNSUPPORTED (nothing
// launched) where no instance serves it.
template <typename T>
int apply_diffusion(const gd_plan* plan, const T* x, T* y, hipStream_t s);

}  // namespace pl
}  // namespace gd
