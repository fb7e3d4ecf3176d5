// Registry and launch of the adjoint plane kernels (gd_padj.hpp): 3D, per-point
// field, FP64.
#pragma once

#include <hip/hip_runtime.h>

#include "gd_internal.hpp"

namespace gd {
namespace pl {

struct AdjArgs;

struct AdjEntry {
  int N, Q;
  int (*launch)(AdjArgs&, bool grad, const double*, double*, hipStream_t);
};

struct AdjList {
  const AdjEntry* e;
  int n;
};

AdjList adjoint_instances_n2();
AdjList adjoint_instances_n3();
AdjList adjoint_instances_n4();
AdjList adjoint_instances_n5();

// z = (mass_coef M + adv_coef A)^T r for a pointwise field;
// GD_ERR_UNSUPPORTED (nothing launched) where no instance serves the plan.
int apply_transpose(const gd_plan* plan, double mass_coef, double adv_coef, const double* r, double* z, hipStream_t s);

// d<r, adv_coef A(beta) u> / d beta, likewise.
int grad_beta(const gd_plan* plan, double adv_coef, const double* u, const double* r, double* dcell,
              double* const* dface, hipStream_t s);

}  // namespace pl
}  // namespace gd
