// Host side of the adjoint plane kernels.
#include <hip/hip_runtime.h>

#include "gd_padj.hpp"
#include "gd_padj_api.hpp"

namespace gd {
namespace pl {

namespace {

const AdjEntry* serving(const gd_plan* plan)
{
  if (plan->generic_pinned[0]) return nullptr;
  if (plan->dim != 3 || plan->padapt || plan->E >= (int64_t)1 << 31 || plan->beta_kind != GD_BETA_POINTWISE)
    return nullptr;
  const int N = plan->desc.order + 1, Q = plan->desc.num_quad;
  AdjList l{nullptr, 0};
  if (N == 2) l = adjoint_instances_n2();
  else if (N == 3) l = adjoint_instances_n3();
  else if (N == 4) l = adjoint_instances_n4();
  else if (N == 5) l = adjoint_instances_n5();
  for (int i = 0; i < l.n; ++i)
    if (l.e[i].N == N && l.e[i].Q == Q) return &l.e[i];
  return nullptr;
}

AdjArgs pack(const gd_plan* plan, double mass_coef, double adv_coef)
{
  AdjArgs a{};
  a.E = (int)plan->E;
  double detJ = 1.0;
  for (int d = 0; d < 3; ++d) detJ *= plan->desc.h[d];
  for (int d = 0; d < 3; ++d) {
    a.M[d] = (int)plan->desc.sizes[d];
    if (plan->desc.periodic[d]) a.periodic_mask |= 1 << d;
    a.c[d] = adv_coef * detJ / plan->desc.h[d];
    a.beta_face[d] = plan->beta_face[d];
  }
  a.mass = mass_coef * detJ;
  a.d0 = fast_div(a.M[0]);
  a.d1 = fast_div(a.M[1]);
  a.gll = plan->desc.basis == GD_BASIS_GLL;
  a.bc_none = plan->bc_mode == GD_BC_NONE;
  a.bc_data = !a.bc_none && plan->bc_host.rank > 0;
  a.beta_cell = plan->beta_cell;
  const FieldDev<double>* f = static_cast<const FieldDev<double>*>(plan->fields64);
  a.sigma = f + 3;
  a.bc = f + 4;
  const Tables1D<double>& t = find_tables(plan, plan->desc.order + 1, plan->desc.num_quad)->once64;
  a.B = t.B;
  a.Gb = t.Gb;
  a.b0 = t.b0;
  a.b1 = t.b1;
  a.w = t.w;
  return a;
}

}  // namespace

int apply_transpose(const gd_plan* plan, double mass_coef, double adv_coef, const double* r, double* z, hipStream_t s)
{
  const AdjEntry* en = serving(plan);
  if (!en) return GD_ERR_UNSUPPORTED;
  AdjArgs a = pack(plan, mass_coef, adv_coef);
  return en->launch(a, false, r, z, s);
}

int grad_beta(const gd_plan* plan, double adv_coef, const double* u, const double* r, double* dcell,
              double* const* dface, hipStream_t s)
{
  const AdjEntry* en = serving(plan);
  if (!en) return GD_ERR_UNSUPPORTED;
  AdjArgs a = pack(plan, 0.0, adv_coef);
  a.dcell = dcell;
  for (int d = 0; d < 3; ++d) a.dface[d] = dface[d];
  return en->launch(a, true, u, const_cast<double*>(r), s);  // reads r through its second vector argument
}

}  // namespace pl
}  // namespace gd
