// Host side of the plane kernel: eligibility, instance lookup and launch.
#include <hip/hip_runtime.h>

#include "gd_plane.hpp"
#include "gd_plane_api.hpp"

namespace gd {
namespace pl {

namespace {

const Entry* find(int N, int Q)
{
  List l{nullptr, 0};
  if (N == 2) l = instances_n2();
  else if (N == 3) l = instances_n3();
  else if (N == 4) l = instances_n4();
  else if (N == 5) l = instances_n5();
  for (int i = 0; i < l.n; ++i)
    if (l.e[i].N == N && l.e[i].Q == Q) return &l.e[i];
  return nullptr;
}

// 3D, uniform order; element and neighbour numbers in 32 bits
const Entry* serving(const gd_plan* plan)
{
  if (plan->dim != 3 || plan->padapt || plan->E >= (int64_t)1 << 31) return nullptr;
  return find(plan->desc.order + 1, plan->desc.num_quad);
}

}  // namespace

template <typename T>
bool available(const gd_plan* plan, bool /*adv*/, bool /*mass*/)
{
  return serving(plan) != nullptr;
}

template <typename T>
bool preferred(const gd_plan* plan, bool adv)
{
  const bool spills = sizeof(T) == 8 && adv && plan->desc.order == 4 && plan->desc.num_quad == 6;
  return !spills || plan->E >= 1000;
}

template <typename T>
int apply(const gd_plan* plan, T mass_coef, T adv_coef, const T* x, T* y, hipStream_t s)
{
  const bool adv = adv_coef != T(0);
  const Entry* en = serving(plan);
  if (!en) return GD_ERR_UNSUPPORTED;
  const TableSet* ts = find_tables(plan, en->N, en->Q);
  Args<T> a;
  a.E = (int)plan->E;
  a.periodic_mask = 0;
  double detJ = 1.0;
  for (int d = 0; d < 3; ++d) {
    a.M[d] = (int)plan->desc.sizes[d];
    if (plan->desc.periodic[d]) a.periodic_mask |= 1 << d;
    a.h[d] = (T)plan->desc.h[d];
    a.invh[d] = (T)(1.0 / plan->desc.h[d]);
    a.origin[d] = (T)plan->desc.origin[d];
    a.affc[d] = (T)plan->affc[d];
    for (int c = 0; c < 3; ++c) a.affA[c][d] = (T)plan->affA[c][d];
    detJ *= plan->desc.h[d];
  }
  a.detJ = (T)detJ;
  a.mass_coef = mass_coef;
  a.adv_coef = adv_coef;
  a.gll = plan->desc.basis == GD_BASIS_GLL;
  a.field = plan->beta_kind == GD_BETA_AFFINE ? kAffine : (plan->beta_kind == GD_BETA_POINTWISE ? kPointwise : kSeparable);
  if constexpr (std::is_same_v<T, double>) {
    a.beta_cell = plan->beta_cell;
    for (int d = 0; d < 3; ++d) a.beta_face[d] = plan->beta_face[d];
  }
  a.bc_none = plan->bc_mode == GD_BC_NONE;
  a.bc_data = !a.bc_none && plan->bc_host.rank > 0;
  const Tables1D<T>* tab;
  if constexpr (std::is_same_v<T, double>) {
    tab = adv ? &ts->once64 : &ts->t64;  // mass applies keep the generic kernel's bits
    a.terms = plan->terms64;
    a.sigma_tab = static_cast<const FieldDev<double>*>(plan->fields64) + 3;
  } else {
    tab = &ts->t32;
    a.terms = plan->terms32;
    a.sigma_tab = static_cast<const FieldDev<float>*>(plan->fields32) + 3;
  }
  a.B = tab->B;
  a.Gb = tab->Gb;
  a.b0 = tab->b0;
  a.b1 = tab->b1;
  a.xq = tab->xq;
  a.w = tab->w;
  // sigma's rows come first, then beta's and the boundary data's
  a.row0 = plan->term_first[mass_coef != T(0) ? kTermSigma : kTermBeta];
  a.row1 = plan->term_first[adv ? kTermBc + 1 : kTermBeta];
  if (a.row1 < a.row0) a.row1 = a.row0;
  auto field = [&](int f) { return Field{plan->term_rank[f], plan->term_mask[f], plan->term_first[f] - a.row0}; };
  a.sigma = field(kTermSigma);
  for (int d = 0; d < 3; ++d) a.beta[d] = field(kTermBeta + d);
  a.bc = field(kTermBc);
  a.d0 = fast_div(a.M[0]);
  a.d1 = fast_div(a.M[1]);
  if constexpr (std::is_same_v<T, double>) return (adv ? en->adv64 : en->mass64)(a, x, y, s);
  else return (adv ? en->adv32 : en->mass32)(a, x, y, s);
}

template bool available<double>(const gd_plan*, bool, bool);
template bool available<float>(const gd_plan*, bool, bool);
template bool preferred<double>(const gd_plan*, bool);
template bool preferred<float>(const gd_plan*, bool);
template int apply<double>(const gd_plan*, double, double, const double*, double*, hipStream_t);
template int apply<float>(const gd_plan*, float, float, const float*, float*, hipStream_t);

}  // namespace pl
}  // namespace gd
