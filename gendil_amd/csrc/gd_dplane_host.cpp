// Host side of the diffusion plane kernel.
#include <hip/hip_runtime.h>

#include "gd_dplane.hpp"
#include "gd_dplane_api.hpp"

namespace gd {
namespace pl {

namespace {

const DEntry* find_diff(int N, int Q)
{
  DList l{nullptr, 0};
  if (N == 2) l = diff_instances_n2();
  else if (N == 3) l = diff_instances_n3();
  else if (N == 4) l = diff_instances_n4();
  for (int i = 0; i < l.n; ++i)
    if (l.e[i].N == N && l.e[i].Q == Q) return &l.e[i];
  return nullptr;
}

}  // namespace

template <typename T>
int apply_diffusion(const gd_plan* plan, const T* x, T* y, hipStream_t s)
{
  if (plan->generic_pinned[sizeof(T) == 8 ? 0 : 1]) return GD_ERR_UNSUPPORTED;
  if (plan->dim != 3 || plan->E >= (int64_t)1 << 31) return GD_ERR_UNSUPPORTED;
  const DEntry* en = find_diff(plan->desc.order + 1, plan->desc.num_quad);
  if (!en) return GD_ERR_UNSUPPORTED;
  // Small meshes in FP64 leave this kernel a few blocks whose phases nothing
  // hides: there the generic kernel is faster with q >= 4 where mu has
  // several terms or n = 4 (9 x 8 x 10, generic against this: n = 4, q = 4 13.2 and 17.6 us, q = 6
  // 12.6 and 20.9; n = 3, q = 4 14.4 and 15.6), and slower from 15 x 14 x 16 on
  // (18.2 and 14.4; 26.8 and 18.6; 17.3 and 12.4).  q = 3, one term with n < 4
  // and FP32 gain at every size measured.
  if (sizeof(T) == 8 && en->Q >= 4 && plan->E < 2500 && (en->N == 4 || plan->term_rank[kTermMu] > 1))
    return GD_ERR_UNSUPPORTED;
  const TableSet* ts = find_tables(plan, en->N, en->Q);
  DArgs<T> a;
  a.E = (int)plan->E;
  a.periodic_mask = 0;
  double detJ = 1.0;
  for (int d = 0; d < 3; ++d) detJ *= plan->desc.h[d];
  for (int d = 0; d < 3; ++d) {
    a.M[d] = (int)plan->desc.sizes[d];
    if (plan->desc.periodic[d]) a.periodic_mask |= 1 << d;
    a.c[d] = (T)(detJ / (plan->desc.h[d] * plan->desc.h[d]));
  }
  a.sigma = (T)plan->ip_sigma;
  a.kappa = (T)plan->ip_kappa;
  a.gll = plan->desc.basis == GD_BASIS_GLL;
  const Tables1D<T>* tab;
  if constexpr (std::is_same_v<T, double>) {
    tab = &ts->once64;
    a.terms = plan->terms64;
  } else {
    tab = &ts->t32;
    a.terms = plan->terms32;
  }
  a.B = tab->B;
  a.Gb = tab->Gb;
  a.b0 = tab->b0;
  a.b1 = tab->b1;
  a.e0 = tab->d0;
  a.e1 = tab->d1;
  a.w = tab->w;
  a.row0 = plan->term_first[kTermMu];
  a.row1 = plan->term_first[kTermMu + 1];
  a.mu = Field{plan->term_rank[kTermMu], plan->term_mask[kTermMu], 0};
  a.d0 = fast_div(a.M[0]);
  a.d1 = fast_div(a.M[1]);
  if constexpr (std::is_same_v<T, double>) return en->f64(a, x, y, s);
  else return en->f32(a, x, y, s);
}

template int apply_diffusion<double>(const gd_plan*, const double*, double*, hipStream_t);
template int apply_diffusion<float>(const gd_plan*, const float*, float*, hipStream_t);

}  // namespace pl
}  // namespace gd
