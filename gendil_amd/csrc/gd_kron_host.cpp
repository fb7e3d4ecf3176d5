// Host side of the 4D-6D Kronecker kernel: which coefficients it serves, the
// terms and their matrices, launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <vector>

#include "gd_kron.hpp"
#include "gd_kron_api.hpp"

namespace gd {
namespace kron {

// One term: matrices along a (and b), offsets into the device blobs; -1 none
struct HostTerm {
  int a = 0, b = 0, inflow = 0;
  int64_t ta = -1, tb = -1, tf = -1;
  double scale = 1.0;
};

struct State {
  bool adv_ok = false, mass_ok = false;
  std::vector<HostTerm> adv, mass;
  double sigma_const = 0.0;  // sum of sigma's constant terms
  // offset of the mass matrix, M / unit; unit^dim goes into the factors of the terms
  int64_t mm = 0;
  double units = 1.0;
  // one allocation, kept from one set of coefficients to the next while they
  // fit: the values in FP64, then in FP32
  void* dev = nullptr;
  size_t capacity = 0, words = 0;  // values
  const double* f64() const { return static_cast<const double*>(dev); }
  const float* f32() const { return reinterpret_cast<const float*>(f64() + words); }
};

void destroy_state(State* s)
{
  if (!s) return;
  if (s->dev) (void)hipFree(s->dev);
  delete s;
}

namespace {

// Matrices are formed in extended precision and rounded once.
using Ext = long double;
constexpr int kMaxN = 5;  // nodes of any instance
using Table = std::vector<Ext>;
using Mat = std::array<Ext, kMaxN * kMaxN>;  // n x n or n x 1, row-major

// inverse by Gauss-Jordan with partial pivoting
Mat inverse(const Mat& a, int n)
{
  Ext m[kMaxN][2 * kMaxN] = {};
  for (int i = 0; i < n; ++i) {
    for (int j = 0; j < n; ++j) m[i][j] = a[i * n + j];
    m[i][n + i] = 1.0L;
  }
  for (int c = 0; c < n; ++c) {
    int p = c;
    for (int i = c + 1; i < n; ++i)
      if (std::fabs(m[i][c]) > std::fabs(m[p][c])) p = i;
    for (int j = 0; j < 2 * n; ++j) std::swap(m[c][j], m[p][j]);
    const Ext d = m[c][c];
    for (int j = 0; j < 2 * n; ++j) m[c][j] /= d;
    for (int i = 0; i < n; ++i) {
      if (i == c) continue;
      const Ext f = m[i][c];
      for (int j = 0; j < 2 * n; ++j) m[i][j] -= f * m[c][j];
    }
  }
  Mat r{};
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) r[i * n + j] = m[i][n + j];
  return r;
}

// The unit in which M rounds best, M_00 / k for the k <= 64 with the smallest
// rounding error: M multiplies along every axis, so an error of its entries adds
// up over the axes, the same in every value.  Left over: at most 0.07 units in
// the last place (n <= 5), against up to half a unit per axis.
Ext mass_unit(const Mat& M, int n)
{
  Ext best = -1.0L, unit = M[0];
  for (int k = 1; k <= 64; ++k) {
    const Ext u = M[0] / k;
    Ext e = 0.0L;
    for (int i = 0; i < n * n; ++i) {
      const Ext v = M[i] / u, d = (Ext)(double)v - v;
      e += d * d;
    }
    e *= u * u;
    if (best < 0.0L || e < best) {
      best = e;
      unit = u;
    }
  }
  return unit;
}

const Entry* find(const gd_plan* plan)
{
  List l{nullptr, 0};
  if (plan->dim == 4) l = instances_d4();
  else if (plan->dim == 5) l = instances_d5();
  else if (plan->dim == 6) l = instances_d6();
  for (int i = 0; i < l.n; ++i)
    if (l.e[i].N == plan->desc.order + 1) return &l.e[i];
  return nullptr;
}

// A field of at most one coordinate, as its axis (-1: constant) and its q + 2
// samples per position along it
struct OneAxis {
  int axis = -1;
  std::vector<double> v;  // axis < 0: one value
};

bool one_axis(const gd_plan* p, int c, const TableSet& ts, OneAxis& out)
{
  const int D = p->dim, q = ts.q;
  if (p->beta_kind == GD_BETA_SEPARABLE) {
    const HostField& f = p->beta_host[c];
    double cst = 0.0;
    int term = -1;
    for (int r = 0; r < f.rank; ++r) {
      int used = 0, ax = -1;
      for (int d = 0; d < D; ++d)
        if (f.offset[r][d] >= 0) {
          ++used;
          ax = d;
        }
      if (used == 0) cst += f.scale[r];
      else if (used > 1 || term >= 0) return false;
      else {
        term = r;
        out.axis = ax;
      }
    }
    if (term < 0) {
      out.v.assign(1, cst);
      return true;
    }
    const int64_t n = p->desc.sizes[out.axis] * (q + 2);
    out.v.resize(n);
    for (int64_t i = 0; i < n; ++i) out.v[i] = cst + f.scale[term] * f.data[f.offset[term][out.axis] + i];
    return true;
  }
  if (p->beta_kind != GD_BETA_AFFINE) return false;
  for (int d = 0; d < D; ++d)
    if (p->affA[c][d] != 0.0) {
      if (out.axis >= 0) return false;
      out.axis = d;
    }
  if (out.axis < 0) {
    out.v.assign(1, p->affc[c]);
    return true;
  }
  const int a = out.axis;
  out.v.resize(p->desc.sizes[a] * (q + 2));
  for (int64_t e = 0; e < p->desc.sizes[a]; ++e)
    for (int k = 0; k < q + 2; ++k) {
      const double xi = k < q ? ts.xq[k] : (k == q ? 0.0 : 1.0);
      out.v[e * (q + 2) + k] =
          p->affc[c] + p->affA[c][a] * ((p->desc.origin[a] + p->desc.h[a] * (double)e) + p->desc.h[a] * xi);
    }
  return true;
}

}  // namespace

int refresh(const gd_plan* plan)
{
  if (!plan->kron_state) plan->kron_state = new State();
  State& st = *plan->kron_state;
  st.adv_ok = st.mass_ok = false;
  st.adv.clear();
  st.mass.clear();
  st.sigma_const = 0.0;
  const int D = plan->dim;
  if (D < 4 || plan->padapt || plan->E >= (int64_t)1 << 31 || !find(plan)) return GD_OK;
  const int n = plan->desc.order + 1, q = plan->desc.num_quad;
  const TableSet* ts = find_tables(plan, n, q);
  if (!ts || q < n) return GD_OK;  // M is singular with fewer points than nodes
  const RuleTables<Ext>& t1 = ts->ext;
  auto gram = [&](const Table& L, const double* f) {  // L^T W f B
    Mat m{};
    for (int k = 0; k < q; ++k) {
      const Ext wf = t1.w[k] * (f ? f[k] : 1.0);
      for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) m[i * n + j] += wf * L[k * n + i] * t1.B[k * n + j];
    }
    return m;
  };
  const Mat M = gram(t1.B, nullptr), Mi = inverse(M, n);
  std::vector<double> blob;
  auto put = [&](std::vector<double>& to, const Mat& m, int count) {
    const int64_t at = (int64_t)to.size();
    for (int i = 0; i < count; ++i) to.push_back((double)m[i]);
    return at;
  };
  auto times = [&](const Mat& m, int cols) {  // M^-1 m
    Mat r{};
    for (int i = 0; i < n; ++i)
      for (int k = 0; k < n; ++k)
        for (int j = 0; j < cols; ++j) r[i * cols + j] += Mi[i * n + k] * m[k * cols + j];
    return r;
  };
  const Ext unit = mass_unit(M, n);
  Mat Mu(M);
  for (Ext& v : Mu) v /= unit;
  st.mm = put(blob, Mu, n * n);
  st.units = (double)std::pow(unit, D);
  // factor matrices M^-1 B^T W f B per position along an axis
  auto factor = [&](int axis, const double* v, double scale) {
    const int64_t at = (int64_t)blob.size();
    std::vector<double> f(q);
    for (int64_t e = 0; e < plan->desc.sizes[axis]; ++e) {
      for (int k = 0; k < q; ++k) f[k] = scale * v[e * (q + 2) + k];
      put(blob, times(gram(t1.B, f.data()), n), n * n);
    }
    return at;
  };

  // ---- sigma ----
  st.mass_ok = true;
  for (int r = 0; r < plan->sigma_host.rank && st.mass_ok; ++r) {
    const HostField& f = plan->sigma_host;
    std::vector<int> ax;
    for (int d = 0; d < D; ++d)
      if (f.offset[r][d] >= 0) ax.push_back(d);
    if (ax.empty()) {
      st.sigma_const += f.scale[r];
      continue;
    }
    if (ax.size() > 2 || st.mass.size() == 4) {
      st.mass_ok = false;
      break;
    }
    HostTerm t;
    t.a = ax[0];
    t.ta = factor(ax[0], f.data.data() + f.offset[r][ax[0]], f.scale[r]);
    t.b = ax.size() > 1 ? ax[1] : (ax[0] == 0 ? 1 : 0);
    if (ax.size() > 1) t.tb = factor(ax[1], f.data.data() + f.offset[r][ax[1]], 1.0);
    st.mass.push_back(t);
  }

  // ---- advection ----
  st.adv_ok = plan->beta_set && (plan->bc_mode == GD_BC_NONE || plan->bc_host.rank == 0 ||
                                 (plan->bc_host.rank == 1 && plan->bc_host.scale[0] == 0.0));
  for (int c = 0; c < D && st.adv_ok; ++c) {
    OneAxis f;
    if (!one_axis(plan, c, *ts, f)) {
      st.adv_ok = false;
      break;
    }
    // one sign on every face point: the rule points along the field's axis, or
    // its ends where that is the normal
    bool pos = false, neg = false, zero = true;
    if (f.axis < 0) {
      pos = f.v[0] > 0.0;
      neg = f.v[0] < 0.0;
      zero = f.v[0] == 0.0;
    } else {
      for (size_t i = 0; i < f.v.size(); ++i) {
        const int k = (int)(i % (q + 2));
        zero = zero && f.v[i] == 0.0;
        if (f.axis == c ? k < q : k >= q) continue;
        pos |= f.v[i] > 0.0;
        neg |= f.v[i] < 0.0;
      }
    }
    for (double v : f.v) st.adv_ok = st.adv_ok && std::isfinite(v);
    if ((pos && neg) || !st.adv_ok) {
      st.adv_ok = false;
      break;
    }
    if (zero) continue;
    const bool per = plan->desc.periodic[c];
    const int64_t Mc = plan->desc.sizes[c];
    HostTerm t;
    t.a = c;
    t.b = f.axis >= 0 && f.axis != c ? f.axis : (c == 0 ? 1 : 0);
    t.inflow = neg ? -1 : 1;
    t.scale = 1.0 / plan->desc.h[c];
    std::vector<double> fv;
    t.ta = (int64_t)blob.size();
    // a component that does not vary along its own axis has one matrix, and one
    // more at a boundary it skips
    Mat A, fc;
    bool same = false, was = false;
    for (int64_t e = 0; e < Mc; ++e) {
      const double* v = f.axis == c ? f.v.data() + e * (q + 2) : nullptr;
      const double cst = f.axis < 0 ? f.v[0] : 1.0;
      // own face at the outflow end: there with a neighbour or inflow data
      const bool own = per || plan->bc_mode != GD_BC_NONE || (neg ? e != 0 : e != Mc - 1);
      if (v || !same || own != was) {
        Mat m = gram(t1.Gb, v);
        for (Ext& s : m) s *= -cst;
        if (own) {
          const Table& be = neg ? t1.b0 : t1.b1;
          const double bo = (v ? v[neg ? q : q + 1] : 1.0) * cst * (neg ? -1.0 : 1.0);
          for (int i = 0; i < n; ++i)
            for (int j = 0; j < n; ++j) m[i * n + j] += bo * be[i] * be[j];
        }
        A = times(m, n);
        // inflow end: -beta b0 (lower face) or +beta b1 (upper face) on the neighbour's trace
        const double bi = (v ? v[neg ? q + 1 : q] : 1.0) * cst * (neg ? 1.0 : -1.0);
        Mat col{};
        for (int i = 0; i < n; ++i) col[i] = bi * (neg ? t1.b1[i] : t1.b0[i]);
        fc = times(col, 1);
        same = true;
        was = own;
      }
      put(blob, A, n * n);
      put(fv, fc, n);
    }
    t.tf = (int64_t)blob.size();
    blob.insert(blob.end(), fv.begin(), fv.end());
    if (f.axis >= 0 && f.axis != c) t.tb = factor(f.axis, f.v.data(), 1.0);
    st.adv.push_back(t);
  }
  if (!st.adv_ok && !st.mass_ok) return GD_OK;
  st.words = blob.size();
  if (st.words > st.capacity) {
    if (st.dev) (void)hipFree(st.dev);
    st.dev = nullptr;
    st.capacity = 0;
    const size_t want = std::max<size_t>(2 * st.words, 4096);
    if (hipMalloc(&st.dev, want * (sizeof(double) + sizeof(float))) != hipSuccess) {
      st.adv_ok = st.mass_ok = false;
      return fail(GD_ERR_ALLOC, "Kronecker tables: device allocation failed");
    }
    st.capacity = want;
  }
  std::vector<char> host(st.words * (sizeof(double) + sizeof(float)));
  std::memcpy(host.data(), blob.data(), st.words * sizeof(double));
  float* h32 = reinterpret_cast<float*>(host.data() + st.words * sizeof(double));
  for (size_t i = 0; i < st.words; ++i) h32[i] = (float)blob[i];
  const hipError_t err = hipMemcpy(st.dev, host.data(), host.size(), hipMemcpyHostToDevice);
  if (err != hipSuccess) {
    st.adv_ok = st.mass_ok = false;
    return hip_fail(err, "hipMemcpy");
  }
  return GD_OK;
}

bool available(const gd_plan* plan, bool adv, bool mass)
{
  const State* st = plan->kron_state;
  return st && (st->adv_ok || st->mass_ok) && (!adv || st->adv_ok) && (!mass || st->mass_ok);
}

template <typename T>
bool preferred(const gd_plan* plan, bool adv, bool mass)
{
  // Meshes of up to 64 elements stay on the generic kernel, which callers see as
  // their variant (tests/test_gpu_n2k.py states it for 2^6 elements); this kernel
  // would be faster there too (one element, advection, generic against this: 4D
  // n = 2 16 and 5.8 us, 6D n = 3 76 and 9.2; mass 5.3 and 5.5, 14 and 6).
  if (plan->E <= 64 || !available(plan, adv, mass)) return false;
  // Mass alone with a variable sigma and q = n: the generic kernel interpolates
  // little, and this one holds few elements of these sizes in a CU.  Generic
  // against this, sigma of two terms, us: FP64 4D n = 4 625 elements 8.5 and 8.3,
  // 1,080 9.1 and 9.7, 8,100 26 and 32, 50,176 124 and 176 (4,096 17 and 16); FP64
  // 4D n = 5 256 8.5 and 10, 1,080 11 and 11, 2,058 19 and 16; FP32 5D n = 4 625
  // 10.4 and 10.6, 2,058 20 and 24, 20,736 132 and 140.  All others gain at every
  // size.
  const int n = plan->desc.order + 1;
  if (!adv && plan->desc.num_quad == n && !plan->kron_state->mass.empty()) {
    if (sizeof(T) == 8 && plan->dim == 4 && n == 4) return plan->E < 1000;
    if (sizeof(T) == 8 && plan->dim == 4 && n == 5) return plan->E >= 1000;
    if (sizeof(T) == 4 && plan->dim == 5 && n == 4) return plan->E < 1000;
  }
  return true;
}

template bool preferred<double>(const gd_plan*, bool, bool);
template bool preferred<float>(const gd_plan*, bool, bool);

template <typename T>
int apply(const gd_plan* plan, T mass_coef, T adv_coef, const T* x, T* y, hipStream_t s)
{
  const bool adv = adv_coef != T(0), mass = mass_coef != T(0);
  if (!available(plan, adv, mass)) return GD_ERR_UNSUPPORTED;
  const Entry* en = find(plan);
  const State& st = *plan->kron_state;
  const TableSet* ts = find_tables(plan, plan->desc.order + 1, plan->desc.num_quad);
  const int D = plan->dim, n = plan->desc.order + 1;
  Args<T> a;
  const T* base;
  const Tables1D<T>* tab;
  if constexpr (std::is_same_v<T, double>) {
    base = st.f64();
    tab = &ts->once64;
  } else {
    base = st.f32();
    tab = &ts->t32;
  }
  a.E = (int)plan->E;
  a.periodic_mask = 0;
  double detJ = 1.0;
  for (int d = 0; d < D; ++d) {
    a.M[d] = (int)plan->desc.sizes[d];
    if (d < 5) a.dv[d] = pl::fast_div(a.M[d]);
    if (plan->desc.periodic[d]) a.periodic_mask |= 1 << d;
    detJ *= plan->desc.h[d];
  }
  detJ *= st.units;
  a.km = mass ? (double)mass_coef * detJ * st.sigma_const : 0.0;
  a.Mm = st.f64() + st.mm;
  a.b0 = tab->b0;
  a.b1 = tab->b1;
  a.nterms = 0;
  auto add = [&](const HostTerm& h, double coef) {
    Term<T>& t = a.t[a.nterms];
    a.coef[a.nterms++] = (T)(coef * detJ * h.scale);
    t.a = h.a;
    t.b = h.b;
    t.inflow = h.inflow;
    t.ta = base + h.ta;
    t.tb = h.tb >= 0 ? base + h.tb : nullptr;
    t.tf = h.tf >= 0 ? base + h.tf : nullptr;
    int k = 0, st_ = 1;
    for (int d = 0; d < D; ++d) {
      if (d == h.a) t.stride[D - 2] = st_;
      else if (d == h.b) t.stride[D - 1] = st_;
      else t.stride[k++] = st_;
      st_ *= n;
    }
  };
  if (adv)
    for (const HostTerm& h : st.adv) add(h, (double)adv_coef);
  if (mass)
    for (const HostTerm& h : st.mass) add(h, (double)mass_coef);
  const bool gll = plan->desc.basis == GD_BASIS_GLL;
  if constexpr (std::is_same_v<T, double>) return en->f64(a, gll, x, y, s);
  else return en->f32(a, gll, x, y, s);
}

template int apply<double>(const gd_plan*, double, double, const double*, double*, hipStream_t);
template int apply<float>(const gd_plan*, float, float, const float*, float*, hipStream_t);

}  // namespace kron
}  // namespace gd
