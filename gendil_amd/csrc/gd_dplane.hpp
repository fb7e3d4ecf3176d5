// gfx950 kernel of the 3D SIPDG diffusion apply, one z-plane of rule points per
// thread (gd_plane.hpp describes the layout and the three phases; what is
// computed is gd_diff.hpp's).
//
// The volume term of plane kz needs B_z u and B'_z u of the element's pencils;
// x and y derivatives are taken and tested in registers.  Both sides of a face
// enter its fluxes only through the jump J = u - u_nb and the sum
// S = du/dn + du_nb/dn (reference derivatives along the axis; at a boundary
// J = u, S = 2 du/dn), so phase 1 forms J and S at the face's nodes and one
// pair is interpolated per face instead of four traces:
//   Du = w detJ mu / h^2 (kappa J -+ S / 2)   tested with the basis values
//   DG = +- w detJ mu / h^2 sigma J / 2       tested with the derivatives
// (upper signs: upper face; DG without the 1/2 at a boundary).
//
// Record of a cell plane: B_z u, B'_z u, then J and S of the four x and y faces
// (z-contracted, n values each); of a z face: J, S.  The outputs overwrite the
// first two fields.
//
// 64^3, p = 3, q = 5, an eight-term diffusivity, FP64: 441 us against 940 us for
// the generic diffusion kernel (every contraction through LDS); 27 x 23 x 19,
// p = 2, q = 4, FP32: 9.4 against 25.9 us.  Bound by waits at six waves a CU
// (4 KB of LDS per element; 197 us of VALU issue): with two cell waves a block
// and one block a CU the first took 685 us; with the diffusivity read term by
// term as each is added 477 us.
#pragma once

#include "gd_plane.hpp"

namespace gd {
namespace pl {

template <typename T>
struct DArgs {
  int E, epb, num_blocks;
  int row0, row1, spitch;
  Field mu;
  FastDiv d0, d1;
  int M[3];
  int periodic_mask;
  int gll;
  T c[3];  // detJ / h^2
  T sigma, kappa;
  const FieldTerms<T>* terms;
  const T *B, *Gb, *b0, *b1, *e0, *e1, *w;  // e0, e1: basis derivatives at the element ends
};

// The diffusivity's row samples of an element, staged in LDS times the weights
// of the rule points: a missing row is the weights, the end samples carry none.
template <typename T, int Q>
struct MuRows {
  const T* sm;
  CPtr<T> w;
  // samples 0..Q of a row
  __device__ __forceinline__ void line(int has, int row, T (&v)[Q]) const
  {
#pragma unroll
    for (int k = 0; k < Q; ++k) v[k] = w[k];
    if (has) {
#pragma unroll
      for (int k = 0; k < Q; ++k) v[k] = sm[row * (Q + 2) + k];
    }
  }
  // the end samples of a row
  __device__ __forceinline__ void ends(int has, int row, T (&v)[2]) const
  {
    v[0] = v[1] = T(1);
    if (has) {
      v[0] = sm[row * (Q + 2) + Q];
      v[1] = sm[row * (Q + 2) + Q + 1];
    }
  }
  // sample k, which may be an end (Q, Q + 1); wk: its weight
  __device__ __forceinline__ T one(int has, int row, int k, T wk) const
  {
    T v = wk;
    if (has) v = sm[row * (Q + 2) + k];
    return v;
  }
};

// Samples of rows [row0, row1) at the block's ne elements into smp (pitch per
// element), four loads in flight, times the rule's weights.
template <typename T, int Q, int NT, class Decode>
__device__ __forceinline__ void stage_rows(CPtr<FieldTerms<T>> ft, int row0, int row1, CPtr<T> w, T* smp, int pitch, int ne, Decode&& decode)
{
  for (int t = threadIdx.x; t < ne * (Q + 2); t += NT) {
    const int el = t / (Q + 2), k = t - el * (Q + 2);
    int sub[3];
    decode(el, sub);
    const T wk = k < Q ? w[k] : T(1);
    T* dst = smp + el * pitch + k;
    for (int f = row0; f < row1; f += 4) {
      T v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int g = f + i < row1 ? f + i : f;  // past the end: the first again
        const int ax = ft->axis[g];
        const int pos = ax == 0 ? sub[0] : (ax == 1 ? sub[1] : (ax == 2 ? sub[2] : 0));
        v[i] = ((GPtr<T>)ft->tab[g])[pos * (Q + 2) + k];
        if (ax == kRowConstant) v[i] = T(1);
        v[i] *= ft->scale[g] * wk;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f + i < row1) dst[(f + i - row0) * (Q + 2)] = v[i];
    }
  }
}

template <typename T, int Q>
struct Diffusivity {
  // One term's samples in a plane.
  struct Term {
    T X[Q], y[Q], z, xe[2], ye[2];
  };

  // f at the points of a plane of sample kz (of weight wz), and (FX, FY) on its
  // lines at the ends of x (points along y) and of y (points along x), times
  // the weights where the rows have them.  The next term's samples are read
  // while one is added: a term's products are about an LDS latency long.
  template <bool FX, bool FY, class Rows>
  __device__ __forceinline__ static void evaluate(const Field& f, const Rows& rows, int kz, T wz, T (&b)[Q][Q],
                                                  T (&bx)[2][Q], T (&by)[2][Q])
  {
    int row = f.row, m = f.mask;
    auto load = [&](Term& t) {
      const int rx = row, ry = rx + (m & 1), rz = ry + ((m >> 1) & 1);
      row = rz + ((m >> 2) & 1);
      rows.line(m & 1, rx, t.X);
      rows.line(m & 2, ry, t.y);
      t.z = rows.one(m & 4, rz, kz, wz);
      if constexpr (FX) rows.ends(m & 1, rx, t.xe);
      if constexpr (FY) rows.ends(m & 2, ry, t.ye);
      m >>= 3;
    };
    auto use = [&](const Term& t, bool first) {
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        const T a = t.y[k] * t.z;
#pragma unroll
        for (int j = 0; j < Q; ++j) b[k][j] = first ? a * t.X[j] : mad(a, t.X[j], b[k][j]);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if constexpr (FX) {
          const T e = t.xe[s] * t.z;
#pragma unroll
          for (int k = 0; k < Q; ++k) bx[s][k] = first ? e * t.y[k] : mad(e, t.y[k], bx[s][k]);
        }
        if constexpr (FY) {
          const T e = t.ye[s] * t.z;
#pragma unroll
          for (int k = 0; k < Q; ++k) by[s][k] = first ? e * t.X[k] : mad(e, t.X[k], by[s][k]);
        }
      }
    };
    if (f.rank == 0) {
#pragma unroll
      for (int k = 0; k < Q; ++k) {
#pragma unroll
        for (int j = 0; j < Q; ++j)
          b[k][j] = T(0);
        if constexpr (FX) bx[0][k] = bx[1][k] = T(0);
        if constexpr (FY) by[0][k] = by[1][k] = T(0);
      }
      return;
    }
    Term t, n;
    load(t);
    if (f.rank > 1) load(n);
    use(t, true);
#pragma unroll 1
    for (int r = 1; r < f.rank; r += 2) {
      if (r + 1 < f.rank) load(t);
      use(n, false);
      if (r + 1 >= f.rank) break;
      if (r + 2 < f.rank) load(n);
      use(t, false);
    }
  }
};

template <int N, int Q>
struct DGeo {
  static constexpr int NN = N * N;
  static constexpr int PITCH = (2 * NN + 8 * N) | 1;  // cell plane
  static constexpr int ZPITCH = (2 * NN) | 1;         // z face
  static constexpr int PER = Q * PITCH + 2 * ZPITCH;
  static constexpr int EPB = 64 / Q;  // cell planes fill one wave, the z faces most of another
  static constexpr int NT = 128;
};

template <typename T, int N, int Q, bool GLL>
__global__ void __launch_bounds__((DGeo<N, Q>::NT)) __attribute__((amdgpu_waves_per_eu(2)))
    diff_plane_kernel(DArgs<T> a, const T* __restrict__ x, T* __restrict__ y)
{
  using G = DGeo<N, Q>;
  using P = Planes<T, N, Q>;
  constexpr int NN = G::NN, ND = NN * N, PITCH = G::PITCH, ZPITCH = G::ZPITCH, NT = G::NT;

  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* rec = reinterpret_cast<T*>(smem_raw);      // [element][plane]
  T* zrec = rec + a.epb * Q * PITCH;            // [element][lower, upper]
  T* smp = zrec + a.epb * 2 * ZPITCH;           // the diffusivity's row samples

  const int blk = dev::xcd_remap(blockIdx.x, a.num_blocks);
  const int e0 = blk * a.epb;
  const int ne = a.E - e0 < a.epb ? a.E - e0 : a.epb;
  const int tid = threadIdx.x;
  const Half<T, N, Q, 1> B(a.B);
  const Half<T, N, Q, -1> Gb(a.Gb);
  CPtr<T> b0 = (CPtr<T>)a.b0;
  CPtr<T> b1 = (CPtr<T>)a.b1;
  CPtr<T> g0 = (CPtr<T>)a.e0;
  CPtr<T> g1 = (CPtr<T>)a.e1;
  CPtr<T> w = (CPtr<T>)a.w;

  auto decode = [&](int e, int* sub) {
    const int q0 = div(a.d0, e), q1 = div(a.d1, q0);
    sub[0] = e - q0 * a.M[0];
    sub[1] = q0 - q1 * a.M[1];
    sub[2] = q1;
  };
  auto neighbour = [&](int e, const int* sub, int d, int side) {
    const int stride = d == 0 ? 1 : (d == 1 ? a.M[0] : a.M[0] * a.M[1]);
    const int M = d == 0 ? a.M[0] : (d == 1 ? a.M[1] : a.M[2]);
    const int s = d == 0 ? sub[0] : (d == 1 ? sub[1] : sub[2]);
    const bool per = (a.periodic_mask >> d) & 1;
    if (side == 0) return s > 0 ? e - stride : (per ? e + (M - 1) * stride : -1);
    return s < M - 1 ? e + stride : (per ? e - (M - 1) * stride : -1);
  };
  // jump and derivative sum of a face pencil: own and neighbour values along
  // the normal (nb < 0: boundary, whose neighbour values are not used)
  auto jump_sum = [&](const T (&own)[N], const T (&nbv)[N], bool upper, bool bnd, T& J, T& S) {
    T ov, nv, og = T(0), ng = T(0);
    if constexpr (GLL) {
      ov = upper ? own[N - 1] : own[0];
      nv = upper ? nbv[0] : nbv[N - 1];
    } else {
      ov = nv = T(0);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        ov += (upper ? b1[i] : b0[i]) * own[i];
        nv += (upper ? b0[i] : b1[i]) * nbv[i];
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      og += (upper ? g1[i] : g0[i]) * own[i];
      ng += (upper ? g0[i] : g1[i]) * nbv[i];
    }
    J = bnd ? ov : ov - nv;
    S = og + (bnd ? og : ng);
  };

  // ---- phase 1 ----
  for (int t = tid; t < ne * NN; t += NT) {
    const int el = t / NN, c = t - el * NN;
    const int e = e0 + el;
    int sub[3];
    decode(e, sub);
    const int lo = neighbour(e, sub, 2, 0), hi = neighbour(e, sub, 2, 1);
    const T* src = x + (int64_t)e * ND + c;
    const T* pl = x + (int64_t)(lo >= 0 ? lo : e) * ND + c;
    const T* ph = x + (int64_t)(hi >= 0 ? hi : e) * ND + c;
    T u[N], l[N], h[N], v[Q];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      u[i] = src[i * NN];
      l[i] = pl[i * NN];
      h[i] = ph[i * NN];
    }
    T* r = rec + el * Q * PITCH + c;
    P::up(B, u, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
    P::up(Gb, u, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH + NN] = v[q];
    T* z = zrec + el * 2 * ZPITCH + c;
    T J, S;
    jump_sum(u, l, false, lo < 0, J, S);
    z[0] = J;
    z[NN] = S;
    jump_sum(u, h, true, hi < 0, J, S);
    z[ZPITCH] = J;
    z[ZPITCH + NN] = S;
  }
  for (int t = tid; t < ne * 4 * N; t += NT) {
    const int el = t / (4 * N), c = t - el * (4 * N);
    const int f = c / N, m = c - f * N;  // faces -x, +x, -y, +y; tangential node
    const int e = e0 + el;
    int sub[3];
    decode(e, sub);
    const int ax = f >> 1;
    const bool upper = f & 1;
    const int nb = neighbour(e, sub, ax, upper);
    const int norm = ax == 0 ? 1 : N, tang = ax == 0 ? m * N : m;
    const T* src = x + (int64_t)e * ND + tang;
    const T* oth = x + (int64_t)(nb >= 0 ? nb : e) * ND + tang;
    T own[N][N], nbv[N][N], J[N], S[N], v[Q];
#pragma unroll
    for (int z = 0; z < N; ++z)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        own[z][i] = src[z * NN + i * norm];
        nbv[z][i] = oth[z * NN + i * norm];
      }
#pragma unroll
    for (int z = 0; z < N; ++z) jump_sum(own[z], nbv[z], upper, nb < 0, J[z], S[z]);
    T* r = rec + el * Q * PITCH + 2 * NN + 2 * f * N + m;
    P::up(B, J, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
    P::up(B, S, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH + N] = v[q];
  }
  stage_rows<T, Q, NT>((CPtr<FieldTerms<T>>)a.terms, a.row0, a.row1, w, smp, a.spitch, ne,
                       [&](int el, int* sub) { decode(e0 + el, sub); });
  __syncthreads();

  // adds the tested row g of point row k: out[m][i] += tab(k, m) g[i]
  auto add = [&](T (&out)[N][N], const auto& tab, int k, const T (&g)[N]) {
#pragma unroll
    for (int m = 0; m < N; ++m)
#pragma unroll
      for (int i = 0; i < N; ++i) out[m][i] = mad(tab(k, m), g[i], out[m][i]);
  };
  // fluxes of one face point: cm = w mu detJ / h^2
  auto fluxes = [&](T cm, T J, T S, bool upper, bool bnd, T& du, T& dg) {
    const T hs = T(0.5) * S, sj = (bnd ? a.sigma : T(0.5) * a.sigma) * J;
    du = cm * (upper ? a.kappa * J - hs : a.kappa * J + hs);
    dg = cm * (upper ? sj : -sj);
  };

  // ---- phase 2: one plane per thread ----
  if (tid < 64) {
    for (int t = tid; t < ne * Q; t += 64) {
      const int el = t / Q, kz = t - el * Q;
      const int e = e0 + el;
      int sub[3];
      decode(e, sub);
      T* r = rec + (el * Q + kz) * PITCH;
      const MuRows<T, Q> rows{smp + el * a.spitch, w};
      const T wz = ((GPtr<T>)a.w)[kz];
      T b[Q][Q], u[N][N], A[N][N];
      T mx[2][Q], my[2][Q];
      Diffusivity<T, Q>::template evaluate<true, true>(a.mu, rows, kz, wz, b, mx, my);
      // z derivative: tested with B' in z, kept apart
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = r[NN + m * N + i];
          A[m][i] = T(0);
        }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        T g[N], f[Q];
        pin(A);
        pin(u);
        P::row(B, u, k, g);
        P::up(B, g, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] *= a.c[2] * b[k][j];
        P::down(B, f, g);
        add(A, B, k, g);
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          r[NN + m * N + i] = A[m][i];
          u[m][i] = r[m * N + i];
          A[m][i] = T(0);
        }
      // x faces at the plane's rows
      T fu[2][Q], fg[2][Q];
      {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          T nd[N], J[Q], S[Q];
#pragma unroll
          for (int m = 0; m < N; ++m) nd[m] = r[2 * NN + 2 * s * N + m];
          P::up(B, nd, J);
#pragma unroll
          for (int m = 0; m < N; ++m) nd[m] = r[2 * NN + (2 * s + 1) * N + m];
          P::up(B, nd, S);
          const bool bnd = neighbour(e, sub, 0, s) < 0;
#pragma unroll
          for (int k = 0; k < Q; ++k) fluxes(a.c[0] * mx[s][k], J[k], S[k], s, bnd, fu[s][k], fg[s][k]);
          pin(fu[s]);
          pin(fg[s]);
        }
      }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        T g[N], f[Q];
        pin(A);
        pin(u);
        P::row(B, u, k, g);
        P::up(Gb, g, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] *= a.c[0] * b[k][j];
        P::down(Gb, f, g);
        if constexpr (GLL) {
          g[0] += fu[0][k];
          g[N - 1] += fu[1][k];
        } else {
#pragma unroll
          for (int i = 0; i < N; ++i) g[i] += b0[i] * fu[0][k] + b1[i] * fu[1][k];
        }
#pragma unroll
        for (int i = 0; i < N; ++i) g[i] += g0[i] * fg[0][k] + g1[i] * fg[1][k];
        add(A, B, k, g);
      }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        T g[N], f[Q];
        pin(A);
        pin(u);
        P::row(Gb, u, k, g);
        P::up(B, g, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] *= a.c[1] * b[k][j];
        P::down(B, f, g);
        add(A, Gb, k, g);
      }
      {  // y faces: two more rows
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          T nd[N], J[Q], S[Q], du[Q], dg[Q], gu[N], gg[N];
          pin(A);
#pragma unroll
          for (int i = 0; i < N; ++i) nd[i] = r[2 * NN + (4 + 2 * s) * N + i];
          P::up(B, nd, J);
#pragma unroll
          for (int i = 0; i < N; ++i) nd[i] = r[2 * NN + (5 + 2 * s) * N + i];
          P::up(B, nd, S);
          const bool bnd = neighbour(e, sub, 1, s) < 0;
#pragma unroll
          for (int j = 0; j < Q; ++j) fluxes(a.c[1] * my[s][j], J[j], S[j], s, bnd, du[j], dg[j]);
          P::down(B, du, gu);
          P::down(B, dg, gg);
#pragma unroll
          for (int m = 0; m < N; ++m)
#pragma unroll
            for (int i = 0; i < N; ++i) {
              A[m][i] += (s ? g1[m] : g0[m]) * gg[i];
              if constexpr (!GLL) A[m][i] += (s ? b1[m] : b0[m]) * gu[i];
            }
          if constexpr (GLL) {
#pragma unroll
            for (int i = 0; i < N; ++i) A[s ? N - 1 : 0][i] += gu[i];
          }
        }
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) r[m * N + i] = A[m][i];
    }
  } else {
    for (int t = tid - 64; t < ne * 2; t += 64) {
      const int el = t >> 1;
      const bool s = t & 1;
      const int e = e0 + el;
      int sub[3];
      decode(e, sub);
      T* r = zrec + (el * 2 + s) * ZPITCH;
      const MuRows<T, Q> rows{smp + el * a.spitch, w};
      const bool bnd = neighbour(e, sub, 2, s) < 0;
      T b[Q][Q], u[N][N], A[N][N];
      T no[2][Q];
      Diffusivity<T, Q>::template evaluate<false, false>(a.mu, rows, Q + s, T(1), b, no, no);
      // du = c mu (kappa J -+ S / 2): one combination of the node values, as the
      // interpolation is linear; then DG from J alone
      const T hs = s ? T(-0.5) : T(0.5);
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = a.kappa * r[m * N + i] + hs * r[NN + m * N + i];
          A[m][i] = T(0);
        }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        T g[N], f[Q];
        pin(A);
        pin(u);
        P::row(B, u, k, g);
        P::up(B, g, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] *= a.c[2] * b[k][j];
        P::down(B, f, g);
        add(A, B, k, g);
      }
      const T sj = (bnd ? a.sigma : T(0.5) * a.sigma) * (s ? a.c[2] : -a.c[2]);
      T* out = r + NN;  // S is consumed
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = r[m * N + i];
          r[m * N + i] = A[m][i];
          A[m][i] = T(0);
        }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        T g[N], f[Q];
        pin(A);
        pin(u);
        P::row(B, u, k, g);
        P::up(B, g, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] *= sj * b[k][j];
        P::down(B, f, g);
        add(A, B, k, g);
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) out[m * N + i] = A[m][i];
    }
  }
  __syncthreads();

  // ---- phase 3: z test functions ----
  for (int t = tid; t < ne * NN; t += NT) {
    const int el = t / NN, c = t - el * NN;
    const T* r = rec + el * Q * PITCH + c;
    const T* z = zrec + el * 2 * ZPITCH + c;
    T f[Q], o[N], o2[N];
#pragma unroll
    for (int q = 0; q < Q; ++q) f[q] = r[q * PITCH];
    P::down(B, f, o);
#pragma unroll
    for (int q = 0; q < Q; ++q) f[q] = r[q * PITCH + NN];
    P::down(Gb, f, o2);
    const T ul = z[0], gl = z[NN], uh = z[ZPITCH], gh = z[ZPITCH + NN];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      o[i] += o2[i] + g0[i] * gl + g1[i] * gh;
      if constexpr (!GLL) o[i] += b0[i] * ul + b1[i] * uh;
    }
    if constexpr (GLL) {
      o[0] += ul;
      o[N - 1] += uh;
    }
    T* dst = y + (int64_t)(e0 + el) * ND + c;
#pragma unroll
    for (int i = 0; i < N; ++i) dst[i * NN] = o[i];
  }
}

template <typename T, int N, int Q, bool GLL>
int launch_diff_kind(DArgs<T>& a, const T* x, T* y, hipStream_t s)
{
  using G = DGeo<N, Q>;
  a.spitch = ((a.row1 - a.row0) * (Q + 2)) | 1;
  const size_t per = (size_t)(G::PER + a.spitch) * sizeof(T);
  a.epb = G::EPB;
  // as many blocks as CUs can take even on small meshes
  while (a.epb > 2 && ((int64_t)a.epb * 512 > a.E || (size_t)a.epb * per > 80 * 1024)) a.epb = (a.epb + 1) / 2;
  a.num_blocks = (int)((a.E + a.epb - 1) / a.epb);
  const size_t lds = a.epb * per;
  auto kern = diff_plane_kernel<T, N, Q, GLL>;
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

template <typename T, int N, int Q>
int launch_diff(DArgs<T>& a, const T* x, T* y, hipStream_t s)
{
  return a.gll ? launch_diff_kind<T, N, Q, true>(a, x, y, s) : launch_diff_kind<T, N, Q, false>(a, x, y, s);
}

}  // namespace pl
}  // namespace gd
