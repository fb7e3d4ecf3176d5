// gfx950 kernels of the adjoint of the 3D advection apply with a per-point
// field (FP64), one z-plane of rule points per thread as in gd_plane.hpp:
//   transpose_plane_kernel  z = (mass_coef M + adv_coef A)^T r
//   grad_plane_kernel       d<r, adv_coef A(beta) u> / d beta
// (gd_kernels.hpp states both; no reference counterpart).
//
// The transpose takes gradients at the points and tests with the basis only, so
// a plane reads B_z r and B'_z r and returns one set of n^2 values.  The
// gradient needs B u, and B r and its three derivatives, at the points; a plane
// keeps them in registers, and its 3 q^2 results replace the record it read, so
// that they leave in consecutive order (written from the planes they would be
// 200-byte runs, one per lane).
//
// 48^3, p = 4, q = 5 (619 MB of vectors and field per kernel): transpose 223 us,
// gradient 282 us, against 450 and 660 us for the generic kernel (and the
// forward apply of the same field on the plane kernel 206 against 450 us).
// Bound by waits: the 200-byte lane runs of the field reads (139 of 199 million
// wave-quads wait) at four to six waves a CU.
#pragma once

#include "gd_plane.hpp"

namespace gd {
namespace pl {

struct AdjArgs {
  int E, epb, num_blocks;
  FastDiv d0, d1;
  int M[3];
  int periodic_mask;
  int gll, bc_none, bc_data;
  double c[3];  // adv_coef detJ / h
  double mass;  // mass_coef detJ
  const double *beta_cell, *beta_face[3];
  const double *B, *Gb, *b0, *b1, *w;
  const FieldDev<double>* sigma;
  const FieldDev<double>* bc;
  double *dcell, *dface[3];
};

template <int N, int Q>
struct AdjGeo {
  static constexpr int NN = N * N, QQ = Q * Q;
  // transpose: B_z r, B'_z r, the neighbours' four pencils
  static constexpr int TP = (2 * NN + 4 * N) | 1, TZ = (2 * NN) | 1;
  // gradient: B_z u, B_z r, B'_z r, two lower neighbours' pencils of u and r; 3 q^2 results
  static constexpr int GIN = 3 * NN + 4 * N;
  static constexpr int GP = (GIN > 3 * QQ ? GIN : 3 * QQ) | 1, GZ = (4 * NN) | 1;
  static constexpr int EPB = 64 / Q;
  static constexpr int NT = 128;
};

// element and neighbour arithmetic of a block
struct AdjMesh {
  const AdjArgs& a;
  __device__ __forceinline__ void decode(int e, int* sub) const
  {
    const int q0 = div(a.d0, e), q1 = div(a.d1, q0);
    sub[0] = e - q0 * a.M[0];
    sub[1] = q0 - q1 * a.M[1];
    sub[2] = q1;
  }
  __device__ __forceinline__ int neighbour(int e, const int* sub, int d, int side) const
  {
    const int stride = d == 0 ? 1 : (d == 1 ? a.M[0] : a.M[0] * a.M[1]);
    const int M = d == 0 ? a.M[0] : (d == 1 ? a.M[1] : a.M[2]);
    const int s = d == 0 ? sub[0] : (d == 1 ? sub[1] : sub[2]);
    const bool per = (a.periodic_mask >> d) & 1;
    if (side == 0) return s > 0 ? e - stride : (per ? e + (M - 1) * stride : -1);
    return s < M - 1 ? e + stride : (per ? e - (M - 1) * stride : -1);
  }
};

// trace of pencil v at the element's lower (0) or upper (1) end
template <int N, bool GLL>
__device__ __forceinline__ double end_of(const double (&v)[N], int end, CPtr<double> b0, CPtr<double> b1)
{
  if constexpr (GLL) return end ? v[N - 1] : v[0];
  else {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) s += (end ? b1[i] : b0[i]) * v[i];
    return s;
  }
}

// the z pencil at tangential node m on side `side` (the side facing us) of
// element nb's face normal to axis ax (0: x, 1: y), zeros if nb < 0
template <int N, bool GLL>
__device__ __forceinline__ void face_pencil(const double* x, int nb, int ax, int m, int end, CPtr<double> b0,
                                            CPtr<double> b1, double (&out)[N])
{
  constexpr int NN = N * N;
  const int norm = ax == 0 ? 1 : N, tang = ax == 0 ? m * N : m;
  const double* src = x + (int64_t)(nb >= 0 ? nb : 0) * (NN * N) + tang;
  if constexpr (GLL) {
    src += end ? (N - 1) * norm : 0;
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = src[i * NN];
  } else {
    double l[N][N];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int k = 0; k < N; ++k) l[i][k] = src[i * NN + k * norm];
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = end_of<N, false>(l[i], end, b0, b1);
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (nb < 0) out[i] = 0.0;
}

template <int N, int Q, bool GLL>
__global__ void __launch_bounds__((AdjGeo<N, Q>::NT)) __attribute__((amdgpu_waves_per_eu(2)))
    transpose_plane_kernel(AdjArgs a, const double* __restrict__ x, double* __restrict__ y)
{
  using G = AdjGeo<N, Q>;
  using P = Planes<double, N, Q>;
  constexpr int NN = G::NN, QQ = G::QQ, ND = NN * N, NT = G::NT, PITCH = G::TP, ZP = G::TZ;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* rec = reinterpret_cast<double*>(smem_raw);  // [element][plane]
  double* zrec = rec + a.epb * Q * PITCH;             // [element][lower, upper]
  const AdjMesh mesh{a};
  const int blk = dev::xcd_remap(blockIdx.x, a.num_blocks);
  const int e0 = blk * a.epb;
  const int ne = a.E - e0 < a.epb ? a.E - e0 : a.epb;
  const int tid = threadIdx.x;
  const Half<double, N, Q, 1> B(a.B);
  const Half<double, N, Q, -1> Gb(a.Gb);
  CPtr<double> b0 = (CPtr<double>)a.b0;
  CPtr<double> b1 = (CPtr<double>)a.b1;
  CPtr<double> w = (CPtr<double>)a.w;

  // ---- phase 1 ----
  for (int t = tid; t < ne * NN; t += NT) {
    const int el = t / NN, c = t - el * NN, e = e0 + el;
    int sub[3];
    mesh.decode(e, sub);
    const int lo = mesh.neighbour(e, sub, 2, 0), hi = mesh.neighbour(e, sub, 2, 1);
    double u[N], v[Q], nlo, nhi;
    const double* src = x + (int64_t)e * ND + c;
    const double* pl = x + (int64_t)(lo >= 0 ? lo : e) * ND + c;
    const double* ph = x + (int64_t)(hi >= 0 ? hi : e) * ND + c;
#pragma unroll
    for (int i = 0; i < N; ++i) u[i] = src[i * NN];
    if constexpr (GLL) {
      nlo = pl[(N - 1) * NN];
      nhi = ph[0];
    } else {
      double l[N], h[N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        l[i] = pl[i * NN];
        h[i] = ph[i * NN];
      }
      nlo = end_of<N, GLL>(l, 1, b0, b1);
      nhi = end_of<N, GLL>(h, 0, b0, b1);
    }
    double* r = rec + el * Q * PITCH + c;
    P::up(B, u, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
    P::up(Gb, u, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH + NN] = v[q];
    double* z = zrec + el * 2 * ZP + c;
    z[0] = end_of<N, GLL>(u, 0, b0, b1);
    z[NN] = lo >= 0 ? nlo : 0.0;
    z[ZP] = end_of<N, GLL>(u, 1, b0, b1);
    z[ZP + NN] = hi >= 0 ? nhi : 0.0;
  }
  for (int t = tid; t < ne * 4 * N; t += NT) {
    const int el = t / (4 * N), c = t - el * (4 * N);
    const int f = c / N, m = c - f * N, e = e0 + el;  // faces -x, +x, -y, +y; tangential node
    int sub[3];
    mesh.decode(e, sub);
    double u[N], v[Q];
    face_pencil<N, GLL>(x, mesh.neighbour(e, sub, f >> 1, f & 1), f >> 1, m, 1 - (f & 1), b0, b1, u);
    P::up(B, u, v);
    double* r = rec + el * Q * PITCH + 2 * NN + c;
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
  }
  __syncthreads();

  // Which values of dot = beta . n give a face its flux: on an inner face all but
  // the negative (what is not a number stays so), at the boundary the positive
  // only, without data none.  Kept as the face's floating-point classes (the sign
  // bit marks the boundary) or as a flag, whichever leaves the registers better
  // off.  Transpose with the classes and with the flag, us: 80^3, n = 2, q = 3 137
  // and 141; 64^3, n = 3, q = 5 353 and 336; 56^3, n = 4, q = 6 362 and 380; 48^3, n =
  // 5, q = 5 218 and 217 (with the rule where the field is read 258: its loads are
  // waited for there).  Conditions that branch around the flux gain up to 16 % on
  // large meshes of n < 5, but cost 8 to 16 % on 12^3 elements and a third at n = 5.
  auto face_rule = [&](int nb) {
    constexpr int nan = 0x3, zero = 0x60, positive = 0x380;
    if constexpr (N % 2 == 0) return nb >= 0 ? nan | zero | positive : (a.bc_none ? 0 : positive) | (1 << 31);
    else return nb < 0;
  };
  // the flux of one face point that this side's test function collects: outflow
  // c dot (own - nb), as the neighbour tests its inflow with -dot
  auto flux = [&](double c, double beta, bool upper, auto rule, double own, double nb) {
    const double dot = upper ? beta : -beta;
    if constexpr (N % 2 == 0) {
      const double v = rule < 0 ? own : own - nb;
      return __builtin_amdgcn_class(dot, rule) ? c * dot * v : 0.0;
    } else {
      const double v = own - nb;  // nb is 0 at the boundary
      const bool skip = (rule && a.bc_none) | (rule & (dot != dot));
      return !(dot <= 0.0) & !skip ? c * dot * v : 0.0;
    }
  };

  // ---- phase 2 ----
  if (tid < 64) {
    for (int t = tid; t < ne * Q; t += 64) {
      const int el = t / Q, kz = t - el * Q, e = e0 + el;
      int sub[3];
      mesh.decode(e, sub);
      double* r = rec + (el * Q + kz) * PITCH;
      const double wz = ((GPtr<double>)a.w)[kz];
      const double* bc = a.beta_cell + (int64_t)e * (3 * Q * QQ) + kz * QQ;
      double u[N][N], d[N][N], A[N][N];
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = r[m * N + i];
          d[m][i] = r[NN + m * N + i];
          A[m][i] = 0.0;
        }
      double xn[2][Q];  // the x neighbours' traces at the rows
      double fx[2][Q];  // beta on the x faces
      decltype(face_rule(0)) xr[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const double* src = a.beta_face[0] + face_index(a, sub, 0, s) * QQ + kz * Q;
#pragma unroll
        for (int k = 0; k < Q; ++k) fx[s][k] = src[k];
        double nd[N];
#pragma unroll
        for (int m = 0; m < N; ++m) nd[m] = r[2 * NN + s * N + m];
        P::up(B, nd, xn[s]);
        xr[s] = face_rule(mesh.neighbour(e, sub, 0, s));
      }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        double bx[Q], by[Q], bz[Q], t0[N], t1[N], g[Q], f[Q], o[N];
#pragma unroll
        for (int j = 0; j < Q; ++j) {
          bx[j] = bc[k * Q + j];
          by[j] = bc[Q * QQ + k * Q + j];
          bz[j] = bc[2 * Q * QQ + k * Q + j];
        }
        pin(A);
        pin(u);
        P::row(B, u, k, t0);
        P::up(Gb, t0, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] *= -a.c[0] * bx[j];
        P::row(Gb, u, k, t1);
        P::up(B, t1, g);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] -= a.c[1] * by[j] * g[j];
        pin(d);
        P::row(B, d, k, t1);
        P::up(B, t1, g);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] = (f[j] - a.c[2] * bz[j] * g[j]) * (wz * w[k] * w[j]);
        P::down(B, f, o);
        const double cw = a.c[0] * wz * w[k];
        const double lo = flux(cw, fx[0][k], false, xr[0], end_of<N, GLL>(t0, 0, b0, b1), xn[0][k]);
        const double hi = flux(cw, fx[1][k], true, xr[1], end_of<N, GLL>(t0, 1, b0, b1), xn[1][k]);
        if constexpr (GLL) {
          o[0] += lo;
          o[N - 1] += hi;
        } else {
#pragma unroll
          for (int i = 0; i < N; ++i) o[i] += b0[i] * lo + b1[i] * hi;
        }
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) A[m][i] = mad(B(k, m), o[i], A[m][i]);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {  // y faces
        const double* src = a.beta_face[1] + face_index(a, sub, 1, s) * QQ + kz * Q;
        double be[Q], nd[N], own[Q], ext[Q], f[Q], o[N];
#pragma unroll
        for (int k = 0; k < Q; ++k) be[k] = src[k];
        pin(A);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          if constexpr (GLL) nd[i] = u[s ? N - 1 : 0][i];
          else {
            nd[i] = 0.0;
#pragma unroll
            for (int m = 0; m < N; ++m) nd[i] += (s ? b1[m] : b0[m]) * u[m][i];
          }
        }
        P::up(B, nd, own);
#pragma unroll
        for (int i = 0; i < N; ++i) nd[i] = r[2 * NN + (2 + s) * N + i];
        P::up(B, nd, ext);
        const auto rule = face_rule(mesh.neighbour(e, sub, 1, s));
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] = flux(a.c[1] * wz * w[j], be[j], s, rule, own[j], ext[j]);
        P::down(B, f, o);
        if constexpr (GLL) {
#pragma unroll
          for (int i = 0; i < N; ++i) A[s ? N - 1 : 0][i] += o[i];
        } else {
#pragma unroll
          for (int m = 0; m < N; ++m)
#pragma unroll
            for (int i = 0; i < N; ++i) A[m][i] += (s ? b1[m] : b0[m]) * o[i];
        }
      }
      if (a.mass != 0.0) {
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          double t0[N], f[Q], o[N];
          pin(A);
          pin(u);
          P::row(B, u, k, t0);
          P::up(B, t0, f);
#pragma unroll
          for (int j = 0; j < Q; ++j) {
            const int kk[3] = {j, k, kz};
            const double sg = dev::eval_sep<double, 3, Q>(*a.sigma, sub, kk);
            f[j] *= a.mass * sg * (wz * w[k] * w[j]);
          }
          P::down(B, f, o);
#pragma unroll
          for (int m = 0; m < N; ++m)
#pragma unroll
            for (int i = 0; i < N; ++i) A[m][i] = mad(B(k, m), o[i], A[m][i]);
        }
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) r[m * N + i] = A[m][i];
    }
  } else {
    for (int t = tid - 64; t < ne * 2; t += 64) {
      const int el = t >> 1, s = t & 1, e = e0 + el;
      int sub[3];
      mesh.decode(e, sub);
      double* r = zrec + (el * 2 + s) * ZP;
      const double* src = a.beta_face[2] + face_index(a, sub, 2, s) * QQ;
      const int nb = mesh.neighbour(e, sub, 2, s);
      const auto rule = face_rule(nb);
      double u[N][N], A[N][N];
      // the flux takes own - nb, one interpolation of the difference
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = nb < 0 ? r[m * N + i] : r[m * N + i] - r[NN + m * N + i];
          A[m][i] = 0.0;
        }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        double be[Q], t0[N], f[Q], o[N];
#pragma unroll
        for (int j = 0; j < Q; ++j) be[j] = src[k * Q + j];
        pin(A);
        pin(u);
        P::row(B, u, k, t0);
        P::up(B, t0, f);
#pragma unroll
        for (int j = 0; j < Q; ++j) f[j] = flux(a.c[2] * (w[k] * w[j]), be[j], s, rule, f[j], 0.0);
        P::down(B, f, o);
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) A[m][i] = mad(B(k, m), o[i], A[m][i]);
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) r[m * N + i] = A[m][i];
    }
  }
  __syncthreads();

  // ---- phase 3 ----
  for (int t = tid; t < ne * NN; t += NT) {
    const int el = t / NN, c = t - el * NN;
    const double* r = rec + el * Q * PITCH + c;
    const double* z = zrec + el * 2 * ZP + c;
    double f[Q], o[N];
#pragma unroll
    for (int q = 0; q < Q; ++q) f[q] = r[q * PITCH];
    P::down(B, f, o);
    if constexpr (GLL) {
      o[0] += z[0];
      o[N - 1] += z[ZP];
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) o[i] += b0[i] * z[0] + b1[i] * z[ZP];
    }
    double* dst = y + (int64_t)(e0 + el) * ND + c;
#pragma unroll
    for (int i = 0; i < N; ++i) dst[i * NN] = o[i];
  }
}

template <int N, int Q, bool GLL>
__global__ void __launch_bounds__((AdjGeo<N, Q>::NT)) __attribute__((amdgpu_waves_per_eu(2)))
    grad_plane_kernel(AdjArgs a, const double* __restrict__ x, const double* __restrict__ rv)
{
  using G = AdjGeo<N, Q>;
  using P = Planes<double, N, Q>;
  constexpr int NN = G::NN, QQ = G::QQ, ND = NN * N, NT = G::NT, PITCH = G::GP, ZP = G::GZ;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* rec = reinterpret_cast<double*>(smem_raw);  // [element][plane]: B_z u, B_z r, B'_z r, -x u, r, -y u, r
  double* zrec = rec + a.epb * Q * PITCH;             // [element]: lower z face own u, own r, nb u, nb r
  const AdjMesh mesh{a};
  const int blk = dev::xcd_remap(blockIdx.x, a.num_blocks);
  const int e0 = blk * a.epb;
  const int ne = a.E - e0 < a.epb ? a.E - e0 : a.epb;
  const int tid = threadIdx.x;
  const Half<double, N, Q, 1> B(a.B);
  const Half<double, N, Q, -1> Gb(a.Gb);
  CPtr<double> b0 = (CPtr<double>)a.b0;
  CPtr<double> b1 = (CPtr<double>)a.b1;
  CPtr<double> w = (CPtr<double>)a.w;

  // ---- phase 1 ----
  for (int t = tid; t < ne * NN; t += NT) {
    const int el = t / NN, c = t - el * NN, e = e0 + el;
    int sub[3];
    mesh.decode(e, sub);
    const int lo = mesh.neighbour(e, sub, 2, 0);
    const int64_t own = (int64_t)e * ND + c, nb = (int64_t)(lo >= 0 ? lo : e) * ND + c;
    double u[N], q[N], v[Q], nu, nr;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      u[i] = x[own + i * NN];
      q[i] = rv[own + i * NN];
    }
    if constexpr (GLL) {
      nu = x[nb + (N - 1) * NN];
      nr = rv[nb + (N - 1) * NN];
    } else {
      double l[N], h[N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        l[i] = x[nb + i * NN];
        h[i] = rv[nb + i * NN];
      }
      nu = end_of<N, GLL>(l, 1, b0, b1);
      nr = end_of<N, GLL>(h, 1, b0, b1);
    }
    double* r = rec + el * Q * PITCH + c;
    P::up(B, u, v);
#pragma unroll
    for (int k = 0; k < Q; ++k) r[k * PITCH] = v[k];
    P::up(B, q, v);
#pragma unroll
    for (int k = 0; k < Q; ++k) r[k * PITCH + NN] = v[k];
    P::up(Gb, q, v);
#pragma unroll
    for (int k = 0; k < Q; ++k) r[k * PITCH + 2 * NN] = v[k];
    double* z = zrec + el * ZP + c;
    z[0] = end_of<N, GLL>(u, 0, b0, b1);
    z[NN] = end_of<N, GLL>(q, 0, b0, b1);
    z[2 * NN] = lo >= 0 ? nu : 0.0;
    z[3 * NN] = lo >= 0 ? nr : 0.0;
  }
  for (int t = tid; t < ne * 4 * N; t += NT) {
    const int el = t / (4 * N), c = t - el * (4 * N);
    const int f = c / N, m = c - f * N, e = e0 + el;  // -x of u, -x of r, -y of u, -y of r; tangential node
    int sub[3];
    mesh.decode(e, sub);
    double u[N], v[Q];
    face_pencil<N, GLL>(f & 1 ? rv : x, mesh.neighbour(e, sub, f >> 1, 0), f >> 1, m, 1, b0, b1, u);
    P::up(B, u, v);
    double* r = rec + el * Q * PITCH + 3 * NN + c;
#pragma unroll
    for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
  }
  __syncthreads();

  // d/d beta at one point of a face: cw = adv_coef detJ w / h
  auto face_grad = [&](double cw, bool upper, bool bnd, double beta, double uo, double un, double ro, double rn) {
    const double nrm = upper ? cw : -cw;
    const bool out = upper ? beta > 0.0 : -beta > 0.0;  // flow leaves this side
    if (bnd) return a.bc_none ? 0.0 : nrm * ro * (out ? uo : un);
    const double up_nb = upper ? (-beta > 0.0 ? un : uo) : (beta > 0.0 ? un : uo);
    return nrm * (ro * (out ? uo : un) - rn * up_nb);
  };
  auto inflow = [&](const int* sub, int kx, int ky, int kz) {
    const int kk[3] = {kx, ky, kz};
    return a.bc_data ? dev::eval_sep<double, 3, Q>(*a.bc, sub, kk) : 0.0;
  };

  // ---- phase 2 ----
  if (tid < 64) {
    for (int t = tid; t < ne * Q; t += 64) {
      const int el = t / Q, kz = t - el * Q, e = e0 + el;
      int sub[3];
      mesh.decode(e, sub);
      double* r = rec + (el * Q + kz) * PITCH;
      const double wz = ((GPtr<double>)a.w)[kz];
      double u[N][N], q[N][N], d[N][N];
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = r[m * N + i];
          q[m][i] = r[NN + m * N + i];
          d[m][i] = r[2 * NN + m * N + i];
        }
      // the lower x and y faces (and upper ones on the boundary) at this plane
#pragma unroll
      for (int ax = 0; ax < 2; ++ax)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int nb = mesh.neighbour(e, sub, ax, s);
          if (s == 1 && nb >= 0) continue;
          const int64_t at = face_index(a, sub, ax, s) * QQ + kz * Q;
          double be[Q], nd[N], uo[Q], ro[Q], un[Q], rn[Q];
#pragma unroll
          for (int k = 0; k < Q; ++k) be[k] = a.beta_face[ax][at + k];
          // own traces: the plane's line at the face, interpolated along it
#pragma unroll
          for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int m = 0; m < N; ++m) {
              double v[N];
#pragma unroll
              for (int i = 0; i < N; ++i) {
                const double p = ax == 0 ? (h ? q[m][i] : u[m][i]) : (h ? q[i][m] : u[i][m]);
                v[i] = p;
              }
              nd[m] = end_of<N, GLL>(v, s, b0, b1);
            }
            P::up(B, nd, h ? ro : uo);
          }
#pragma unroll
          for (int m = 0; m < N; ++m) nd[m] = r[3 * NN + 2 * ax * N + m];
          P::up(B, nd, un);
#pragma unroll
          for (int m = 0; m < N; ++m) nd[m] = r[3 * NN + (2 * ax + 1) * N + m];
          P::up(B, nd, rn);
#pragma unroll
          for (int k = 0; k < Q; ++k) {
            if (nb < 0) un[k] = inflow(sub, ax == 0 ? Q + s : k, ax == 0 ? k : Q + s, kz);
            a.dface[ax][at + k] =
                face_grad(a.c[ax] * wz * w[k], s, nb < 0, be[k], uo[k], un[k], ro[k], rn[k]);
          }
        }
      // all inputs of the record are in registers: the results replace them
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        double t0[N], v[Q], g[Q];
        pin(u);
        P::row(B, u, k, t0);
        P::up(B, t0, v);
#pragma unroll
        for (int j = 0; j < Q; ++j) v[j] *= -(wz * w[k] * w[j]);
        pin(q);
        P::row(B, q, k, t0);
        P::up(Gb, t0, g);
#pragma unroll
        for (int j = 0; j < Q; ++j) r[k * Q + j] = a.c[0] * v[j] * g[j];
        P::row(Gb, q, k, t0);
        P::up(B, t0, g);
#pragma unroll
        for (int j = 0; j < Q; ++j) r[QQ + k * Q + j] = a.c[1] * v[j] * g[j];
        pin(d);
        P::row(B, d, k, t0);
        P::up(B, t0, g);
#pragma unroll
        for (int j = 0; j < Q; ++j) r[2 * QQ + k * Q + j] = a.c[2] * v[j] * g[j];
      }
    }
  } else {
    // z faces: one row of a face per thread
    for (int t = tid - 64; t < ne * Q; t += 64) {
      const int el = t / Q, k = t - el * Q, e = e0 + el;
      int sub[3];
      mesh.decode(e, sub);
      const double* z = zrec + el * ZP;
      const double wk = ((GPtr<double>)a.w)[k];
      double row[N];
#pragma unroll
      for (int m = 0; m < N; ++m) row[m] = ((GPtr<double>)a.B)[k * N + m];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int nb = mesh.neighbour(e, sub, 2, s);
        if (s == 1 && nb >= 0) continue;
        const int64_t at = face_index(a, sub, 2, s) * QQ + k * Q;
        double be[Q], v[4][Q];
#pragma unroll
        for (int j = 0; j < Q; ++j) be[j] = a.beta_face[2][at + j];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          double nd[N];
#pragma unroll
          for (int i = 0; i < N; ++i) {
            nd[i] = 0.0;
#pragma unroll
            for (int m = 0; m < N; ++m) {
              double p;
              if (s == 0) p = z[h * NN + m * N + i];
              else if (h < 2) {  // an upper boundary face: its traces from the element's own pencils
                double pen[N];
#pragma unroll
                for (int l = 0; l < N; ++l) pen[l] = (h ? rv : x)[(int64_t)e * ND + l * NN + m * N + i];
                p = end_of<N, GLL>(pen, 1, b0, b1);
              } else p = 0.0;
              nd[i] += row[m] * p;
            }
          }
          P::up(B, nd, v[h]);
        }
#pragma unroll
        for (int j = 0; j < Q; ++j) {
          if (nb < 0) v[2][j] = inflow(sub, j, k, Q + s);
          a.dface[2][at + j] = face_grad(a.c[2] * wk * w[j], s, nb < 0, be[j], v[0][j], v[2][j], v[1][j], v[3][j]);
        }
      }
    }
  }
  __syncthreads();

  // ---- phase 3: the cell results, consecutive in the elements of the block ----
  for (int t = tid; t < ne * 3 * Q * QQ; t += NT) {
    const int el = t / (3 * Q * QQ), i = t - el * (3 * Q * QQ);
    const int c = i / (Q * QQ), p = i - c * (Q * QQ);
    const int kz = p / QQ, ij = p - kz * QQ;
    a.dcell[(int64_t)e0 * (3 * Q * QQ) + t] = rec[(el * Q + kz) * PITCH + c * QQ + ij];
  }
}

template <int N, int Q, bool GLL>
int launch_adjoint(AdjArgs& a, bool grad, const double* x, double* y, hipStream_t s)
{
  using G = AdjGeo<N, Q>;
  const size_t per = (grad ? Q * G::GP + G::GZ : Q * G::TP + 2 * G::TZ) * sizeof(double);
  a.epb = G::EPB;
  while (a.epb > 2 && (int64_t)a.epb * 512 > a.E) a.epb = (a.epb + 1) / 2;
  a.num_blocks = (int)((a.E + a.epb - 1) / a.epb);
  const size_t lds = a.epb * per;
  constexpr int tr = Q * G::TP + 2 * G::TZ, gr = Q * G::GP + G::GZ;
  constexpr size_t most = (size_t)G::EPB * (tr > gr ? tr : gr) * sizeof(double);
  static_assert(most <= 64 * 1024, "LDS of one block without an attribute");
  if (grad) hipLaunchKernelGGL((grad_plane_kernel<N, Q, GLL>), dim3((unsigned)a.num_blocks), dim3(G::NT), lds, s, a, x, y);
  else hipLaunchKernelGGL((transpose_plane_kernel<N, Q, GLL>), dim3((unsigned)a.num_blocks), dim3(G::NT), lds, s, a, x, y);
  GD_HIP(hipGetLastError());
  return GD_OK;
}

template <int N, int Q>
int launch_adj(AdjArgs& a, bool grad, const double* x, double* y, hipStream_t s)
{
  return a.gll ? launch_adjoint<N, Q, true>(a, grad, x, y, s) : launch_adjoint<N, Q, false>(a, grad, x, y, s);
}

}  // namespace pl
}  // namespace gd
