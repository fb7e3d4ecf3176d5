// gfx950 kernel of the uniform 3D apply for any basis, rule and separable or
// affine field (the forms the Kronecker and register kernels do not take):
// y = mass_coef M x + adv_coef A x with cell, interior-facet and boundary
// terms in one pass (MassElementOperator, massoperator.hpp:39-89;
// AdvectionFusedOperatorWith[out]BC, advectionoperator.hpp:106-441).
//
// One thread holds one z-plane of rule points of one element in registers, so
// the x and y contractions of the plane, the coefficient at its points and the
// x and y test functions run without LDS; only the z contractions cross
// threads.  Three phases with one block barrier between them:
//   1. one thread per (element, x-y node): loads the node's z pencil from HBM
//      and writes B_z of it, and the traces at z = 0 and 1, into the plane
//      records in LDS; one thread per (element, x or y face, tangential node)
//      does the same with the neighbour's pencil on that face;
//   2. one thread per plane record: the q cell planes of an element and, in a
//      wave of their own, its two z faces.  The own trace on an x face is the
//      end value of the y-interpolated row, and the flux enters the row before
//      the y test, so an x face costs its neighbour pencil's interpolation; a y
//      face is one more row of the plane;
//   3. one thread per (element, x-y node): z test functions, store.
// The two outputs of a plane (the part tested with B in z and the part tested
// with B') go into the record it read, so the LDS need is q + 2 records of
// 2 n^2 values per element and no point data is ever stored.
//
// Bound by FP64 issue and the waits a block's two barriers leave exposed at two
// waves a SIMD: 53 x 47 x 41, p = 3, q = 5, inflow data, a field over two
// coordinates, FP64: 90 us, 2,280 VALU instructions per wave (47 us of issue),
// against 438 us for the generic kernel, whose every 1D contraction goes
// through LDS.  43 x 37 x 29 mass, p = 2, q = 5, FP32, three-term sigma: 8.1
// against 34 us (latency: one round of blocks).
// Measured without a gain at the first size: one wave per block with the z
// faces' rows spread over the cell planes (140 us: five waves a CU), 25-element
// blocks (134 us: three waves each, the SIMDs unevenly filled).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gd_internal.hpp"
#include "gd_kernels.hpp"

namespace gd {
namespace pl {

// division by a launch constant: n / d for n < 2^31 (multiply by
// floor(2^k / d) + 1, k = 31 + ceil(log2 d); exact there since n d < 2^k)
struct FastDiv {
  uint32_t mul;
  int shift;
  int d;
};

inline FastDiv fast_div(int64_t d)
{
  int l = 0;
  while (((int64_t)1 << l) < d) ++l;
  return FastDiv{(uint32_t)((((uint64_t)1 << (31 + l)) / (uint64_t)d) + 1), 31 + l, (int)d};
}

__device__ __forceinline__ int div(const FastDiv& f, int n)
{
  return (int)(((uint64_t)(uint32_t)n * f.mul) >> f.shift);
}

// A separable field as the kernel reads it: its terms' masks and its first row
// (FieldTerms), in scalar registers.
struct Field {
  int rank, mask, row;
};

// Kernel arguments: only what this kernel reads (the generic parameter block
// costs the host as much to fill as the launch of a small mesh)
template <typename T>
struct Args {
  int E, epb, num_blocks;
  int row0, row1;  // rows of the coefficients in use (FieldTerms)
  int spitch;      // their samples per element in LDS, odd
  Field sigma, beta[3], bc;  // rows relative to row0
  FastDiv d0, d1;
  int M[3];
  int periodic_mask;
  int gll, field;    // instance: traces are node layers; how beta is given
  int bc_none;       // boundary faces carry no flux
  int bc_data;       // inflow data with at least one term
  T h[3], invh[3], origin[3];
  T detJ, mass_coef, adv_coef;
  T affA[3][3], affc[3];
  const T *beta_cell, *beta_face[3];  // pointwise beta
  const FieldTerms<T>* terms;
  const FieldDev<T>* sigma_tab;
  const T *B, *Gb, *b0, *b1, *xq, *w;
};

enum { kSeparable = 0, kAffine = 1, kPointwise = 2 };

// number of element sub's lower (0) or upper (1) face normal to axis a, in the
// order of the per-face-point arrays (extents M, along a M + 1 unless periodic)
template <typename A>
__device__ __forceinline__ int64_t face_index(const A& a, const int* sub, int ax, int side)
{
  const bool per = (a.periodic_mask >> ax) & 1;
  int s[3] = {sub[0], sub[1], sub[2]};
  int64_t ext[2] = {a.M[0], a.M[1]};
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (d == ax) {
      s[d] += side;
      if (per && s[d] == a.M[d]) s[d] = 0;
      if (d < 2) ext[d] += per ? 0 : 1;
    }
  return s[0] + ext[0] * (s[1] + ext[1] * s[2]);
}

// scalar (constant address space) view of a table: uniform reads become
// scalar loads whatever the surrounding stores
template <typename T>
using CPtr = const __attribute__((address_space(4))) T*;
template <typename T>
using GPtr = const __attribute__((address_space(1))) T*;

// one rounding, in the order written (left to contraction, the first sum of a
// chain may take either product as the rounded one)
__device__ __forceinline__ double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// A 1D table [q][n] in scalar registers.
template <typename T, int N, int Q>
struct Full {
  T v[N * Q];
  __device__ __forceinline__ explicit Full(const T* tab)
  {
    CPtr<T> c = (CPtr<T>)tab;
#pragma unroll
    for (int i = 0; i < N * Q; ++i) v[i] = c[i];
  }
  __device__ __forceinline__ T operator()(int j, int i) const { return v[j * N + i]; }
};

// The same for a rule and basis that are symmetric about the middle of
// the element: the half of it that is not the mirror image (SIGN = 1: B) or the
// negated mirror image (SIGN = -1: B') of the other.  The halves of both tables
// fit the scalar registers (n = 4, q = 5: 40 of about 100); the full ones with
// their weighted transposes do not (889 scalar spills in that kernel).  The
// weights go into the coefficient instead.
template <typename T, int N, int Q, int SIGN>
struct Half {
  static constexpr int H = (N * Q + 1) / 2;
  T v[H];
  __device__ __forceinline__ explicit Half(const T* tab)
  {
    CPtr<T> c = (CPtr<T>)tab;
#pragma unroll
    for (int i = 0; i < H; ++i) v[i] = c[i];
  }
  __device__ __forceinline__ T operator()(int j, int i) const
  {
    const int k = j * N + i;
    return k < H ? v[k] : (SIGN > 0 ? v[N * Q - 1 - k] : -v[N * Q - 1 - k]);
  }
};

// Orders the point rows of a plane: values pinned here are complete before, and
// used only after, this point.  A row has enough independent chains to fill
// the FP64 pipeline; left to itself the compiler interleaves the rows and
// keeps several rows' temporaries live (n = 4, q = 5: 147 spilled registers).
// FP32 planes fit without it.
template <typename T, int K>
__device__ __forceinline__ void pin(T (&v)[K])
{
  if constexpr (sizeof(T) == 8) {
#pragma unroll
    for (int i = 0; i < K; ++i) asm volatile("" : "+v"(v[i]));
  }
}

template <typename T, int K, int L>
__device__ __forceinline__ void pin(T (&v)[K][L])
{
#pragma unroll
  for (int i = 0; i < K; ++i) pin(v[i]);
}

template <int N, int Q, bool ADV>
struct Geo {
  static constexpr int NN = N * N;
  static constexpr int NB = NN > 4 * N ? NN : 4 * N;  // neighbour pencils (x, y faces) or second output
  static constexpr int PITCH = (ADV ? NN + NB : NN) | 1;  // odd: consecutive records fall on different banks
  static constexpr int PL = ADV ? Q + 2 : Q;
  // most elements per block: two z faces each fill the last wave; the mass
  // planes fill two waves
  static constexpr int EPB = N >= 5 ? 128 / Q : 32;
  static constexpr int CELLW = (EPB * Q + 63) / 64 * 64;  // waves that take cell planes in phase 2
  static constexpr int NT = ADV ? CELLW + 64 : (CELLW < 128 ? 128 : CELLW);
};

// Samples k0.. of a row of the element's into v, 1 where the term has no such
// row.  The rows are staged in LDS: read from the tables at each use, a term is
// two dependent memory latencies.
template <typename T, int S>
struct LdsRows {
  const T* sm;
  template <int K>
  __device__ __forceinline__ void get(int has, int row, int k0, T (&v)[K]) const
  {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = T(1);
    if (has) {
#pragma unroll
      for (int k = 0; k < K; ++k) v[k] = sm[row * S + k0 + k];
    }
  }
};

template <typename T, int N, int Q>
struct Planes {
  static constexpr int S = Q + 2;

  // f at the points of a plane of sample kz, times wz and (WGT) the plane's
  // weights: they enter with the rows, Q products each instead of Q^2
  template <bool WGT, class Rows>
  __device__ __forceinline__ static void separable(const Field& f, const Rows& rows, int kz, CPtr<T> w, T wz,
                                                   T (&b)[Q][Q])
  {
    int row = f.row, m = f.mask;
#pragma unroll
    for (int k = 0; k < Q; ++k)
#pragma unroll
      for (int j = 0; j < Q; ++j) b[k][j] = T(0);
#pragma unroll 1
    for (int r = 0; r < f.rank; ++r, m >>= 3) {
      const int rx = row, ry = rx + (m & 1), rz = ry + ((m >> 1) & 1);
      row = rz + ((m >> 2) & 1);
      T a[Q], X[Q], z[1];
      rows.get(m & 1, rx, 0, X);
      rows.get(m & 2, ry, 0, a);
      rows.get(m & 4, rz, kz, z);
      z[0] *= wz;
      if constexpr (WGT) {
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          X[k] *= w[k];
          a[k] *= w[k];
        }
      }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        a[k] *= z[0];
#pragma unroll
        for (int j = 0; j < Q; ++j) b[k][j] += a[k] * X[j];
      }
    }
  }

  // f at the points of a plane straight from its tables, each term's product
  // taken along x, y, z
  __device__ __forceinline__ static void points(const FieldDev<T>* fd, const int* sub, int kz, T (&b)[Q][Q])
  {
    CPtr<FieldDev<T>> f = (CPtr<FieldDev<T>>)fd;
#pragma unroll
    for (int k = 0; k < Q; ++k)
#pragma unroll
      for (int j = 0; j < Q; ++j) b[k][j] = T(0);
    const int rank = f->rank;
#pragma unroll 1
    for (int r = 0; r < rank; ++r) {
#pragma clang fp contract(off)
      GPtr<T> tx = (GPtr<T>)f->tab[r][0];
      GPtr<T> ty = (GPtr<T>)f->tab[r][1];
      GPtr<T> tz = (GPtr<T>)f->tab[r][2];
      const T scale = f->scale[r];
      T X[Q], y[Q], z = T(1);
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        X[k] = scale;
        y[k] = T(1);
      }
      if (tx) {
#pragma unroll
        for (int k = 0; k < Q; ++k) X[k] = scale * tx[sub[0] * S + k];
      }
      if (ty) {
#pragma unroll
        for (int k = 0; k < Q; ++k) y[k] = ty[sub[1] * S + k];
      }
      if (tz) z = tz[sub[2] * S + kz];
#pragma unroll
      for (int k = 0; k < Q; ++k)
#pragma unroll
        for (int j = 0; j < Q; ++j) {
          const T t = X[j] * y[k] * z;
          b[k][j] = b[k][j] + t;
        }
    }
  }

  // f on the two lines of the plane at the ends of axis AX (0: x = ends, points
  // along y; 1: y = ends, points along x), with weights as above
  template <int AX, bool WGT, class Rows>
  __device__ __forceinline__ static void separable_ends(const Field& f, const Rows& rows, int kz, CPtr<T> w, T wz,
                                                        T (&b)[2][Q])
  {
    int row = f.row, m = f.mask;
#pragma unroll
    for (int k = 0; k < Q; ++k) b[0][k] = b[1][k] = T(0);
#pragma unroll 1
    for (int r = 0; r < f.rank; ++r, m >>= 3) {
      const int rx = row, ry = rx + (m & 1), rz = ry + ((m >> 1) & 1);
      row = rz + ((m >> 2) & 1);
      const int re = AX == 0 ? rx : ry, ro = AX == 0 ? ry : rx;
      T e[2], o[Q], z[1];
      rows.get(m & (1 << AX), re, Q, e);
      rows.get(m & (2 >> AX), ro, 0, o);
      rows.get(m & 4, rz, kz, z);
      z[0] *= wz;
      e[0] *= z[0];
      e[1] *= z[0];
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        if constexpr (WGT) o[k] *= w[k];
        b[0][k] += e[0] * o[k];
        b[1][k] += e[1] * o[k];
      }
    }
  }

  __device__ __forceinline__ static T cell(const Args<T>& p, int d, const int* sub)
  {
    return p.origin[d] + p.h[d] * (T)sub[d];
  }

  __device__ __forceinline__ static T affine_base(const Args<T>& p, int c, const int* sub, int kz)
  {
    return p.affc[c] + p.affA[c][2] * (cell(p, 2, sub) + p.h[2] * (kz < Q ? ((GPtr<T>)p.xq)[kz] : (kz == Q ? T(0) : T(1))));
  }

  // component c of an affine field at the points of a plane
  __device__ __forceinline__ static void affine(const Args<T>& p, int c, const int* sub, int kz, CPtr<T> w, T wz,
                                                T (&b)[Q][Q])
  {
    CPtr<T> xq = (CPtr<T>)p.xq;
    const T base = affine_base(p, c, sub, kz);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const T row = base + p.affA[c][1] * (cell(p, 1, sub) + p.h[1] * xq[k]);
#pragma unroll
      for (int j = 0; j < Q; ++j)
        b[k][j] = w[j] * (wz * w[k]) * (row + p.affA[c][0] * (cell(p, 0, sub) + p.h[0] * xq[j]));
    }
  }

  // component AX of an affine field on the lines at the ends of axis AX
  template <int AX>
  __device__ __forceinline__ static void affine_ends(const Args<T>& p, const int* sub, int kz, CPtr<T> w, T wz,
                                                     T (&b)[2][Q])
  {
    constexpr int O = 1 - AX;
    CPtr<T> xq = (CPtr<T>)p.xq;
    const T base = affine_base(p, AX, sub, kz);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const T line = base + p.affA[AX][O] * (cell(p, O, sub) + p.h[O] * xq[k]);
      b[0][k] = wz * w[k] * (line + p.affA[AX][AX] * cell(p, AX, sub));
      b[1][k] = wz * w[k] * (line + p.affA[AX][AX] * (cell(p, AX, sub) + p.h[AX]));
    }
  }

  __device__ __forceinline__ static void plane_of(const T* src, T (&b)[Q][Q])
  {
#pragma unroll
    for (int k = 0; k < Q; ++k)
#pragma unroll
      for (int j = 0; j < Q; ++j) b[k][j] = src[k * Q + j];
  }

  // out[j] = sum_i tab[j][i] in[i]: n nodes to q points
  template <class Tab>
  __device__ __forceinline__ static void up(const Tab& tab, const T (&in)[N], T (&out)[Q])
  {
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      T s = tab(j, 0) * in[0];
#pragma unroll
      for (int i = 1; i < N; ++i) s = mad(tab(j, i), in[i], s);
      out[j] = s;
    }
  }

  // out[i] = sum_j tab[j][i] in[j]: q points to n nodes
  template <class Tab>
  __device__ __forceinline__ static void down(const Tab& tab, const T (&in)[Q], T (&out)[N])
  {
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = tab(0, i) * in[0];
#pragma unroll
    for (int j = 1; j < Q; ++j)
#pragma unroll
      for (int i = 0; i < N; ++i) out[i] = mad(tab(j, i), in[j], out[i]);
  }

  // row k of points (x nodes) of a plane of n x n nodes (rows y, columns x)
  template <class Tab>
  __device__ __forceinline__ static void row(const Tab& B, const T (&u)[N][N], int k, T (&out)[N])
  {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      T s = B(k, 0) * u[0][i];
#pragma unroll
      for (int m = 1; m < N; ++m) s = mad(B(k, m), u[m][i], s);
      out[i] = s;
    }
  }

  // plane of n x n nodes to the q x q points, and the traces xo at the rows' ends
  template <bool GLL, class Tab>
  __device__ __forceinline__ static void interp(const Tab& B, T (&u)[N][N], T (&v)[Q][Q], T (&xo)[2][Q],
                                                CPtr<T> b0, CPtr<T> b1)
  {
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      T t[N];
      pin(u);
      row(B, u, k, t);
      up(B, t, v[k]);
      pin(v[k]);
      if constexpr (GLL) {
        xo[0][k] = t[0];
        xo[1][k] = t[N - 1];
      } else {
        T s0 = T(0), s1 = T(0);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          s0 += b0[i] * t[i];
          s1 += b1[i] * t[i];
        }
        xo[0][k] = s0;
        xo[1][k] = s1;
      }
    }
  }
};

// GLL: the basis values at the element ends are unit vectors, so a trace is a
// node layer.  FIELD: how beta is given (kSeparable, kAffine, kPointwise).
template <typename T, int N, int Q, bool ADV, bool GLL, int FIELD>
__global__ void __launch_bounds__((Geo<N, Q, ADV>::NT)) __attribute__((amdgpu_waves_per_eu(2)))
    plane_kernel(Args<T> a, const T* __restrict__ x, T* __restrict__ y)
{
  using G = Geo<N, Q, ADV>;
  using P = Planes<T, N, Q>;
  constexpr int NN = G::NN, ND = NN * N, PL = G::PL, PITCH = G::PITCH, NT = G::NT;

  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* rec = reinterpret_cast<T*>(smem_raw);
  T* smp = rec + a.epb * PL * PITCH;  // the coefficients' row samples, a.spitch per element

  const int blk = dev::xcd_remap(blockIdx.x, a.num_blocks);
  const int e0 = blk * a.epb;
  const int ne = a.E - e0 < a.epb ? a.E - e0 : a.epb;
  const int tid = threadIdx.x;
  using Interp = std::conditional_t<ADV, Half<T, N, Q, 1>, Full<T, N, Q>>;
  const Interp B(a.B);
  const Half<T, N, Q, -1> Gb(a.Gb);
  CPtr<T> w = (CPtr<T>)a.w;
  CPtr<T> b0 = (CPtr<T>)a.b0;
  CPtr<T> b1 = (CPtr<T>)a.b1;

  auto decode = [&](int e, int* sub) {
    const int q0 = div(a.d0, e), q1 = div(a.d1, q0);
    sub[0] = e - q0 * a.M[0];
    sub[1] = q0 - q1 * a.M[1];
    sub[2] = q1;
  };
  // neighbour of element e (at sub) across its lower (0) or upper (1) face
  // normal to axis d, -1 at the boundary
  auto neighbour = [&](int e, const int* sub, int d, int side) {
    const int stride = d == 0 ? 1 : (d == 1 ? a.M[0] : a.M[0] * a.M[1]);
    const int M = d == 0 ? a.M[0] : (d == 1 ? a.M[1] : a.M[2]);
    const int s = d == 0 ? sub[0] : (d == 1 ? sub[1] : sub[2]);
    const bool per = (a.periodic_mask >> d) & 1;
    if (side == 0) return s > 0 ? e - stride : (per ? e + (M - 1) * stride : -1);
    return s < M - 1 ? e + stride : (per ? e - (M - 1) * stride : -1);
  };

  auto rows = [](const T* sm) { return LdsRows<T, Q + 2>{sm}; };
  // the advection field times the weights of its plane (times wz) or line; a
  // pointwise field's plane comes without (its weights go into v)
  auto beta_at = [&](int c, int e, const int* sub, const T* sm, int kz, T wz, T (&b)[Q][Q]) {
    if constexpr (FIELD == kAffine) P::affine(a, c, sub, kz, w, wz, b);
    else if constexpr (FIELD == kPointwise) {
      const T* src = kz < Q ? a.beta_cell + ((int64_t)e * 3 + c) * (Q * Q * Q) + kz * (Q * Q)
                            : a.beta_face[2] + face_index(a, sub, 2, kz - Q) * (Q * Q);
      P::plane_of(src, b);
    } else P::template separable<true>(a.beta[c], rows(sm), kz, w, wz, b);
  };
  auto beta_ends = [&](auto ax, const int* sub, const T* sm, int kz, T wz, T (&b)[2][Q]) {
    constexpr int AX = decltype(ax)::value;
    if constexpr (FIELD == kAffine) P::template affine_ends<AX>(a, sub, kz, w, wz, b);
    else if constexpr (FIELD == kPointwise) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const T* src = a.beta_face[AX] + face_index(a, sub, AX, s) * (Q * Q) + kz * Q;
#pragma unroll
        for (int k = 0; k < Q; ++k) b[s][k] = src[k];
      }
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        b[0][k] *= wz * w[k];
        b[1][k] *= wz * w[k];
      }
    } else P::template separable_ends<AX, true>(a.beta[AX], rows(sm), kz, w, wz, b);
  };

  // ---- phase 1: z contractions of the own and the neighbours' pencils ----
  // every load of the phase is issued before the first is used
  constexpr int ITA = (G::EPB * NN + NT - 1) / NT, ITB = ADV ? (G::EPB * 4 * N + NT - 1) / NT : 0;
  T ua[ITA][N], za[ITA][2], ub[ITB + 1][N];
#pragma unroll
  for (int it = 0; it < ITA; ++it) {
    const int t = tid + it * NT;
    if (t < ne * NN) {
      const int el = t / NN, c = t - el * NN;
      const T* src = x + (int64_t)(e0 + el) * ND + c;
#pragma unroll
      for (int i = 0; i < N; ++i) ua[it][i] = src[i * NN];
    }
  }
  if constexpr (ADV) {
#pragma unroll
    for (int it = 0; it < ITA; ++it) {
      const int t = tid + it * NT;
      za[it][0] = za[it][1] = T(0);
      if (t < ne * NN) {
        const int el = t / NN, c = t - el * NN;
        int sub[3];
        decode(e0 + el, sub);
        const int lo = neighbour(e0 + el, sub, 2, 0), hi = neighbour(e0 + el, sub, 2, 1);
        if constexpr (GLL) {
          if (lo >= 0) za[it][0] = x[(int64_t)lo * ND + (N - 1) * NN + c];
          if (hi >= 0) za[it][1] = x[(int64_t)hi * ND + c];
        } else {
          // no branch on the boundary: all 2 n loads are in flight together
          const T* pl = x + (int64_t)(lo >= 0 ? lo : e0 + el) * ND + c;
          const T* ph = x + (int64_t)(hi >= 0 ? hi : e0 + el) * ND + c;
          T l[N], h[N];
#pragma unroll
          for (int i = 0; i < N; ++i) {
            l[i] = pl[i * NN];
            h[i] = ph[i * NN];
          }
#pragma unroll
          for (int i = 0; i < N; ++i) {
            za[it][0] += b1[i] * l[i];
            za[it][1] += b0[i] * h[i];
          }
          if (lo < 0) za[it][0] = T(0);
          if (hi < 0) za[it][1] = T(0);
        }
      }
    }
#pragma unroll
    for (int it = 0; it < ITB; ++it) {
      const int t = tid + it * NT;
#pragma unroll
      for (int i = 0; i < N; ++i) ub[it][i] = T(0);
      if (t < ne * 4 * N) {
        const int el = t / (4 * N), c = t - el * (4 * N);
        const int f = c / N, m = c - f * N;  // faces -x, +x, -y, +y; tangential node
        int sub[3];
        decode(e0 + el, sub);
        const int ax = f >> 1, side = f & 1;
        const int nb = neighbour(e0 + el, sub, ax, side);
        const int tang = ax == 0 ? m * N : m, norm = ax == 0 ? 1 : N;
        if constexpr (GLL) {
          if (nb >= 0) {
            const T* src = x + (int64_t)nb * ND + tang + (side ? 0 : (N - 1) * norm);
#pragma unroll
            for (int i = 0; i < N; ++i) ub[it][i] = src[i * NN];
          }
        } else {
          const T* src = x + (int64_t)(nb >= 0 ? nb : e0 + el) * ND + tang;
          T l[N][N];
#pragma unroll
          for (int k = 0; k < N; ++k)
#pragma unroll
            for (int i = 0; i < N; ++i) l[k][i] = src[i * NN + k * norm];
#pragma unroll
          for (int k = 0; k < N; ++k) {
            const T w = nb < 0 ? T(0) : (side ? b0[k] : b1[k]);
#pragma unroll
            for (int i = 0; i < N; ++i) ub[it][i] += w * l[k][i];
          }
        }
      }
    }
  }
  // the samples of the coefficients' rows at the block's elements, four loads in flight
  for (int t = tid; ADV && t < ne * (Q + 2); t += NT) {
    const int el = t / (Q + 2), k = t - el * (Q + 2);
    int sub[3];
    decode(e0 + el, sub);
    CPtr<FieldTerms<T>> ft = (CPtr<FieldTerms<T>>)a.terms;
    T* dst = smp + el * a.spitch + k;
    for (int f = a.row0; f < a.row1; f += 4) {
      T v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int g = f + i < a.row1 ? f + i : f;  // past the end: the first again
        const int ax = ft->axis[g];
        const int pos = ax == 0 ? sub[0] : (ax == 1 ? sub[1] : (ax == 2 ? sub[2] : 0));
        v[i] = ((GPtr<T>)ft->tab[g])[pos * (Q + 2) + k];
        if (ax == kRowConstant) v[i] = T(1);
        v[i] *= ft->scale[g];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f + i < a.row1) dst[(f + i - a.row0) * (Q + 2)] = v[i];
    }
  }
#pragma unroll
  for (int it = 0; it < ITA; ++it) {
    const int t = tid + it * NT;
    if (t < ne * NN) {
      const int el = t / NN, c = t - el * NN;
      T* r = rec + el * PL * PITCH + c;
      T v[Q];
      P::up(B, ua[it], v);
#pragma unroll
      for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
      if constexpr (ADV) {
        T lo = ua[it][0], hi = ua[it][N - 1];
        if constexpr (!GLL) {
          lo = hi = T(0);
#pragma unroll
          for (int i = 0; i < N; ++i) {
            lo += b0[i] * ua[it][i];
            hi += b1[i] * ua[it][i];
          }
        }
        r[Q * PITCH] = lo;
        r[(Q + 1) * PITCH] = hi;
        r[Q * PITCH + NN] = za[it][0];
        r[(Q + 1) * PITCH + NN] = za[it][1];
      }
    }
  }
  if constexpr (ADV) {
#pragma unroll
    for (int it = 0; it < ITB; ++it) {
      const int t = tid + it * NT;
      if (t < ne * 4 * N) {
        const int el = t / (4 * N), c = t - el * (4 * N);
        T* r = rec + el * PL * PITCH + NN + c;
        T v[Q];
        P::up(B, ub[it], v);
#pragma unroll
        for (int q = 0; q < Q; ++q) r[q * PITCH] = v[q];
      }
    }
  }
  __syncthreads();

  // ---- phase 2: one plane per thread ----
  if (!ADV || tid < G::CELLW) {
    for (int t = tid; t < ne * Q; t += G::CELLW) {
      const int el = t / Q, kz = t - el * Q;
      const int e = e0 + el;
      int sub[3];
      decode(e, sub);
      T* r = rec + (el * PL + kz) * PITCH;
      const T* sm = smp + el * a.spitch;
      const T wz = ((GPtr<T>)a.w)[kz];
      T v[Q][Q], xo[2][Q], b[Q][Q];
      // a pointwise field's first plane is on its way during the interpolation
      if constexpr (ADV && FIELD == kPointwise) beta_at(0, e, sub, smp, kz, wz, b);
      {
        T u[N][N];
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) u[m][i] = r[m * N + i];
        P::template interp<GLL>(B, u, v, xo, b0, b1);
      }
      if constexpr (ADV && FIELD == kPointwise) {
#pragma unroll
        for (int k = 0; k < Q; ++k)
#pragma unroll
          for (int j = 0; j < Q; ++j) v[k][j] *= wz * w[k] * w[j];
      }
      T A[N][N];
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) A[m][i] = T(0);
      // adds the tested row g of point row k: A[m][i] += tab[k][m] g[i]
      auto add = [&](T (&out)[N][N], const auto& tab, int k, const T (&g)[N]) {
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) out[m][i] = mad(tab(k, m), g[i], out[m][i]);
      };
      if constexpr (ADV) {
        const bool none = a.bc_none;
        // upwind flux of one face point: c = adv_coef detJ / h times the
        // field, nrm the sign of the outer normal; boundary points without
        // data carry no flux
        auto flux = [&](T c, T beta, bool plus, T own, T ext, bool bnd) {
          const T dot = (plus ? beta : -beta);
          const T up = dot > T(0) ? dot * own : dot * ext;
          return bnd && none ? T(0) : c * up;
        };
        {  // x component: cell rows and the x faces
          const T c = a.adv_coef * a.detJ * a.invh[0];
          T fx[2][Q];
          {
            T be[2][Q], ge[2][Q];
            beta_ends(std::integral_constant<int, 0>{}, sub, sm, kz, wz, be);
            if (a.bc_data) P::template separable_ends<0, false>(a.bc, rows(sm), kz, w, T(1), ge);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
              T nd[N], ext[Q];
#pragma unroll
              for (int m = 0; m < N; ++m) nd[m] = r[NN + s * N + m];
              pin(nd);
              P::up(B, nd, ext);
              const bool bnd = neighbour(e, sub, 0, s) < 0;
              if (a.bc_data && bnd) {
#pragma unroll
                for (int k = 0; k < Q; ++k) ext[k] = ge[s][k];
              }
#pragma unroll
              for (int k = 0; k < Q; ++k) fx[s][k] = flux(c, be[s][k], s == 1, xo[s][k], ext[k], bnd);
              pin(fx[s]);
            }
          }
          if constexpr (FIELD != kPointwise) beta_at(0, e, sub, sm, kz, wz, b);
#pragma unroll
          for (int k = 0; k < Q; ++k) {
            T f[Q], g[N];
            pin(A);
            pin(v[k]);
#pragma unroll
            for (int j = 0; j < Q; ++j) f[j] = -c * b[k][j] * v[k][j];
            P::down(Gb, f, g);
            if constexpr (GLL) {
              g[0] += fx[0][k];
              g[N - 1] += fx[1][k];
            } else {
#pragma unroll
              for (int i = 0; i < N; ++i) g[i] += b0[i] * fx[0][k] + b1[i] * fx[1][k];
            }
            add(A, B, k, g);
          }
        }
        {  // y component: cell rows, and the y faces as two more rows
          const T c = a.adv_coef * a.detJ * a.invh[1];
          {
            T be[2][Q], ge[2][Q];
            beta_ends(std::integral_constant<int, 1>{}, sub, sm, kz, wz, be);
            if (a.bc_data) P::template separable_ends<1, false>(a.bc, rows(sm), kz, w, T(1), ge);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
              T nd[N], own[Q], ext[Q], f[Q], g[N];
              if constexpr (GLL) {
#pragma unroll
                for (int i = 0; i < N; ++i) nd[i] = r[(s ? N - 1 : 0) * N + i];
              } else {
#pragma unroll
                for (int i = 0; i < N; ++i) {
                  nd[i] = T(0);
#pragma unroll
                  for (int m = 0; m < N; ++m) nd[i] += (s ? b1[m] : b0[m]) * r[m * N + i];
                }
              }
              pin(A);
              pin(nd);
              P::up(B, nd, own);
#pragma unroll
              for (int i = 0; i < N; ++i) nd[i] = r[NN + (2 + s) * N + i];
              P::up(B, nd, ext);
              const bool bnd = neighbour(e, sub, 1, s) < 0;
              if (a.bc_data && bnd) {
#pragma unroll
                for (int k = 0; k < Q; ++k) ext[k] = ge[s][k];
              }
#pragma unroll
              for (int j = 0; j < Q; ++j) f[j] = flux(c, be[s][j], s == 1, own[j], ext[j], bnd);
              P::down(B, f, g);
              if constexpr (GLL) {
#pragma unroll
                for (int i = 0; i < N; ++i) A[s ? N - 1 : 0][i] += g[i];
              } else {
#pragma unroll
                for (int m = 0; m < N; ++m)
#pragma unroll
                  for (int i = 0; i < N; ++i) A[m][i] += (s ? b1[m] : b0[m]) * g[i];
              }
            }
          }
          beta_at(1, e, sub, sm, kz, wz, b);
#pragma unroll
          for (int k = 0; k < Q; ++k) {
            T f[Q], g[N];
            pin(A);
            pin(v[k]);
#pragma unroll
            for (int j = 0; j < Q; ++j) f[j] = -c * b[k][j] * v[k][j];
            P::down(B, f, g);
            add(A, Gb, k, g);
          }
        }
      }
      if constexpr (!ADV) {
        // the generic kernel's products in its order, so that mass applies (and
        // the CG iterations that use them) keep its bits
        P::points(a.sigma_tab, sub, kz, b);
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          T f[Q], g[N];
#pragma unroll
          for (int j = 0; j < Q; ++j) f[j] = a.mass_coef * (w[j] * w[k] * wz * a.detJ * b[k][j] * v[k][j]);
          P::down(B, f, g);
          add(A, B, k, g);
        }
      } else if (a.mass_coef != T(0)) {
        const T c = a.mass_coef * a.detJ;
        if constexpr (FIELD == kPointwise) P::template separable<false>(a.sigma, rows(sm), kz, w, T(1), b);
        else P::template separable<true>(a.sigma, rows(sm), kz, w, wz, b);
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          T f[Q], g[N];
          pin(A);
          pin(v[k]);
#pragma unroll
          for (int j = 0; j < Q; ++j) f[j] = c * b[k][j] * v[k][j];
          P::down(B, f, g);
          add(A, B, k, g);
        }
      }
      if constexpr (ADV) {  // z component: tested with B' in z, kept apart
        const T c = a.adv_coef * a.detJ * a.invh[2];
        beta_at(2, e, sub, sm, kz, wz, b);
        // the part tested with B in z leaves first: its registers are free
        // for this one.  The record's inputs are all consumed by here.
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) {
            r[m * N + i] = A[m][i];
            A[m][i] = T(0);
          }
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          T f[Q], g[N];
          pin(A);
          pin(v[k]);
#pragma unroll
          for (int j = 0; j < Q; ++j) f[j] = -c * b[k][j] * v[k][j];
          P::down(B, f, g);
          add(A, B, k, g);
        }
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) r[NN + m * N + i] = A[m][i];
      } else {
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) r[m * N + i] = A[m][i];
      }
    }
  } else {
    for (int t = tid - G::CELLW; t < ne * 2; t += NT - G::CELLW) {
      const int el = t >> 1, s = t & 1;
      const int e = e0 + el;
      int sub[3];
      decode(e, sub);
      T* r = rec + (el * PL + Q + s) * PITCH;
      const T* sm = smp + el * a.spitch;
      T b[Q][Q], u[N][N], A[N][N];
      beta_at(2, e, sub, sm, Q + s, T(1), b);
      const bool bnd = neighbour(e, sub, 2, s) < 0;
      const bool skip = bnd && a.bc_none;  // no flux, whatever the field is there (it may be infinite)
      const T c = a.adv_coef * a.detJ * a.invh[2];
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          u[m][i] = r[m * N + i];
          A[m][i] = T(0);
        }
      auto point_row = [&](int k, const T (&ext)[Q]) {
        T own[Q], f[Q], g[N];
        pin(A);
        pin(u);
        P::row(B, u, k, g);
        P::up(B, g, own);
#pragma unroll
        for (int j = 0; j < Q; ++j) {
          const T dot = s ? b[k][j] : -b[k][j];
          T up = c * (dot > T(0) ? dot * own[j] : dot * ext[j]);
          if constexpr (FIELD == kPointwise) up *= w[k] * w[j];
          f[j] = skip ? T(0) : up;
        }
        P::down(B, f, g);
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) A[m][i] += B(k, m) * g[i];
      };
      if (a.bc_data && bnd) {
        T gb[Q][Q];
        P::template separable<false>(a.bc, rows(sm), Q + s, w, T(1), gb);
#pragma unroll
        for (int k = 0; k < Q; ++k) point_row(k, gb[k]);
      } else {
        T w[N][N];
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
          for (int i = 0; i < N; ++i) w[m][i] = r[NN + m * N + i];
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          T g[N], ext[Q];
          pin(A);
          pin(w);
          P::row(B, w, k, g);
          P::up(B, g, ext);
          point_row(k, ext);
        }
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) r[m * N + i] = A[m][i];
    }
  }
  __syncthreads();

  // ---- phase 3: z test functions ----
  for (int t = tid; t < ne * NN; t += NT) {
    const int el = t / NN, c = t - el * NN;
    const T* r = rec + el * PL * PITCH + c;
    T f[Q], o[N];
#pragma unroll
    for (int q = 0; q < Q; ++q) f[q] = r[q * PITCH];
    P::down(B, f, o);
    if constexpr (ADV) {
      T o2[N];
#pragma unroll
      for (int q = 0; q < Q; ++q) f[q] = r[q * PITCH + NN];
      P::down(Gb, f, o2);
      const T lo = r[Q * PITCH], hi = r[(Q + 1) * PITCH];
#pragma unroll
      for (int i = 0; i < N; ++i) o[i] += o2[i];
      if constexpr (GLL) {
        o[0] += lo;
        o[N - 1] += hi;
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] += b0[i] * lo + b1[i] * hi;
      }
    }
    T* dst = y + (int64_t)(e0 + el) * ND + c;
#pragma unroll
    for (int i = 0; i < N; ++i) dst[i * NN] = o[i];
  }
}

}  // namespace pl
}  // namespace gd
