// gfx950 kernel of the uniform 4D-6D apply as a sum of Kronecker products: any
// basis and rule, every advection component a constant or a function of one
// coordinate that keeps one sign on the faces, sigma a sum of terms of at most
// two factors, no inflow data other than 0 (advectionoperator.hpp:106-441 and
// massoperator.hpp:39-89 regrouped; the tensor rule factorises every integral,
// so this is the same operator).
//
// With M the 1D mass matrix on the rule, every term is M along all axes but at
// most two, so it is written as (M (x) .. (x) M) of a product along those two:
//   y = (M (x) .. (x) M) [ sum_k s_k A_k (along a_k) B_k (along b_k) u
//                          + inflow: s_k f_k (along a_k) (x) B_k slab_k ]
// A_k = M^-1 (own face - D), f_k = -+M^-1 b(inflow end), B_k = M^-1 B^T W beta B
// for component k (a_k its axis, b_k the axis its field depends on); both
// matrices have one row set per element position along their axis.
// A sum of t terms costs 2 t + D one-dimensional contractions of n^D values
// whatever q is; the quadrature kernel's 2 D + 2 t ones work on up to q^D.
//
// A thread holds the n x n slice of two axes at fixed other indices; a block
// takes as many elements as fill its threads.  U and the sum V stay in LDS
// through all passes, with the block's matrices.
//
// Rounding: M^-1 in the terms and M behind them amplify what the terms round.
// So the matrices are formed in extended precision, rounded once; M is held in FP64
// in units in which its entries round to almost nothing, and the passes with it
// multiply in FP64 in either precision (an FP64 FMA costs what an FP32 one
// does); a term's sum is formed apart and added once; with n = 2, where the
// quadrature kernel has the fewest sums, the terms are formed in FP64 too.
// Error against an extended-precision apply, in units of the generic kernel's:
// FP64 Lobatto up to 1.5 before, 0.05 to 0.64 now (Legendre, on the generic
// kernel's tables, 0.8 to 1.1); FP32 up to 4.4 before (n = 3, q = 4 Lobatto), 0.2
// to 1.1 now.  FP32 applies before and now: 6D p = 2 82 and 88 us, 6D p = 1 10.9
// and 13.0, 4D p = 3 22.3 and 23.6; FP64 unchanged.
//
// 6 x 6 x 6 x 5 x 5 x 5 elements, p = 2, q = 3, beta = (v, a), FP64 (315 MB in
// and out): 163 us against 2,650 us for the generic kernel.  Bound by the waits
// of the passes (60 % of the wave cycles), then VALU issue (60 us) and LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "gd_plane.hpp"
#include "gd_sizing.hpp"

namespace gd {
namespace kron {

constexpr int kMaxTermsK = 10;  // D components and up to four sigma terms

// One term on the device: matrices [position][n][n] along its axes
template <typename T>
struct Term {
  int a, b;            // axes; b: the matrix tb is along b (tb nullptr: none)
  int inflow;          // 0: no face; +1: the lower neighbour's upper end flows in, -1: the upper neighbour's lower end
  const T *ta, *tb, *tf;  // tf: [position along a][n]
  int stride[6];       // strides of the other axes, ascending, then of a and b
};

template <typename T>
struct Args {
  int E, epb, num_blocks, nterms, mpitch;
  int M[6];
  pl::FastDiv dv[5];
  int periodic_mask;
  double km;            // constant part of sigma
  T coef[kMaxTermsK];   // factors of the terms
  const double* Mm;
  const T *b0, *b1;
  Term<T> t[kMaxTermsK];
};

template <int B, int E>
constexpr int ipow() { int r = 1; for (int i = 0; i < E; ++i) r *= B; return r; }

template <typename T, int D, int N>
struct Geo {
  static constexpr int ND = ipow<N, D>();
  static constexpr int NS = ipow<N, D - 2>();  // slices of a pair of axes
  static constexpr int PITCH = ND | 1;
  // elements that fill 256 threads with slices, within 40 KB of U and V
  static constexpr int FILL = 256 / NS < 1 ? 1 : 256 / NS;
  static constexpr int ROOM = 40 * 1024 / (2 * PITCH * (int)sizeof(T));
  static constexpr int EPB = ROOM < 1 ? 1 : (FILL < ROOM ? FILL : ROOM);
  static constexpr int NT = EPB * NS >= 256 ? 256 : (EPB * NS + 63) / 64 * 64;
  static constexpr int TW = 2 * N * N + N;  // matrix words per element and term
};

template <typename T, int D, int N, bool GLL>
__global__ void __launch_bounds__((Geo<T, D, N>::NT)) kron_kernel(Args<T> p, const T* __restrict__ x, T* __restrict__ y)
{
  using G = Geo<T, D, N>;
  constexpr int ND = G::ND, NS = G::NS, PITCH = G::PITCH, NT = G::NT, NN = N * N, TW = G::TW;
  using C = std::conditional_t<N == 2, double, T>;  // the terms' arithmetic
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* U = reinterpret_cast<T*>(smem_raw);
  T* V = U + p.epb * PITCH;
  T* mat = V + p.epb * PITCH;  // [element][term]: A, B, f
  int* nbs = reinterpret_cast<int*>(mat + p.epb * p.mpitch);  // [element][term] inflow neighbour

  const int blk = dev::xcd_remap(blockIdx.x, p.num_blocks);
  const int e0 = blk * p.epb;
  const int ne = p.E - e0 < p.epb ? p.E - e0 : p.epb;
  const int tid = threadIdx.x;

  for (int i = tid; i < ne * ND; i += NT) {
    const int el = i / ND;
    U[el * PITCH + (i - el * ND)] = x[(int64_t)e0 * ND + i];
  }
  // the matrices of each (element, term), and its inflow neighbour
  for (int t = tid; t < ne * p.nterms * TW; t += NT) {
    const int el = t / (p.nterms * TW), r = t - el * (p.nterms * TW);
    const int k = r / TW, i = r - k * TW;
    const Term<T>& tm = p.t[k];
    const int ax = i >= NN && i < 2 * NN ? tm.b : tm.a;
    int rem = e0 + el, pos = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int q = d < D - 1 ? pl::div(p.dv[d], rem) : 0;
      const int s = rem - q * (d < D - 1 ? p.M[d] : 0);
      if (d == ax) pos = s;
      rem = q;
    }
    T v = T(0);
    if (i < NN) v = p.coef[k] * tm.ta[pos * NN + i];
    else if (i < 2 * NN) v = tm.tb ? tm.tb[pos * NN + i - NN] : T(0);
    else if (tm.inflow) v = p.coef[k] * tm.tf[pos * N + i - 2 * NN];
    mat[el * p.mpitch + k * TW + i] = v;
  }
  for (int t = tid; t < ne * p.nterms; t += NT) {
    const int el = t / p.nterms, k = t - el * p.nterms;
    const int dir = p.t[k].inflow, ax = p.t[k].a, e = e0 + el;
    int nb = -1, rem = e, st = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int q = d < D - 1 ? pl::div(p.dv[d], rem) : 0;
      const int s = rem - q * (d < D - 1 ? p.M[d] : 0);
      if (d == ax && dir) {
        const bool per = (p.periodic_mask >> d) & 1;
        if (dir > 0) nb = s > 0 ? e - st : (per ? e + (p.M[d] - 1) * st : -1);
        else nb = s < p.M[d] - 1 ? e + st : (per ? e - (p.M[d] - 1) * st : -1);
      }
      st *= p.M[d];
      rem = q;
    }
    nbs[t] = nb;
  }
  __syncthreads();

  // one slice per (element, thread): its digits along the D - 2 other axes
  for (int k = 0; k < p.nterms; ++k) {
    const Term<T>& tm = p.t[k];
    const bool two = tm.tb != nullptr, face = tm.inflow != 0;
    const int sa = tm.stride[D - 2], sb = tm.stride[D - 1];
    for (int t = tid; t < ne * NS; t += NT) {
      const int el = t / NS;
      int r = t - el * NS, base = 0;
#pragma unroll
      for (int j = 0; j < D - 2; ++j) {
        base += (r % N) * tm.stride[j];
        r /= N;
      }
      const T* mk = mat + el * p.mpitch + k * TW;
      const int nb = face ? nbs[el * p.nterms + k] : -1;
      // the neighbour's line at the shared face, along b
      C s[N];
#pragma unroll
      for (int j = 0; j < N; ++j) s[j] = C(0);
      if (nb >= 0) {
        const T* src = x + (int64_t)nb * ND + base;
        if constexpr (GLL) {
          src += tm.inflow > 0 ? (N - 1) * sa : 0;
#pragma unroll
          for (int j = 0; j < N; ++j) s[j] = src[j * sb];
        } else {
          const T* be = tm.inflow > 0 ? p.b1 : p.b0;
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const C c = be[i];
#pragma unroll
            for (int j = 0; j < N; ++j) s[j] += c * src[i * sa + j * sb];
          }
        }
      }
      C S[N][N];
      const T* u = U + el * PITCH + base;
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) S[i][j] = u[i * sa + j * sb];
      T* v = V + el * PITCH + base;
      C W[N][N];
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) W[i][j] = k == 0 ? (C)p.km * S[i][j] : v[i * sa + j * sb];
      if (two) {
        C R[N][N], q[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
          q[j] = C(0);
#pragma unroll
          for (int i = 0; i < N; ++i) R[i][j] = C(0);
        }
#pragma unroll
        for (int l = 0; l < N; ++l)
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const C m = mk[NN + j * N + l];
            q[j] += m * s[l];
#pragma unroll
            for (int i = 0; i < N; ++i) R[i][j] += m * S[i][l];
          }
#pragma unroll
        for (int j = 0; j < N; ++j) {
          s[j] = q[j];
#pragma unroll
          for (int i = 0; i < N; ++i) S[i][j] = R[i][j];
        }
      }
      C Z[N][N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const C f = face ? mk[2 * NN + i] : T(0);
#pragma unroll
        for (int j = 0; j < N; ++j) Z[i][j] = f * s[j];
      }
#pragma unroll
      for (int l = 0; l < N; ++l)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const C m = mk[i * N + l];
#pragma unroll
          for (int j = 0; j < N; ++j) Z[i][j] += m * S[l][j];
        }
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) v[i * sa + j * sb] = (T)(W[i][j] + Z[i][j]);
    }
    __syncthreads();
  }

  // M along every axis, two at a time; the last pair goes out
  pl::CPtr<double> M = (pl::CPtr<double>)p.Mm;
  const T* from = p.nterms ? V : U;
  const double first = p.nterms ? 1.0 : p.km;
  constexpr int PAIRS = (D + 1) / 2;
  dev::static_for<0, PAIRS>([&](auto pr_) {
    constexpr int pr = decltype(pr_)::value;
    // odd D: the first pass takes axis 0 alone with axis 1 untouched
    constexpr bool single = D % 2 == 1 && pr == 0;
    constexpr int A = D % 2 == 0 ? 2 * pr : (pr == 0 ? 0 : 2 * pr - 1);
    constexpr int Bx = A + 1;
    constexpr int sa = ipow<N, A>(), sb = ipow<N, Bx>();
    constexpr bool last = pr == PAIRS - 1;
    for (int t = tid; t < ne * NS; t += NT) {
      const int el = t / NS, r = t - el * NS;
      const int lowd = r % sa, high = r / sa;  // axes below A, above Bx
      const int base = lowd + high * (sb * N);
      const T* src = (pr == 0 ? from : V) + el * PITCH + base;
      double S[N][N], R[N][N];
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) {
          S[i][j] = src[i * sa + j * sb];
          if constexpr (pr == 0) S[i][j] *= first;
        }
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) {
          double q = M[i * N] * S[0][j];
#pragma unroll
          for (int l = 1; l < N; ++l) q += M[i * N + l] * S[l][j];
          R[i][j] = q;
        }
      if constexpr (!single) {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int j = 0; j < N; ++j) {
            double q = M[j * N] * R[i][0];
#pragma unroll
            for (int l = 1; l < N; ++l) q += M[j * N + l] * R[i][l];
            S[i][j] = q;
          }
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int j = 0; j < N; ++j) S[i][j] = R[i][j];
      }
      if constexpr (last) {
        T* dst = y + (int64_t)(e0 + el) * ND + base;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int j = 0; j < N; ++j) dst[i * sa + j * sb] = (T)S[i][j];
      } else {
        T* dst = V + el * PITCH + base;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int j = 0; j < N; ++j) dst[i * sa + j * sb] = (T)S[i][j];
      }
    }
    if constexpr (!last) __syncthreads();
  });
}

template <typename T, int D, int N, bool GLL>
int launch(Args<T>& a, const T* x, T* y, hipStream_t s)
{
  using G = Geo<T, D, N>;
  a.mpitch = (a.nterms * G::TW) | 1;
  auto kern = kron_kernel<T, D, N, GLL>;
  static const int resident = blocks_per_cu(kern, G::NT);
  const size_t per = (2 * G::PITCH + a.mpitch) * sizeof(T) + a.nterms * sizeof(int);
  a.epb = elements_per_block(a.E, 1, G::EPB, per, resident);
  a.num_blocks = (int)(((int64_t)a.E + a.epb - 1) / a.epb);
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

template <typename T, int D, int N>
int launch_any(Args<T>& a, bool gll, const T* x, T* y, hipStream_t s)
{
  return gll ? launch<T, D, N, true>(a, x, y, s) : launch<T, D, N, false>(a, x, y, s);
}

}  // namespace kron
}  // namespace gd
