// Device-resident Arnoldi process for restarted GMRES(m), m <= 32.
//
// One iteration k (basis vectors V_0..V_k stored with scales s_j, true vector
// v_j = s_j V_j, and W = V_{k+1} holding K V_k) is three fused passes over the
// basis:
//   pass A: h1_j = s_j <V_j, W>                         (classical GS)
//   pass B: W -= sum_j s_j h1_j V_j, then h2_j = s_j <V_j, W>, ||W||^2
//           (re-orthogonalisation, the "twice is enough" CGS2 step)
//   pass C: Z = (W - sum_j s_j h2_j V_j) / p with p^2 = ||W||^2 - sum_j h2_j^2
//           (Pythagoras), stored as V_{k+1}; nu = ||Z|| exactly; s_{k+1} = 1/nu
// then the Hessenberg column H_{jk} = s_k (h1_j + h2_j), H_{k+1,k} = s_k p nu is
// formed and rotated by the previous Givens rotations and a new one
// (gmres.hpp:170-210).  Stored vectors are kept at unit norm (up to rounding),
// so the operator is applied with scale 1 and FP32 bases cannot drift out of
// range.
//
// The passes are bandwidth-bound (FP32, 2.1 M values, 30 vectors: 252 MB in
// ~47 us), so what is left to save is the time between them.  Each pass leaves
// one partial per block and column; the next pass sums them in its own prologue,
// every block for itself in the same fixed order (at most 256 partials of 33
// columns, 512 of 9, or 512 of 32 in FP64: 36 to 128 KB from L2), and pass C's
// column is finished by one wave of the next step's pass A (or by a one-wave
// kernel before the cycle's update).  Against one-block finishing kernels between
// the passes (4-6 us each and a launch gap): the 32^3, p = 3 implicit step in
// mixed precision (47 cycles of 30) 160.6 -> 145.4 ms.  Walking every second pass
// downwards for the L2 and loading the first packs before the sums measured the
// same, with spills.
//
// The residual estimate |g_{k+1}| goes to the caller's pointer (pinned host
// memory, so a host loop can poll it with no copy or event in the stream) from
// the first block of the next kernel on the workspace that runs on for a while
// (the next step's pass A or the cycle's update): a store to host memory at the
// end of a kernel holds the kernel's completion for the bus round trip.
//
// Bases are read 16 bytes per lane where the basis and its leading dimension
// are 16-byte aligned (pass B in FP32, which keeps every loaded value live, 8
// bytes): one block per CU needs that many bytes in flight (with 8 in FP64 a solve
// took 5 % longer).  FP64 passes A and C take two blocks per CU for any number of
// vectors (pass B's registers hold one): FP64 solves, 32^3, p = 3 (1885 iterations)
// 402 ms with one block, 376 with two (399 with the finishing kernels), 16^3 81,
// 80 (103), 28^3, p = 2 41.9, 40.6 (47.3).
//
// The cycle end solves the triangular system H y = g in one wave (with the last
// column's finish) and adds x += sum_j s_j y_j V_j in FP64.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "gd_internal.hpp"
#include "gd_reduce.hpp"

namespace gd {
namespace arnoldi {

constexpr int kThreads = 512;       // two waves per SIMD: up to 256 registers for the loads in flight
constexpr int kMaxM = 32;           // restart length
constexpr int kStride = kMaxM + 1;  // partial columns per block: k+1 dots + norm
constexpr int kMaxBlocks = 512;     // partials per column
// blocks of a pass over KK vectors: two per CU while there are few loads per
// thread (and few columns to sum), else one
constexpr int max_blocks(int KK) { return KK <= 8 ? kMaxBlocks : kMaxBlocks / 2; }
// of passes A and C: more in flight for FP64 vectors, twice as long
template <typename TV>
constexpr int max_blocks_ac(int KK) { return sizeof(TV) == 8 ? kMaxBlocks : max_blocks(KK); }

struct Workspace {
  double H[kMaxM][kMaxM + 1];  // column k, rows 0..k+1 (rotated)
  double cs[kMaxM], sn[kMaxM];
  double g[kMaxM + 1];
  double s[kMaxM + 1];
  double c[kMaxM];   // coefficients on the stored vectors for the cycle's update
  double h1[kMaxM];  // accumulated true GS coefficients of the current column
  double pnorm;
  int owed, owed_blocks;  // columns whose rotation is still to be formed (its number + 1, or 0), partials in pc
  double* owed_out;       // where that column's residual estimate goes
  double* pending;        // caller pointer still owed the last residual estimate
  double pending_value;
  double pa[kMaxM][kMaxBlocks];  // [column][block]: a column is contiguous
  double pb[kStride][kMaxBlocks];
  double pc[kMaxBlocks];
};

// W values of one vector, loaded or stored as one access of up to 16 bytes
// alignment (a 32-byte pack is two 16-byte accesses)
template <typename T, int W>
struct alignas(W * sizeof(T) > 16 ? 16 : W * sizeof(T)) Pack {
  T v[W];
};

template <typename T, int W>
__device__ __forceinline__ Pack<T, W> ld(const T* p)
{
  return *reinterpret_cast<const Pack<T, W>*>(p);
}

template <typename T, int W>
__device__ __forceinline__ void st(T* p, const Pack<T, W>& v)
{
  *reinterpret_cast<Pack<T, W>*>(p) = v;
}

// One pack per thread until the grid is at its largest: a small basis spread
// over all CUs (four packs per thread left 28^3 p = 2 in FP32 on 72 of them:
// 37.2 ms a solve against 29.0; start 33.7).
inline int grid_for(int64_t n, int w, int most)
{
  const int64_t per = (int64_t)kThreads * w;
  const int64_t b = (n + per - 1) / per;
  return (int)(b < 1 ? 1 : (b > most ? most : b));
}

// Lane i's value, i the same in the whole wave.
__device__ __forceinline__ double lane_value(double v, int i)
{
  union {
    double d;
    int w[2];
  } u{v};
  u.w[0] = __builtin_amdgcn_readlane(u.w[0], i);
  u.w[1] = __builtin_amdgcn_readlane(u.w[1], i);
  return u.d;
}

template <int K>
__device__ __forceinline__ void store_block_partials(const double (&acc)[K], double (*partial)[kMaxBlocks])
{
  __shared__ double row[K];
  red::block_sum<kThreads, K>(acc, row);
  for (int j = threadIdx.x; j < K; j += kThreads) partial[j][blockIdx.x] = row[j];
}

// col[j] = sum over nblk <= MAXB partials of column j, j < K: TPC threads per
// column, the loads of 256 partials in flight together, then a shuffle sum; a
// fixed order for a given grid.  Visible to every thread on return.
template <int K, int MAXB>
__device__ __forceinline__ void sum_columns(const double (*partial)[kMaxBlocks], int nblk, double* col)
{
  constexpr int TPC = K <= 8 ? 64 : K <= 16 ? 32 : 16;
  constexpr int CPP = kThreads / TPC;  // columns per round
  constexpr int ROUND = MAXB < 256 ? MAXB : 256;
  constexpr int PER = ROUND / TPC;     // partials per thread and round
  const int lane = threadIdx.x % TPC, c0 = threadIdx.x / TPC;
#pragma unroll
  for (int r = 0; r < (K + CPP - 1) / CPP; ++r) {
    const int j = c0 + r * CPP;
    if (j < K) {  // uniform over each group of TPC threads; the shuffles stay inside it
      const double* cp = partial[j];
      double sum = 0.0;
#pragma unroll 1
      for (int b0 = 0; b0 < nblk; b0 += ROUND) {  // nblk is the same in every thread
        double v[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int bb = b0 + lane + TPC * i;
          const double x = cp[bb < nblk ? bb : nblk - 1];
          v[i] = bb < nblk ? x : 0.0;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) sum += v[i];
      }
#pragma unroll
      for (int off = TPC / 2; off > 0; off >>= 1) sum += __shfl_down(sum, off, TPC);
      if (lane == 0) col[j] = sum;
    }
  }
  __syncthreads();
}

// One whole wave: the owed column of the Hessenberg matrix (row j in lane j),
// its Givens rotation and residual estimate (left pending).
__device__ __forceinline__ void finish_column(Workspace* __restrict__ ws)
{
  const int owed = ws->owed;
  if (owed == 0) return;
  const int k = owed - 1, lane = threadIdx.x & 63, nblk = ws->owed_blocks;
  double part = 0.0;
#pragma unroll
  for (int i = 0; i < kMaxBlocks / 64; ++i) {
    const int bb = lane + 64 * i;
    const double x = ws->pc[bb < nblk ? bb : nblk - 1];
    part += bb < nblk ? x : 0.0;
  }
  const double sk = ws->s[k];
  const double c_l = lane < k ? ws->cs[lane] : 1.0, s_l = lane < k ? ws->sn[lane] : 0.0;
  double h = lane <= k ? sk * ws->h1[lane < kMaxM ? lane : 0] : 0.0;
  const double nu = sqrt(lane_value(red::wave_sum(part), 0));
  if (lane == owed) h = sk * ws->pnorm * nu;
  double carry = lane_value(h, 0), out = 0.0;
  for (int i = 0; i < k; ++i) {
    const double b = lane_value(h, i + 1), c = lane_value(c_l, i), sn = lane_value(s_l, i);
    if (lane == i) out = c * carry + sn * b;
    carry = -sn * carry + c * b;
  }
  const double a = carry, b = lane_value(h, owed);
  const double rho = hypot(a, b);
  const double cs = rho > 0.0 ? a / rho : 1.0, sn = rho > 0.0 ? b / rho : 0.0;
  if (lane == k) out = rho;
  if (lane <= owed) ws->H[k][lane] = out;
  if (lane == 0) {
    ws->s[owed] = nu > 0.0 ? 1.0 / nu : 0.0;
    ws->cs[k] = cs;
    ws->sn[k] = sn;
    const double gk = ws->g[k];
    const double g1 = -sn * gk;
    ws->g[owed] = g1;
    ws->g[k] = cs * gk;
    ws->pending = ws->owed_out;
    ws->pending_value = fabs(g1);
    ws->owed = 0;
  }
}

__device__ __forceinline__ void publish_pending(Workspace* ws) { red::publish_pending(&ws->pending, &ws->pending_value); }

// The basis passes take the number of stored vectors KK as a template
// parameter: every load of a pass is then unconditional and independent, so
// all of them are in flight together (a runtime count made each load a
// predicated branch followed by a wait).  W values per lane and access; the
// n % W values past the last whole pack are taken one per lane afterwards.

// Pass A: partial row = <V_j, W>, j < KK.
template <typename TV, int KK, int W>
__global__ void __launch_bounds__(kThreads) k_pass_a(int64_t n, const TV* __restrict__ V, int64_t ldv,
                                                     Workspace* __restrict__ ws)
{
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    finish_column(ws);
    publish_pending(ws);
  }
  const TV* __restrict__ w = V + (int64_t)KK * ldv;
  double acc[KK];
#pragma unroll
  for (int j = 0; j < KK; ++j) acc[j] = 0.0;
  const int64_t nv = n / W, stride = (int64_t)gridDim.x * kThreads;
  const int64_t t0 = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (int64_t i = t0; i < nv; i += stride) {
    const Pack<TV, W> wp = ld<TV, W>(w + i * W);
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      const Pack<TV, W> vp = ld<TV, W>(V + j * ldv + i * W);
#pragma unroll
      for (int l = 0; l < W; ++l) acc[j] += (double)vp.v[l] * (double)wp.v[l];
    }
  }
  for (int64_t i = nv * W + t0; i < n; i += stride) {
    const double wi = (double)w[i];
#pragma unroll
    for (int j = 0; j < KK; ++j) acc[j] += (double)V[j * ldv + i] * wi;
  }
  store_block_partials<KK>(acc, ws->pa);
}

// Pass B: h1_j = s_j <V_j, W>, c_j = s_j h1_j; W -= sum_j c_j V_j; partial row = <V_j, W_new>, ||W_new||^2.
template <typename TV, int KK, int W>
__global__ void __launch_bounds__(kThreads) k_pass_b(int64_t n, TV* __restrict__ V, int64_t ldv, int na,
                                                     Workspace* __restrict__ ws)
{
  TV* __restrict__ w = V + (int64_t)KK * ldv;
  __shared__ double col[KK];
  sum_columns<KK, max_blocks_ac<TV>(KK)>(ws->pa, na, col);
  double c_l = 0.0;
  {
    const int j = threadIdx.x & 63;
    if (j < KK) {
      const double sj = ws->s[j], h = sj * col[j];
      if (blockIdx.x == 0 && threadIdx.x < 64) ws->h1[j] = h;
      c_l = sj * h;
    }
  }
  double cj[KK];
#pragma unroll
  for (int j = 0; j < KK; ++j) cj[j] = lane_value(c_l, j);
  double acc[KK + 1];
#pragma unroll
  for (int j = 0; j <= KK; ++j) acc[j] = 0.0;
  const int64_t nv = n / W, stride = (int64_t)gridDim.x * kThreads;
  const int64_t t0 = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (int64_t i = t0; i < nv; i += stride) {
    Pack<TV, W> vp[KK];
    double s[W];
#pragma unroll
    for (int l = 0; l < W; ++l) s[l] = 0.0;
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      vp[j] = ld<TV, W>(V + j * ldv + i * W);
#pragma unroll
      for (int l = 0; l < W; ++l) s[l] += cj[j] * (double)vp[j].v[l];
    }
    const Pack<TV, W> wp = ld<TV, W>(w + i * W);
    Pack<TV, W> wt;
#pragma unroll
    for (int l = 0; l < W; ++l) wt.v[l] = (TV)((double)wp.v[l] - s[l]);
    st<TV, W>(w + i * W, wt);
#pragma unroll
    for (int l = 0; l < W; ++l) {
      const double wr = (double)wt.v[l];
#pragma unroll
      for (int j = 0; j < KK; ++j) acc[j] += (double)vp[j].v[l] * wr;
      acc[KK] += wr * wr;
    }
  }
  for (int64_t i = nv * W + t0; i < n; i += stride) {
    double v[KK];
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      v[j] = (double)V[j * ldv + i];
      s += cj[j] * v[j];
    }
    const TV wt = (TV)((double)w[i] - s);
    w[i] = wt;
    const double wr = (double)wt;
#pragma unroll
    for (int j = 0; j < KK; ++j) acc[j] += v[j] * wr;
    acc[KK] += wr * wr;
  }
  store_block_partials<KK + 1>(acc, ws->pb);
}

// Pass C: h2_j = s_j <V_j, W>, h1_j += h2_j, c_j = s_j h2_j,
// p = sqrt(||W||^2 - sum_j h2_j^2); Z = (W - sum_j c_j V_j) / p stored as V_KK;
// partial = ||Z||^2.
template <typename TV, int KK, int W>
__global__ void __launch_bounds__(kThreads) k_pass_c(int64_t n, TV* __restrict__ V, int64_t ldv, int nb,
                                                     Workspace* __restrict__ ws, double* resid_out)
{
  TV* __restrict__ w = V + (int64_t)KK * ldv;
  __shared__ double col[KK + 1];
  sum_columns<KK + 1, max_blocks(KK)>(ws->pb, nb, col);
  double c_l = 0.0, h2 = 0.0;
  const int lane = threadIdx.x & 63;
  if (lane < KK) {
    const double sj = ws->s[lane];
    h2 = sj * col[lane];
    c_l = sj * h2;
  }
  double cj[KK];
  double ss = 0.0;
#pragma unroll
  for (int j = 0; j < KK; ++j) {
    cj[j] = lane_value(c_l, j);
    const double hj = lane_value(h2, j);
    ss += hj * hj;
  }
  const double p2 = col[KK] - ss;
  const double p = p2 > 0.0 ? sqrt(p2) : 0.0;
  const double pinv = p > 0.0 ? 1.0 / p : 0.0;
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    if (lane < KK) ws->h1[lane] += h2;
    if (lane == 0) {
      ws->pnorm = p;
      ws->owed = KK;
      ws->owed_blocks = gridDim.x;
      ws->owed_out = resid_out;
    }
  }
  double acc[1] = {0.0};
  const int64_t nv = n / W, stride = (int64_t)gridDim.x * kThreads;
  const int64_t t0 = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (int64_t i = t0; i < nv; i += stride) {
    double s[W];
#pragma unroll
    for (int l = 0; l < W; ++l) s[l] = 0.0;
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      const Pack<TV, W> vp = ld<TV, W>(V + j * ldv + i * W);
#pragma unroll
      for (int l = 0; l < W; ++l) s[l] += cj[j] * (double)vp.v[l];
    }
    const Pack<TV, W> wp = ld<TV, W>(w + i * W);
    Pack<TV, W> zt;
#pragma unroll
    for (int l = 0; l < W; ++l) {
      zt.v[l] = (TV)(((double)wp.v[l] - s[l]) * pinv);
      const double zr = (double)zt.v[l];
      acc[0] += zr * zr;
    }
    st<TV, W>(w + i * W, zt);
  }
  for (int64_t i = nv * W + t0; i < n; i += stride) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < KK; ++j) s += cj[j] * (double)V[j * ldv + i];
    const TV zt = (TV)(((double)w[i] - s) * pinv);
    w[i] = zt;
    const double zr = (double)zt;
    acc[0] += zr * zr;
  }
  store_block_partials<1>(acc, &ws->pc);
}

// Cycle start: g = beta e_0, s_0 = s0, no residual estimate owed (the
// workspace may hold anything before the first cycle).
__global__ void k_begin(double beta, double s0, Workspace* __restrict__ ws)
{
  const int t = threadIdx.x;
  if (t <= kMaxM) ws->g[t] = t == 0 ? beta : 0.0;
  if (t == 0) {
    ws->s[0] = s0;
    ws->pending = nullptr;
    ws->owed = 0;
  }
}

// Cycle end, one wave: the last column, then y = H(0:k,0:k)^{-1} g(0:k) by
// columns (row j in lane j) and c_j = s_j y_j.
__global__ void __launch_bounds__(64) k_solve_cycle(int k, Workspace* __restrict__ ws)
{
  finish_column(ws);
  __threadfence_block();
  const int lane = threadIdx.x;
  const int row = lane < k ? lane : 0;
  double acc = ws->g[row];
  for (int i = k - 1; i >= 0; --i) {
    const double hij = ws->H[i][row];
    const double y = lane_value(acc, i) / lane_value(hij, i);
    if (lane == i) acc = y;
    else if (lane < i) acc -= hij * y;
  }
  if (lane < k) ws->c[lane] = ws->s[lane] * acc;
}

// x += sum_j c_j V_j.
template <typename TV, int KK, int W>
__global__ void __launch_bounds__(kThreads) k_update_x(int64_t n, const TV* __restrict__ V, int64_t ldv,
                                                       Workspace* __restrict__ ws, double* __restrict__ x)
{
  publish_pending(ws);
  double cj[KK];
#pragma unroll
  for (int j = 0; j < KK; ++j) cj[j] = ws->c[j];
  const int64_t nv = n / W, stride = (int64_t)gridDim.x * kThreads;
  const int64_t t0 = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (int64_t i = t0; i < nv; i += stride) {
    double s[W];
#pragma unroll
    for (int l = 0; l < W; ++l) s[l] = 0.0;
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      const Pack<TV, W> vp = ld<TV, W>(V + j * ldv + i * W);
#pragma unroll
      for (int l = 0; l < W; ++l) s[l] += cj[j] * (double)vp.v[l];
    }
    Pack<double, W> xp = ld<double, W>(x + i * W);
#pragma unroll
    for (int l = 0; l < W; ++l) xp.v[l] += s[l];
    st<double, W>(x + i * W, xp);
  }
  for (int64_t i = nv * W + t0; i < n; i += stride) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < KK; ++j) s += cj[j] * (double)V[j * ldv + i];
    x[i] += s;
  }
}

// f(std::integral_constant<int, k>) for a runtime 1 <= k <= kMaxM
template <int LO, typename F>
void with_count(int k, F&& f)
{
  if constexpr (LO <= kMaxM) {
    if (k == LO) f(std::integral_constant<int, LO>{});
    else with_count<LO + 1>(k, f);
  }
}

// 16-byte accesses: a 16-byte aligned basis (and x for the update) whose
// leading dimension is a whole number of packs; else one value per lane
template <typename TV>
constexpr int kPack = 16 / (int)sizeof(TV);
template <typename TV>
bool packed(const void* V, int64_t ldv, const void* x = nullptr)
{
  return reinterpret_cast<uintptr_t>(V) % 16 == 0 && ldv % kPack<TV> == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
}

template <typename TV>
int step(int64_t n, int m, int k, TV* V, int64_t ldv, void* wsp, double* resid_out, hipStream_t st)
{
  if (n < 1 || m < 1 || m > kMaxM || k < 0 || k >= m || !V || !wsp || ldv < n)
    return fail(GD_ERR_INVALID, "gd_arnoldi_step: bad arguments");
  Workspace* ws = static_cast<Workspace*>(wsp);
  auto launch = [&](auto W_) {
    constexpr int W = decltype(W_)::value;
    // pass B keeps every loaded value until the updated W is known: at most
    // two values per lane, so 32 stored vectors stay in registers
    constexpr int WB = W < 2 ? W : 2;
    with_count<1>(k + 1, [&](auto KK_) {
      constexpr int KK = decltype(KK_)::value;
      const int nb = grid_for(n, W, max_blocks(KK)), na = grid_for(n, W, max_blocks_ac<TV>(KK));
      hipLaunchKernelGGL((k_pass_a<TV, KK, W>), dim3(na), dim3(kThreads), 0, st, n, V, ldv, ws);
      hipLaunchKernelGGL((k_pass_b<TV, KK, WB>), dim3(nb), dim3(kThreads), 0, st, n, V, ldv, na, ws);
      hipLaunchKernelGGL((k_pass_c<TV, KK, W>), dim3(na), dim3(kThreads), 0, st, n, V, ldv, nb, ws, resid_out);
    });
  };
  if (packed<TV>(V, ldv)) launch(std::integral_constant<int, kPack<TV>>{});
  else launch(std::integral_constant<int, 1>{});
  GD_HIP(hipGetLastError());
  return GD_OK;
}

template <typename TV>
int update(int64_t n, int m, int k, const TV* V, int64_t ldv, void* wsp, double* x, hipStream_t st)
{
  if (n < 1 || m < 1 || m > kMaxM || k < 0 || k > m || !V || !wsp || !x || ldv < n)
    return fail(GD_ERR_INVALID, "gd_gmres_update: bad arguments");
  if (k == 0) return GD_OK;
  Workspace* ws = static_cast<Workspace*>(wsp);
  auto launch = [&](auto W_) {
    constexpr int W = decltype(W_)::value;
    hipLaunchKernelGGL(k_solve_cycle, dim3(1), dim3(64), 0, st, k, ws);
    with_count<1>(k, [&](auto KK_) {
      constexpr int KK = decltype(KK_)::value;
      hipLaunchKernelGGL((k_update_x<TV, KK, W>), dim3(grid_for(n, W, 2 * kMaxBlocks)), dim3(kThreads), 0, st, n, V, ldv, ws, x);
    });
  };
  if (packed<TV>(V, ldv, x)) launch(std::integral_constant<int, kPack<TV>>{});
  else launch(std::integral_constant<int, 1>{});
  GD_HIP(hipGetLastError());
  return GD_OK;
}

}  // namespace arnoldi
}  // namespace gd

using gd::fail;

extern "C" {

size_t gd_gmres_workspace_bytes(void) { return sizeof(gd::arnoldi::Workspace); }

int gd_gmres_begin(void* ws, double beta, double s0, gd_stream stream)
{
  if (!ws) return fail(GD_ERR_INVALID, "gd_gmres_begin: null workspace");
  hipLaunchKernelGGL(gd::arnoldi::k_begin, dim3(1), dim3(64), 0, (hipStream_t)stream, beta, s0,
                     static_cast<gd::arnoldi::Workspace*>(ws));
  GD_HIP(hipGetLastError());
  return GD_OK;
}

int gd_arnoldi_step_f64(int64_t n, int32_t m, int32_t k, double* V, int64_t ldv, void* ws, double* resid_out,
                        gd_stream stream)
{
  return gd::arnoldi::step<double>(n, m, k, V, ldv, ws, resid_out, (hipStream_t)stream);
}

int gd_arnoldi_step_f32(int64_t n, int32_t m, int32_t k, float* V, int64_t ldv, void* ws, double* resid_out,
                        gd_stream stream)
{
  return gd::arnoldi::step<float>(n, m, k, V, ldv, ws, resid_out, (hipStream_t)stream);
}

int gd_gmres_update_f64(int64_t n, int32_t m, int32_t k, const double* V, int64_t ldv, void* ws, double* x,
                        gd_stream stream)
{
  return gd::arnoldi::update<double>(n, m, k, V, ldv, ws, x, (hipStream_t)stream);
}

int gd_gmres_update_f32(int64_t n, int32_t m, int32_t k, const float* V, int64_t ldv, void* ws, double* x,
                        gd_stream stream)
{
  return gd::arnoldi::update<float>(n, m, k, V, ldv, ws, x, (hipStream_t)stream);
}

}  // extern "C"
