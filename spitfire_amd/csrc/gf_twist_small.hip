// Twisted block factorisation (gf_twist.hip) for many systems of small blocks (1..11 unknowns): one wave per chain, the
// block in the wave's registers, no barriers inside an inverse. The MFMA kernel pads a block to panels of eight and
// tiles of sixteen and keeps several waves per chain; once the systems alone fill the chip, small blocks are faster
// without either (launch_btd_inv_factor). The same for the one-block systems of large batches of larger blocks: nothing is
// padded, and none of a chain's LDS is held for a block that has no neighbours.
#include "gf_internal.h"
#include "gf_wave.h"
#include "../../include/griffon_amd.h"

#include <utility>

namespace gfa {

namespace {

using wave::lane_value;
using wave::wave_first_argmax;

// Gauss-Jordan inverse of an N x N block held in the registers of one wave, with partial (row) pivoting.
//
// Layout: lane l holds one row, x[k] the entry in slot k. The entry of lane l, slot k is element
// (rowid of lane l, colid of slot k) of the logical matrix, where colid of slot k is held by lane k of
// `colid`. Rows are never interchanged: the pivot of step j is the unused lane with the largest |entry| in
// the pivot column (ties: lowest lane), and the exchange at (pivot lane p, slot j) is done in place. After N
// steps the block holds the inverse in the same kind of layout: the lane pivoted at step j holds row
// colid_j of the inverse, slot j holds its column rowid_{p_j}.
//
// The slots form a queue: the pivot column is always x[0]; each step shifts the other columns down by one
// and appends the transformed pivot column at x[N-1], so that all register indices are compile-time
// constants and after N steps every column is back in its slot. The pivot row is broadcast through scalar
// registers (readlane), so a step has no LDS traffic and no barrier.
//
// Row scaling is deferred: lane r keeps its row unscaled and a factor sig_r, the true row being sig_r times
// the stored one. Every row is pivoted exactly once and has sig = 1 until then, so at the step that pivots
// lane p (stored pivot value d):
//   rows r != p:   x_r[c] -= g_r x_p[c] (c != k),  x_r[k] = -g_r,  with g_r = x_r[k] / d
//   row p:         x_p[c] unchanged,  x_p[k] = 1,  sig_p = 1 / d
// which is the usual step (row p divided by its pivot) with the division of row p left to the end: the update
// of a slot is one fma, with no separate scaling of the pivot row. After N steps every row is multiplied by
// its sig.
template <typename T, int N>
__device__ __forceinline__ void reg_gj_inverse(T (&x)[N], int &rowid, int &colid, int lane) {
  bool used = lane >= N;
  T sig = T(1);
  for (int j = 0; j < N; ++j) {
    const T f = x[0];
    const T rf = T(1) / f;  // every lane's reciprocal, formed beside the pivot search instead of after it
    const int p = wave_first_argmax(fabs(f), !used);  // N - j unused lanes remain, so p >= 0
    const T ipv = lane_value(rf, p);
    const bool isp = lane == p;
    const T g = isp ? T(0) : f * ipv;  // multiplier of the broadcast pivot row (none for the pivot row)
#pragma unroll
    for (int c = 1; c < N; ++c) x[c - 1] = fma(-g, lane_value(x[c], p), x[c]);
    x[N - 1] = isp ? T(1) : -g;  // the pivot column
    if (isp) sig = ipv;
    const int cj = __builtin_amdgcn_readlane(colid, j);
    const int rp = __builtin_amdgcn_readlane(rowid, p);
    if (isp) {
      rowid = cj;
      used = true;
    }
    if (lane == j) colid = rp;
  }
#pragma unroll
  for (int c = 0; c < N; ++c) x[c] *= sig;
}

// Block i of the values in the identity layout (lane = row, slot = column).
template <typename T, int N>
__device__ __forceinline__ void reg_load_block(T (&x)[N], const double *Vi, int &rowid, int &colid, int lane) {
  rowid = lane;
  colid = lane;
#pragma unroll
  for (int k = 0; k < N; ++k) x[k] = lane < N ? (T)Vi[k * N + lane] : T(0);
}

// x <- V_i - diag(rs) X diag(cs), where x holds X (an inverse from the previous block of the chain) in its
// permuted layout; the result keeps that layout.
template <typename T, int N>
__device__ __forceinline__ void reg_schur(T (&x)[N], const double *Vi, const double *rs, const double *cs,
                                          int rowid, int colid, int lane) {
  const bool act = lane < N;
  const double r = act ? rs[rowid] : 0.;
  const double csl = act ? cs[lane] : 0.;  // lane q holds cs[q]
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int c = __builtin_amdgcn_readlane(colid, k);
    const double cc = lane_value(csl, c);
    if (act) x[k] = (T)(Vi[c * N + rowid] - r * cc * (double)x[k]);
  }
}

template <typename T, int N>
__device__ __forceinline__ void reg_store_block(const T (&x)[N], T *Di, int rowid, int colid, int lane) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int c = __builtin_amdgcn_readlane(colid, k);
    if (lane < N) Di[c * N + rowid] = x[k];
  }
}

// Twisted (burn-at-both-ends) block factorisation, one workgroup of two waves per system. Row i of the
// system is diag(sub_{i-1}) x_{i-1} + V_i x_i + diag(sup_i) x_{i+1} = b_i; with m = (n - 1) / 2
//   wave 0:  D_0 = V_0,      D_i = V_i - diag(sub_{i-1}) D_{i-1}^{-1} diag(sup_{i-1}),  i = 1 .. m-1
//   wave 1:  E_{n-1} = V_{n-1},  E_i = V_i - diag(sup_i) E_{i+1}^{-1} diag(sub_i),      i = n-2 .. m+1
//   middle:  C_m = V_m - diag(sub_{m-1}) D_{m-1}^{-1} diag(sup_{m-1}) - diag(sup_m) E_{m+1}^{-1} diag(sub_m)
// and block i of dinv receives D_i^{-1} (i < m), C_m^{-1} (i = m) or E_i^{-1} (i > m), column-major. The top
// half is the reference's forward block Thomas recurrence; running the bottom half at the same time halves
// the serial chain. The bottom wave hands its term of C_m to the top wave through LDS.
template <typename T, int N>
__global__ void __launch_bounds__(128) small_factor_kernel(const int *nblocks, const double *values,
                                                               const long *voff, T *dinv, const long *doff) {
  __shared__ double sb[N * N];
  constexpr long NB2 = (long)N * N;
  const int sys = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const bool top = threadIdx.x < 64;
  const int nb = nblocks[sys];
  const int m = (nb - 1) / 2;
  const double *V = values + voff[sys];
  const double *sub = V + nb * NB2;
  const double *sup = sub + (long)(nb - 1) * N;
  T *Dg = dinv + doff[sys];
  T x[N];
  int rowid = lane, colid = lane;
  const int len = top ? m : nb - 1 - m;
  for (int t = 0; t < len; ++t) {
    const int i = top ? t : nb - 1 - t;
    if (t == 0) reg_load_block<T, N>(x, V + i * NB2, rowid, colid, lane);
    else if (top) reg_schur<T, N>(x, V + i * NB2, sub + (i - 1) * N, sup + (i - 1) * N, rowid, colid, lane);
    else reg_schur<T, N>(x, V + i * NB2, sup + i * N, sub + i * N, rowid, colid, lane);
    reg_gj_inverse<T, N>(x, rowid, colid, lane);
    reg_store_block<T, N>(x, Dg + i * NB2, rowid, colid, lane);
  }
  const bool below = nb - 1 - m > 0;
  if (!top && below) {
    const double r = lane < N ? sup[m * N + rowid] : 0.;
    const double csl = lane < N ? sub[m * N + lane] : 0.;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int c = __builtin_amdgcn_readlane(colid, k);
      const double cc = lane_value(csl, c);
      if (lane < N) sb[c * N + rowid] = r * (double)x[k] * cc;
    }
  }
  __syncthreads();
  if (top) {
    if (m == 0) reg_load_block<T, N>(x, V + m * NB2, rowid, colid, lane);
    else reg_schur<T, N>(x, V + m * NB2, sub + (m - 1) * N, sup + (m - 1) * N, rowid, colid, lane);
    if (below) {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int c = __builtin_amdgcn_readlane(colid, k);
        if (lane < N) x[k] = (T)((double)x[k] - sb[c * N + rowid]);
      }
    }
    reg_gj_inverse<T, N>(x, rowid, colid, lane);
    reg_store_block<T, N>(x, Dg + m * NB2, rowid, colid, lane);
  }
}

// The one-block systems of a batch, one wave each; systems of several blocks are left alone. Four waves per workgroup, so that
// 1,024 systems are a wave for every SIMD (workgroups of one or two waves double up on some: 1,024 blocks of 20 11.9 -> 16.7 us).
template <typename T, int N>
__global__ void __launch_bounds__(256) single_factor_kernel(int nsys, const int *nblocks, const double *values,
                                                            const long *voff, T *dinv, const long *doff) {
  const int sys = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (sys >= nsys || nblocks[sys] != 1) return;
  const int lane = threadIdx.x & 63;
  T x[N];
  int rowid, colid;
  reg_load_block<T, N>(x, values + voff[sys], rowid, colid, lane);
  reg_gj_inverse<T, N>(x, rowid, colid, lane);
  reg_store_block<T, N>(x, dinv + doff[sys], rowid, colid, lane);
}

template <typename T, int N>
void launch_small(int nsys, const int *nblocks, const double *values, const long *voff, T *dinv, const long *doff,
                  hipStream_t st) {
  hipLaunchKernelGGL((small_factor_kernel<T, N>), dim3(nsys), dim3(128), 0, st, nblocks, values, voff, dinv, doff);
}

template <typename T, int N>
void launch_single(int nsys, const int *nblocks, const double *values, const long *voff, T *dinv, const long *doff,
                   hipStream_t st) {
  hipLaunchKernelGGL((single_factor_kernel<T, N>), dim3((nsys + 3) / 4), dim3(256), 0, st, nsys, nblocks, values, voff,
                     dinv, doff);
}

template <typename T>
using SmallFn = void (*)(int, const int *, const double *, const long *, T *, const long *, hipStream_t);

template <typename T, int... I>
SmallFn<T> small_fn(int bs, std::integer_sequence<int, I...>) {
  constexpr SmallFn<T> tab[] = {&launch_small<T, I + 1>...};
  return tab[bs - 1];
}

template <typename T, int... I>
SmallFn<T> single_fn(int bs, std::integer_sequence<int, I...>) {
  constexpr SmallFn<T> tab[] = {&launch_single<T, I + kSingleFrom>...};
  return tab[bs - kSingleFrom];
}

}  // namespace

template <typename T>
int launch_btd_inv_factor_single(int nsys, const int *nblocks, int bs, const double *values, const long *voff, T *dinv,
                                 const long *doff, hipStream_t st) {
  single_fn<T>(bs, std::make_integer_sequence<int, 64 - kSingleFrom + 1>{})(nsys, nblocks, values, voff, dinv, doff, st);
  return hipGetLastError() == hipSuccess ? GF_OK : fail(GF_ERR_HIP, "btd inverse factor launch failed");
}

template int launch_btd_inv_factor_single<double>(int, const int *, int, const double *, const long *, double *,
                                                  const long *, hipStream_t);
template int launch_btd_inv_factor_single<float>(int, const int *, int, const double *, const long *, float *,
                                                 const long *, hipStream_t);

template <typename T>
int launch_btd_inv_factor_small(int nsys, const int *nblocks, int bs, const double *values, const long *voff, T *dinv,
                                const long *doff, hipStream_t st) {
  small_fn<T>(bs, std::make_integer_sequence<int, kSmallFactor>{})(nsys, nblocks, values, voff, dinv, doff, st);
  return hipGetLastError() == hipSuccess ? GF_OK : fail(GF_ERR_HIP, "btd inverse factor launch failed");
}

template int launch_btd_inv_factor_small<double>(int, const int *, int, const double *, const long *, double *,
                                                 const long *, hipStream_t);
template int launch_btd_inv_factor_small<float>(int, const int *, int, const double *, const long *, float *,
                                                const long *, hipStream_t);

}  // namespace gfa
