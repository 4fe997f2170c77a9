// Batched block-tridiagonal factor/solve with diagonal off-diagonal blocks (griffon's BTDDOD format), with
// FP64 factors (in place, as the reference) or FP32 factors in separate arrays (the mixed-precision path of
// the flamelet solvers: FP32 block LU, FP64 right-hand sides, solutions and residuals).
//
// Algorithm restated from btddod_matrix_kernels.cpp:19-119 (block Thomas):
//   D_0 = LU(D_0);  for i >= 1:  L_i = diag(sub_{i-1}) D_{i-1}^{-1},  D_i -= L_i diag(sup_{i-1}),  D_i = LU(D_i)
//   forward  y_0 = b_0,  y_i = b_i - L_i y_{i-1};   backward  x_{n-1} = D^{-1} y,  x_i = D_i^{-1}(y_i - sup_i * x_{i+1})
// with LAPACK dgetrf/dgetrs semantics for each dense block (partial pivoting, first maximum, 1-based pivots,
// factors stored in place in the values array, column-major blocks).
//
// Factorization: one workgroup per system, the factored diagonal block and the L block live in LDS
// (2 x bs^2 values); right-looking LU with a wave-reduced pivot search; D^{-1} by column-parallel
// forward/back substitution on the identity. Solve: one wave per system, lane = row, each block staged in LDS
// by one coalesced load, register-resident vectors, shuffles broadcast the pivot/substitution values.
//
// The batched flamelet solver uses a throughput form of the same recurrence (btd_inv_*): each chain is
// eliminated from both ends at once (twisted factorisation, halving the serial chain), every Schur-updated
// diagonal block is inverted by blocked Gauss-Jordan elimination with partial pivoting on the matrix cores (gf_twist.hip)
// and stored as its inverse, so no L blocks are stored and both sweeps of a solve are matrix-vector products.
#include "gf_internal.h"
#include "../../include/griffon_amd.h"

#include <utility>
#include "gf_wave.h"


namespace gfa {

namespace {

using wave::lane_value;

constexpr int BW = 64;
constexpr int BT_THREADS = 256;

// LU with partial pivoting of a bs x bs column-major block in LDS (LAPACK dgetf2 order of operations).
template <typename T>
__device__ void lds_lu(T *A, int bs, int *piv_lds, int *gpiv) {
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  __shared__ int s_p;
  for (int j = 0; j < bs; ++j) {
    if (wave == 0) {
      double v = -1.0;
      int idx = bs;
      if (lane >= j && lane < bs) { v = fabs((double)A[j * bs + lane]); idx = lane; }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double ov = __shfl_xor(v, o, 64);
        const int oi = __shfl_xor(idx, o, 64);
        if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
      }
      if (idx >= bs) idx = j;  // no comparable pivot candidate (NaN column): keep the diagonal
      if (lane == 0) {
        s_p = idx;
        piv_lds[j] = idx + 1;
        if (gpiv) gpiv[j] = idx + 1;
      }
    }
    __syncthreads();
    const int p = s_p;
    if (p != j)
      for (int c = t; c < bs; c += BT_THREADS) {
        const T a0 = A[c * bs + j];
        A[c * bs + j] = A[c * bs + p];
        A[c * bs + p] = a0;
      }
    __syncthreads();
    const T d = A[j * bs + j];
    if (d != T(0)) {
      const T id = T(1) / d;
      for (int k = j + 1 + t; k < bs; k += BT_THREADS) A[j * bs + k] *= id;
    }
    __syncthreads();
    const int m = bs - j - 1;
    for (int e = t; e < m * m; e += BT_THREADS) {
      const int c = j + 1 + e / m, k = j + 1 + e % m;
      A[c * bs + k] -= A[j * bs + k] * A[c * bs + j];
    }
    __syncthreads();
  }
}

// X <- A^{-1} X for bs right-hand sides, A an LU factorization with pivots in LDS (LAPACK dgetrs, 'N').
template <typename T>
__device__ void lds_lu_solve_multi(const T *A, const int *piv, int bs, T *X) {
  const int t = threadIdx.x;
  for (int j = 0; j < bs; ++j) {  // row interchanges, applied in order
    const int p = piv[j] - 1;
    if (p != j)
      for (int c = t; c < bs; c += BT_THREADS) {
        const T a0 = X[c * bs + j];
        X[c * bs + j] = X[c * bs + p];
        X[c * bs + p] = a0;
      }
    __syncthreads();
  }
  for (int j = 0; j < bs; ++j) {  // unit lower triangular
    const int m = bs - j - 1;
    for (int e = t; e < m * bs; e += BT_THREADS) {
      const int c = e / m, k = j + 1 + e % m;
      X[c * bs + k] -= A[j * bs + k] * X[c * bs + j];
    }
    __syncthreads();
  }
  for (int j = bs - 1; j >= 0; --j) {  // upper triangular
    for (int c = t; c < bs; c += BT_THREADS) X[c * bs + j] /= A[j * bs + j];
    __syncthreads();
    for (int e = t; e < j * bs; e += BT_THREADS) {
      const int c = e / j, k = e % j;
      X[c * bs + k] -= A[j * bs + k] * X[c * bs + j];
    }
    __syncthreads();
  }
}

// Factors of system sys: D blocks to dout + doff[sys] (for FP64 the values array itself, in place), L blocks to
// lout + loff[sys]; the input blocks and off-diagonals are the FP64 values array.
template <typename T>
__global__ void __launch_bounds__(BT_THREADS) btd_factor_kernel(const int *nblocks, int bs, double *values,
                                                               const long *voff, T *dout, const long *doff, T *lout,
                                                               const long *loff, int *piv, const long *poff) {
  extern __shared__ double sm_raw[];
  T *sm = reinterpret_cast<T *>(sm_raw);
  const int sys = blockIdx.x;
  const int nb = nblocks[sys];
  const int nb2 = bs * bs;
  const double *V = values + voff[sys];
  T *Dg = dout + doff[sys];
  T *L = lout + loff[sys];
  int *P = piv + poff[sys];
  const double *sub = V + (long)nb * nb2;
  const double *sup = sub + (long)(nb - 1) * bs;
  T *D = sm, *Lb = sm + nb2;                // factored diagonal block, L block
  int *pv = reinterpret_cast<int *>(sm + 2 * nb2);
  const int t = threadIdx.x;

  for (int e = t; e < nb2; e += BT_THREADS) D[e] = (T)V[e];
  __syncthreads();
  lds_lu(D, bs, pv, P);
  for (int e = t; e < nb2; e += BT_THREADS) Dg[e] = D[e];
  for (int i = 1; i < nb; ++i) {
    const long o1 = (long)i * nb2;
    for (int e = t; e < nb2; e += BT_THREADS) Lb[e] = ((e % bs) == (e / bs)) ? T(1) : T(0);
    __syncthreads();
    lds_lu_solve_multi(D, pv, bs, Lb);  // Lb = D_{i-1}^{-1}
    const int b1 = (i - 1) * bs;
    for (int e = t; e < nb2; e += BT_THREADS) {
      const int j = e / bs, k = e % bs;
      const T l = Lb[e] * (T)sub[b1 + k];
      L[o1 + e] = l;
      D[e] = (T)(V[o1 + e] + (-sup[b1 + j]) * (double)l);
    }
    __syncthreads();
    lds_lu(D, bs, pv, P + i * bs);
    for (int e = t; e < nb2; e += BT_THREADS) Dg[o1 + e] = D[e];
  }
}

// One wave per system, lane = row; each block is staged in LDS with one coalesced load before it is used.
// FP64 arithmetic; FP32 factors are widened on load.
template <typename T>
__global__ void __launch_bounds__(BW) btd_solve_kernel(int nsys, const int *nblocks, int bs, const double *values,
                                                      const long *voff, const T *dfac, const long *doff,
                                                      const T *lval, const long *loff, const int *piv,
                                                      const long *poff, const double *rhs, double *x,
                                                      const long *xoff) {
  extern __shared__ double sm_raw[];
  T *Bk = reinterpret_cast<T *>(sm_raw);
  int *pvs = reinterpret_cast<int *>(Bk + bs * bs);
  const int sys = blockIdx.x;
  if (sys >= nsys) return;
  const int lane = threadIdx.x;
  const int nb = nblocks[sys];
  const int nb2 = bs * bs;
  const double *V = values + voff[sys];
  const T *DF = dfac + doff[sys];
  const T *L = lval + loff[sys];
  const int *P = piv + poff[sys];
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  const double *sup = V + (long)nb * nb2 + (long)(nb - 1) * bs;
  const bool act = lane < bs;

  // forward: y_i = b_i - L_i y_{i-1}; y kept in X
  double y = act ? b[lane] : 0.;
  if (act) X[lane] = y;
  for (int i = 1; i < nb; ++i) {
    const T *Li = L + (long)i * nb2;
    for (int e = lane; e < nb2; e += BW) Bk[e] = Li[e];
    __syncthreads();
    double yi = act ? b[(long)i * bs + lane] : 0.;
    for (int c = 0; c < bs; ++c) {
      const double yc = __shfl(y, c, 64);
      if (act) yi = yi + (double)Bk[c * bs + lane] * (-1. * yc);
    }
    y = yi;
    if (act) X[(long)i * bs + lane] = y;
    __syncthreads();
  }
  // backward
  double xn = 0.;
  for (int i = nb - 1; i >= 0; --i) {
    const T *Dg = DF + (long)i * nb2;
    for (int e = lane; e < nb2; e += BW) Bk[e] = Dg[e];
    if (act) pvs[lane] = P[i * bs + lane];
    __syncthreads();
    double r = act ? X[(long)i * bs + lane] : 0.;
    if (i < nb - 1 && act) r = r - sup[(long)i * bs + lane] * xn;
    for (int j = 0; j < bs; ++j) {  // row interchanges
      const int p = pvs[j] - 1;
      if (p != j) {
        const double vj = __shfl(r, j, 64), vp = __shfl(r, p, 64);
        if (lane == j) r = vp;
        else if (lane == p) r = vj;
      }
    }
    for (int j = 0; j < bs; ++j) {  // unit lower
      const double rj = __shfl(r, j, 64);
      if (act && lane > j) r -= (double)Bk[j * bs + lane] * rj;
    }
    for (int j = bs - 1; j >= 0; --j) {  // upper
      if (lane == j) r /= (double)Bk[j * bs + j];
      const double rj = __shfl(r, j, 64);
      if (act && lane < j) r -= (double)Bk[j * bs + lane] * rj;
    }
    xn = r;
    if (act) X[(long)i * bs + lane] = r;
    __syncthreads();
  }
}

// ---------------- block Thomas with explicit diagonal-block inverses ----------------

// Solve with the twisted factors, one workgroup of eight waves per system: waves 0 .. 3 the top chain, 4 .. 7 the bottom one,
//   top:     y_0 = b_0,  y_i = b_i - sub_{i-1} (D_{i-1}^{-1} y_{i-1}),  i < m
//   bottom:  y_{n-1} = b_{n-1},  y_i = b_i - sup_i (E_{i+1}^{-1} y_{i+1}),  i > m
//   middle:  x_m = C_m^{-1} (b_m - sub_{m-1} (D_{m-1}^{-1} y_{m-1}) - sup_m (E_{m+1}^{-1} y_{m+1}))
//   top:     x_i = D_i^{-1} (y_i - sup_i x_{i+1}),  i = m-1 .. 0;   bottom:  x_i = E_i^{-1} (y_i - sub_{i-1} x_{i-1}),  i > m
// A chain is a series of 2 len + 1 products with its blocks, inwards, the middle one, outwards again. Each is shared by four
// waves (lane = row): wave q multiplies the columns 4 k + q of the block, the vector's entries broadcast through scalar
// registers, and the sum of the four partial sums, exchanged through LDS behind one barrier, is formed by every wave, which
// so holds the next vector. With few chains the steps between two products bound it (the exchange, the broadcasts, about
// 1,000 cycles at 53), with many the two reads of the inverses: 1,024 chains move 7.1 GB in 1.8 ms. Loads are issued two
// products ahead (FP32 three): more is no faster, and takes the registers that let two workgroups share a
// compute unit, which batches of single blocks need. Before, two waves per system did a whole product each, in
// batches of sixteen column loads that were waited for one after the other. Measured before and after (53x53, us):
//   systems                     FP64             FP32
//   one chain of 126 blocks       277 ->   150     268 -> 108
//   48 / 192 chains of 62..254    788 / 1,079 -> 311 / 438     722 / 925 -> 231 / 267
//   512 / 1,024 chains          1,293 / 1,931 -> 940 / 1,811   1,073 / 1,301 -> 501 / 975
//   4,000 blocks                   19 ->    19      14 ->  13
// The partial sums are those of columns c mod 4 in ascending order, the columns beyond the last group of four in the
// first one, and the sum is (m0 + m1) + (m2 + m3), as before: solutions are bitwise the same.
template <typename T>
constexpr int kAhead = sizeof(T) == 8 ? 2 : 3;

template <typename T, int N>
__global__ void __launch_bounds__(512) btd_twist_solve_kernel(const int *nblocks, const double *values, const long *voff,
                                                              const T *dinv, const long *doff, const double *rhs,
                                                              double *x, const long *xoff) {
  constexpr int K = N / 4, E = N % 4;
  __shared__ double part[2][2][4][64];  // [parity of the product][chain][wave][row]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chain = wave >> 2, q = wave & 3;
  const bool top = chain == 0;
  const int sys = blockIdx.x;
  const int nb = __builtin_amdgcn_readfirstlane(nblocks[sys]);
  if (!top && nb == 1) return;  // no bottom chain
  const bool act = lane < N;
  const int rl = act ? lane : 0;
  const int m = (nb - 1) / 2;
  const T *DI = dinv + doff[sys] + rl;
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  const double *sub = values + voff[sys] + (long)nb * (N * N);
  const double *sup = sub + (long)(nb - 1) * N;

  // What a product needs: the block's columns of this wave (e: those beyond the groups of four, for wave 0), and the two
  // vectors a, c that form the next product's vector a - c * (this product). y_i is kept in X. Every product loads the same
  // number of words without a branch (clamped where there is nothing to load), so that a wait counts the loads it
  // needs and leaves the later products' in flight.
  struct Ahead {
    T d[K > 0 ? K : 1], e[E > 0 ? E : 1];
    double a, c;
  };
  auto columns = [&](Ahead &B, int blk) {
    const T *D = DI + (long)blk * (N * N);
#pragma unroll
    for (int k = 0; k < E; ++k) B.e[k] = D[(4 * K + k) * N];
    D += q * N;
#pragma unroll
    for (int k = 0; k < K; ++k) B.d[k] = D[4 * k * N];
  };
  double v;
  auto multiply = [&](const Ahead &B, double *out) {
    double acc = 0.;
#pragma unroll
    for (int k = 0; k < K; ++k) acc = fma((double)B.d[k], lane_value(v, 4 * k + q), acc);
    if (E > 0 && q == 0) {
#pragma unroll
      for (int k = 0; k < E; ++k) acc = fma((double)B.e[k], lane_value(v, 4 * K + k), acc);
    }
    out[lane] = acc;
  };
  auto sum = [&](const double (*p)[64]) { return (p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane]); };
  if (nb == 1) {
    Ahead B;
    v = b[rl];
    columns(B, 0);
    multiply(B, part[0][0][q]);
    __syncthreads();
    if (q == 0 && act) X[lane] = sum(part[0][0]);
    return;
  }

  // Both chains run L products inwards, the middle one and L outwards; a top chain that is one shorter waits for one at
  // either end (off). Product s of a chain is with the block of its place len - |len - s|, the next one's coupling is that
  // between the two blocks, row min of the two of sub or sup.
  const int L = nb - 1 - m;
  const int len = top ? m : L, off = L - len;
  const int first = top ? 0 : nb - 1, dir = top ? 1 : -1;
  auto block = [&](int s) { return first + dir * max(len - abs(len - s), 0); };
  auto at = [&](int i) { return (unsigned)(i * N + rl); };
  const double bm = b[at(m)], ct = m > 0 ? sub[at(m - 1)] : 0., cb = sup[at(m)];
  double last = 0.;
  v = b[at(block(0))];
  if (len > 0 && act) X[at(block(0))] = v;  // every wave writes, and later reads, its own
  auto operands = [&](Ahead &B, int s) {
    const int i = block(s), j = block(s + 1);
    columns(B, i);
    B.c = (top == (s < len) ? sub : sup)[at(min(min(i, j), nb - 2))];
  };
  auto addend = [&](Ahead &B, int s) { B.a = (s < len ? b : X)[at(block(s + 1))]; };
  Ahead buf[kAhead<T>];
#pragma unroll
  for (int k = 0; k < kAhead<T>; ++k) {
    operands(buf[k], max(k - off, 0));
    addend(buf[k], max(k - off, 0));
  }

  const bool out = act && q == 0;
  auto product = [&](Ahead &B, int g) {
    const int s = g - off;
    multiply(B, part[g & 1][chain][q]);
    // Loads that do not depend on this product go before the barrier. The addend has to be here by then: x may be rhs, and
    // behind the barrier other waves write what it was read from.
    const double a = s == len ? last : B.a, c = B.c;
    asm volatile("" ::"v"(B.a));
    operands(B, s + kAhead<T>);
    __syncthreads();
    if (g == L - 1) {
#pragma clang fp contract(off)
      const double tt = m > 0 ? ct * sum(part[g & 1][0]) : 0., tb = cb * sum(part[g & 1][1]);
      last = v;
      v = bm - tt - tb;
    } else if ((unsigned)s <= (unsigned)(2 * len)) {
      const bool in = s < len;
      const double mv = sum(part[g & 1][chain]);
      v = fma(-c, mv, a);
      // y of the next block or x of this one (both chains write x_m, the same)
      if (in ? act : out) X[at(block(in ? s + 1 : s))] = in ? v : mv;
    }
    addend(B, s + kAhead<T>);
  };
  for (int g = 0; g <= 2 * L; g += kAhead<T>) {
#pragma unroll
    for (int k = 0; k < kAhead<T>; ++k) {
      if (g + k > 2 * L) break;
      product(buf[k], g + k);
    }
  }
}

template <typename T>
using InvSolve = void (*)(const int *, const double *, const long *, const T *, const long *, const double *, double *,
                          const long *);
template <typename T, int... I>
InvSolve<T> inv_solve_kernel(int bs, std::integer_sequence<int, I...>) {
  constexpr InvSolve<T> tab[] = {&btd_twist_solve_kernel<T, I + 1>...};
  return tab[bs - 1];
}

}  // namespace

int launch_btd_factor(int nsys, const int *nblocks, int bs, double *values, const long *voff, double *l_values,
                      const long *loff, int *pivots, const long *poff, hipStream_t st) {
  return launch_btd_factor_t<double>(nsys, nblocks, bs, values, voff, values, voff, l_values, loff, pivots, poff, st);
}

int launch_btd_solve(int nsys, const int *nblocks, int bs, const double *values, const long *voff,
                     const double *l_values, const long *loff, const int *pivots, const long *poff, const double *rhs,
                     double *x, const long *xoff, hipStream_t st) {
  return launch_btd_solve_t<double>(nsys, nblocks, bs, values, voff, values, voff, l_values, loff, pivots, poff, rhs,
                                    x, xoff, st);
}

template <typename T>
int launch_btd_factor_t(int nsys, const int *nblocks, int bs, double *values, const long *voff, T *dfac,
                        const long *doff, T *l_values, const long *loff, int *pivots, const long *poff,
                        hipStream_t st) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  const size_t lds = sizeof(T) * 2 * bs * bs + sizeof(int) * 64 + 16;
  auto kern = btd_factor_kernel<T>;
  if (lds > 65536)
    if (hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return fail(GF_ERR_UNSUPPORTED, "block too large for LDS");
  hipLaunchKernelGGL(kern, dim3(nsys), dim3(BT_THREADS), lds, st, nblocks, bs, values, voff, dfac, doff, l_values,
                     loff, pivots, poff);
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "btd factor launch failed");
  return GF_OK;
}

template <typename T>
int launch_btd_solve_t(int nsys, const int *nblocks, int bs, const double *values, const long *voff, const T *dfac,
                       const long *doff, const T *l_values, const long *loff, const int *pivots, const long *poff,
                       const double *rhs, double *x, const long *xoff, hipStream_t st) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  const size_t lds = sizeof(T) * bs * bs + sizeof(int) * 64 + 16;
  hipLaunchKernelGGL(btd_solve_kernel<T>, dim3(nsys), dim3(BW), lds, st, nsys, nblocks, bs, values, voff, dfac, doff,
                     l_values, loff, pivots, poff, rhs, x, xoff);
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "btd solve launch failed");
  return GF_OK;
}

template <typename T>
int launch_btd_inv_solve(int nsys, const int *nblocks, int bs, const double *values, const long *voff,
                         const T *dinv, const long *doff, const double *rhs, double *x, const long *xoff,
                         hipStream_t st) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  const auto kern = inv_solve_kernel<T>(bs, std::make_integer_sequence<int, 64>{});
  hipLaunchKernelGGL(kern, dim3(nsys), dim3(512), 0, st, nblocks, values, voff, dinv, doff, rhs, x, xoff);
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "btd inverse solve launch failed");
  return GF_OK;
}

template int launch_btd_inv_solve<double>(int, const int *, int, const double *, const long *, const double *,
                                          const long *, const double *, double *, const long *, hipStream_t);
template int launch_btd_inv_solve<float>(int, const int *, int, const double *, const long *, const float *,
                                         const long *, const double *, double *, const long *, hipStream_t);
template int launch_btd_factor_t<float>(int, const int *, int, double *, const long *, float *, const long *, float *,
                                        const long *, int *, const long *, hipStream_t);
template int launch_btd_solve_t<float>(int, const int *, int, const double *, const long *, const float *,
                                       const long *, const float *, const long *, const int *, const long *,
                                       const double *, double *, const long *, hipStream_t);

}  // namespace gfa
