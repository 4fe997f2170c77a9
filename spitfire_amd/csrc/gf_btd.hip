// Batched block-tridiagonal factor/solve with diagonal off-diagonal blocks (griffon's BTDDOD format), in two forms.
//
// As the reference has it, restated from btddod_matrix_kernels.cpp:19-119 (block Thomas):
//   D_0 = LU(D_0);  for i >= 1:  L_i = diag(sub_{i-1}) D_{i-1}^{-1},  D_i -= L_i diag(sup_{i-1}),  D_i = LU(D_i)
//   forward  y_0 = b_0,  y_i = b_i - L_i y_{i-1};   backward  x_{n-1} = D^{-1} y,  x_i = D_i^{-1}(y_i - sup_i * x_{i+1})
// with LAPACK dgetrf/dgetrs semantics for each dense block (partial pivoting, first maximum, 1-based pivots,
// factors stored in place in the values array, column-major blocks, FP64). btd_factor_kernel: one workgroup of eight waves per
// system, a block and its inverse in registers, lane = row. btd_solve_kernel: a wave that runs the chain and one that prepares the
// next block. Blocks that are singular or hold infinities or NaN go through a plain form of the same operations.
//
// The batched flamelet and reactor solvers use a throughput form of the same recurrence: each chain is
// eliminated from both ends at once (twisted factorisation, halving the serial chain), every Schur-updated
// diagonal block is inverted by Gauss-Jordan elimination with partial pivoting (gf_twist.hip on the matrix cores,
// gf_twist_small.hip one wave per chain) and stored as its inverse, in FP64 or FP32, so no L blocks are stored and both sweeps of a
// solve are matrix-vector products. Their solves: btd_twist_solve_kernel, four waves per chain; btd_wave_solve_kernel, one;
// btd_chain_solve_kernel and btd_middle_solve_kernel, a compute unit per chain. All three give bitwise the same.
#include "gf_btd_index.h"
#include "gf_internal.h"
#include "gf_wave.h"
#include "../../include/griffon_amd.h"

#include <type_traits>
#include <utility>

namespace gfa {

namespace {

using wave::lane_value;

// ---------------- block Thomas with LAPACK's factors ----------------

constexpr int kLuWaves = 8;

// Whether the magnitude of f is outside 2^-range .. 2^range (zero, infinities and NaN are)
template <int range>
__device__ __forceinline__ bool extreme(double f) {
  const unsigned e = (unsigned)__double2hiint(f) & 0x7fffffffu;
  return e - ((unsigned)(1023 - range) << 20) > ((unsigned)(2 * range) << 20);
}

// x / u with id the rounded 1 / u: the rounded quotient, unless out of range
__device__ __forceinline__ double quotient(double x, double u, double id) {
  const double q = x * id;
  return fma(fma(-u, q, x), id, q);
}

// A block in LDS, [column][row], factored by a workgroup step by step as LAPACK's dgetf2 does: nothing but the rows and columns
// beyond a pivot is touched, so an infinity goes no further than there, and a pivot of zero leaves its column as it is.
__device__ void plain_lu(double (*A)[64], int *piv, int bs, int t) {
  constexpr int NT = 64 * kLuWaves;
  const int lane = t & 63;
#pragma unroll 1
  for (int j = 0; j < bs; ++j) {
    if (t < 64) {
      double v = -1.;
      int idx = bs;
      const double q = lane < bs ? fabs(A[j][lane]) : -1.;
      if (lane >= j && q >= 0.) {
        v = q;
        idx = lane;
      }
#pragma unroll 1
      for (int o = 32; o > 0; o >>= 1) {
        const double ov = __shfl_xor(v, o, 64);
        const int oi = __shfl_xor(idx, o, 64);
        if (ov > v || (ov == v && oi < idx)) {
          v = ov;
          idx = oi;
        }
      }
      if (lane == 0) piv[j] = idx >= bs ? j : idx;  // (NaN is not chosen; of nothing else, the diagonal is)
    }
    __syncthreads();
    const int p = piv[j];
    if (p != j)
#pragma unroll 1
      for (int c = t; c < bs; c += NT) {
        const double q = A[c][j];
        A[c][j] = A[c][p];
        A[c][p] = q;
      }
    __syncthreads();
    const double d = A[j][j];
    if (d != 0.) {
      const double id = 1. / d;
#pragma unroll 1
      for (int k = j + 1 + t; k < bs; k += NT) A[j][k] *= id;
    }
    __syncthreads();
    const int m = bs - j - 1;
#pragma unroll 1
    for (int e = t; e < m * m; e += NT) {
      const int c = j + 1 + e / m, k = j + 1 + e % m;
      A[c][k] = fma(-A[j][k], A[c][j], A[c][k]);
    }
    __syncthreads();
  }
}

// X = A^{-1}, column-major in memory, from these factors, with a division for every entry
__device__ void plain_inverse(const double (*A)[64], const int *piv, int bs, int t, double *X) {
  constexpr int NT = 64 * kLuWaves;
#pragma unroll 1
  for (int e = t; e < bs * bs; e += NT) X[e] = e / bs == e % bs ? 1. : 0.;
  __syncthreads();
#pragma unroll 1
  for (int j = 0; j < bs; ++j) {
    const int p = piv[j];
    if (p != j)
#pragma unroll 1
      for (int c = t; c < bs; c += NT) {
        const double q = X[c * bs + j];
        X[c * bs + j] = X[c * bs + p];
        X[c * bs + p] = q;
      }
    __syncthreads();
  }
#pragma unroll 1
  for (int j = 0; j < bs; ++j) {
    const int m = bs - j - 1;
#pragma unroll 1
    for (int e = t; e < m * bs; e += NT) {
      const int c = e / m, k = j + 1 + e % m;
      X[c * bs + k] = fma(-A[j][k], X[c * bs + j], X[c * bs + k]);
    }
    __syncthreads();
  }
#pragma unroll 1
  for (int j = bs - 1; j >= 0; --j) {
#pragma unroll 1
    for (int c = t; c < bs; c += NT) X[c * bs + j] /= A[j][j];
    __syncthreads();
#pragma unroll 1
    for (int e = t; e < j * bs; e += NT) {
      const int c = e / j, k = e % j;
      X[c * bs + k] = fma(-A[j][k], X[c * bs + j], X[c * bs + k]);
    }
    __syncthreads();
  }
}

// Factors of one system per workgroup: LU with partial pivoting of every diagonal block (LAPACK dgetf2's order of operations,
// interchanges as dgetrf returns them), in place in values; the L blocks sub_{i-1} D_{i-1}^{-1}, to l; and the
// pivots. A block is in registers, lane = row, wave w of eight holding columns w, 8 + w, .. (C of them) of it (a) and of what
// becomes its inverse (x, the identity at first, eliminated along with it). Rows stay in their lanes: `cur` is the
// position that LAPACK's interchanges have given a row, and where they end is the next block's order of rows.
// What bounds it is the chain of pivots, blocks after blocks: the wave with column j searches it, publishes the
// multipliers in LDS, and one barrier later all waves update their columns. The next column's owner does that column first
// and searches it before its other ones. The back substitution of the inverse needs no barrier: every wave has the
// columns of U that it wants from LDS, divided by their pivots, so the inverse's rows are divided once at the end instead of
// every entry in its turn. (Errors of L blocks against long double, 60 systems of three diagonally dominant blocks: of 12 / 24 /
// 37 / 53 unknowns 0.99 / 0.99 / 1.00 / 1.00 of those with a division for every entry; with products with rounded
// reciprocals 1.06 / 1.00 / 1.01 / 1.01.) The next block's values are loaded while a block is factored. Before, a block in
// LDS took four barriers a pivot, two more and a division for the substitutions. About 1,000 cycles a pivot now: the two LDS
// words, the update, search and reciprocal of one column and the way back, one after the other. Measured before and after
// (us): one system of 60 blocks of 53 10,140 -> 2,290, 24 of 30..60 9,620 -> 2,180, 1,500 of 2..11 4,070 -> 1,400; 24 of 24x24
// blocks 2,600 -> 790, of 10x10 920 -> 330. Putting a searching wave's other columns off behind the next barrier gained nothing.
// Finished rows are updated along with the others, with a multiplier of zero, and U is scaled by reciprocals: where a block has
// infinities, NaN or a pivot outside 2^-300 .. 2^300 (a singular one among them), that is not what LAPACK's order of operations
// gives. Such a block is found when it is done, before it is stored; from there on the system is factored in LDS by plain_lu and
// plain_inverse (behind the loop of the others, so that nothing of it takes their registers).
template <int C>
__global__ void __launch_bounds__(64 * kLuWaves) __attribute__((amdgpu_waves_per_eu(C == 7 ? 6 : 1)))
btd_factor_kernel(const int *nblocks, int bs, double *values, const long *voff, double *lout, const long *loff, int *piv,
                  const long *poff) {
  __shared__ double A[8 * C][64], gb[2][64];  // columns of U for the substitution, [column][lane]; what a step publishes, by
  __shared__ double diagonal[64];             // parity of the step; of U, by lane
  __shared__ int pb[2];
  __shared__ int odd[2], plain_piv[64];       // by parity of the block: whether it has to be factored plainly
  const int sys = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = nblocks[sys];
  const long nb2 = (long)bs * bs;
  double *V = values + voff[sys];
  double *L = lout + loff[sys];
  int *P = piv + poff[sys];
  const double *sub = V + nb * nb2;
  const double *sup = sub + (long)(nb - 1) * bs;
  const bool act = lane < bs;
  const int rl = act ? lane : 0;
  int cur = act ? lane : -1;
  double a[C], x[C], v[C], idl = 0.;
  int pivot = 0, row_of = 0;  // of step = lane: LAPACK's interchange, and the lane of the row
  auto load = [&](double(&to)[C], const double *from) {
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const double t = from[min(8 * k + w, bs - 1) * bs + rl];
      to[k] = act && 8 * k + w < bs ? t : 0.;
    }
  };
  // pivot of column j = f: the multipliers (the reciprocal for the pivot row) and its lane to LDS; returns the column as the
  // factors have it
  auto publish = [&](double f, int j) {
    const bool cand = cur >= j;
    const unsigned key = cand & (f == f) ? (unsigned)__double2hiint(f) & 0x7fffffffu : 0u;
    unsigned most = key;
    auto rc = wave::recip_of(f);
    rc.template step<0>(); most = wave::max_step<0>(most);
    rc.template step<1>(); most = wave::max_step<1>(most);
    rc.template step<2>(); most = wave::max_step<2>(most);
    rc.template step<3>(); most = wave::max_step<3>(most);
    rc.template step<4>(); most = wave::max_step<4>(most);
    rc.template step<5>(); most = wave::max_step<5>(most);
    rc.template step<6>();
    const unsigned top = (unsigned)__builtin_amdgcn_readlane((int)most, 63);
    unsigned long long hit = __ballot(key == top);
    if (hit & (hit - 1)) {  // rare: the low words decide, then the position
      const bool in = cand & (key == top);
      const unsigned lo = in & (f == f) ? (unsigned)__double2loint(f) : 0u;
      const unsigned big = wave::dpp_wave_max_u32(lo);
      const unsigned at = in & (lo == big) ? 64u - (unsigned)cur : 0u;
      const unsigned low = wave::dpp_wave_max_u32(at);
      hit = __ballot(in & (at == low));
    }
    const int p = __builtin_ctzll(hit);
    const double id = lane_value(rc.r, p);
    const double l = f * (top != 0u || lane_value(f, p) != 0. ? id : 1.);
    const bool below = cand & (lane != p);
    gb[j & 1][lane] = lane == p ? id : below ? l : 0.;
    pb[j & 1] = p;
    return below ? l : f;
  };
  if (threadIdx.x == 0) odd[0] = odd[1] = 0;
  int plain = nb;
  load(a, V);
  for (int i = 0; i < nb; ++i) {
    asm volatile("" : "+s"(bs));  // opaque: addresses and conditions are formed anew rather than kept (and spilled)
    double subv = 0., supv = 0.;
    if (i + 1 < nb) {
      load(v, V + (i + 1) * nb2);
      subv = sub[(long)i * bs + rl];
      supv = sup[(long)i * bs + rl];
    }
#pragma unroll
    for (int k = 0; k < C; ++k) x[k] = cur == 8 * k + w ? 1. : 0.;
    if (w == 0) a[0] = publish(a[0], 0);
    double l = 0.;
    int p = 0;
    auto begin = [&](int j) {
      __syncthreads();
      p = __builtin_amdgcn_readfirstlane(pb[j & 1]);
      const double g = gb[j & 1][lane];
      l = lane == p ? 0. : g;
      const int at = __builtin_amdgcn_readlane(cur, p);
      idl = lane == p ? g : idl;
      pivot = lane == j ? at + 1 : pivot;
      row_of = lane == j ? p : row_of;
      cur = lane == p ? j : cur == j ? at : cur;
    };
    auto update = [&](double &y) { y = fma(-l, lane_value(y, p), y); };
    auto eliminate = [&](auto inverse) {
      auto rest = [&](int after) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
          if (c > after) update(a[c]);
          if (inverse) update(x[c]);
        }
      };
#pragma unroll
      for (int k = 0; k < C; ++k) {
#pragma unroll 1
        for (int q = 0; q < 7; ++q) {
          const int j = 8 * k + q;
          if (j >= bs) break;
          begin(j);
          if (w > q) update(a[k]);
          if (w == q + 1 && j + 1 < bs) a[k] = publish(a[k], j + 1);
          rest(k);
        }
        const int j = 8 * k + 7;
        if (j < bs) {
          begin(j);
          constexpr int last = C - 1;
          if (k < last) update(a[k < last ? k + 1 : last]);
          if (w == 0 && j + 1 < bs) a[k < last ? k + 1 : last] = publish(a[k < last ? k + 1 : last], j + 1);
          rest(k + 1);
        }
      }
    };
    // The last block's inverse is not needed: single blocks 10 to 30% faster, chains even. (With seven columns a wave two versions of
    // the loop take more than the 80 registers of three workgroups per compute unit: 1,500 chains of 2..11 of 53 1,410 -> 1,510 us.)
    if (C == 7 || i + 1 < nb) eliminate(std::true_type{});
    else eliminate(std::false_type{});
    double za = 0., zx = 0., own = 0.;  // NaN where an entry is not finite; the diagonal of U if this wave has it
#pragma unroll
    for (int k = 0; k < C; ++k) {
      za = fma(a[k], 0., za);
      zx = fma(x[k], 0., zx);
      // (the reciprocal is its row's; rows at and below the diagonal have no part in the substitution)
      const int r = __builtin_amdgcn_readlane(row_of, 8 * k + w);
      const double q = quotient(a[k], lane_value(a[k], r), lane_value(idl, r));
      A[8 * k + w][lane] = cur < 8 * k + w ? q : 0.;
      own = cur == 8 * k + w ? a[k] : own;
    }
    if (act && (cur & 7) == w) diagonal[lane] = own;
    if (__any((act && extreme<300>(idl)) || za + zx != 0.)) odd[i & 1] = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(odd[i & 1])) {
      plain = i;
      break;
    }
    if (threadIdx.x == 0) odd[(i + 1) & 1] = 0;  // read before this block, set again behind the next one's barriers
#pragma unroll
    for (int k = 0; k < C; ++k)
      if (act && 8 * k + w < bs) V[i * nb2 + (8 * k + w) * bs + cur] = a[k];
    if (w == 0 && act) P[(long)i * bs + lane] = pivot;
    if (i + 1 == nb) break;
#pragma unroll 4
    for (int j = bs - 1; j >= 0; --j) {
      p = __builtin_amdgcn_readlane(row_of, j);
      l = A[j][lane];
#pragma unroll
      for (int c = 0; c < C; ++c) update(x[c]);
    }
    const double subr = __shfl(subv, cur, 64), u = diagonal[lane];
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const int c = 8 * k + w;
      const double lx = quotient(x[k], u, idl) * subr;
      if (act && c < bs) L[(i + 1) * nb2 + c * bs + cur] = lx;
      const double up = lane_value(supv, min(c, 63));
      a[k] = act && c < bs ? fma(-up, lx, __shfl(v[k], cur, 64)) : 0.;
    }
  }
  // that block and those behind it: A = V_i - L_i diag(sup_{i-1}), its factors, L_{i+1}
  const int t = threadIdx.x;
#pragma unroll 1
  for (int i = plain; i < nb; ++i) {
    double *Vi = V + i * nb2, *Li = L + i * nb2;
#pragma unroll 1
    for (int e = t; e < bs * bs; e += 64 * kLuWaves)
      A[e / bs][e % bs] = i == 0 ? Vi[e] : fma(-sup[(long)(i - 1) * bs + e / bs], Li[e], Vi[e]);
    __syncthreads();
    plain_lu(A, plain_piv, bs, t);
#pragma unroll 1
    for (int e = t; e < bs * bs; e += 64 * kLuWaves) Vi[e] = A[e / bs][e % bs];
    if (t < bs) P[(long)i * bs + t] = plain_piv[t] + 1;
    if (i + 1 == nb) break;
    plain_inverse(A, plain_piv, bs, t, Li + nb2);
#pragma unroll 1
    for (int e = t; e < bs * bs; e += 64 * kLuWaves) Li[nb2 + e] *= sub[(long)i * bs + e % bs];
    __syncthreads();
  }
}

// Solve with these factors, one workgroup per system. Wave 0 runs the chain, lane = row, with the columns of a block in
// registers (NC >= bs of them; those beyond are zero) and the next block's on their way:
//   y_i = b_i - L_i y_{i-1}, forward;  x_i = D_i^{-1} (y_i - sup_i x_{i+1}), backward: interchanges, unit lower, upper.
// What bounds it is the substitutions: a broadcast through scalar registers and a fused multiply-add for every column, for the
// upper one the division as well. Wave 1 prepares the next block meanwhile: the interchanges as one permutation, and
// the reciprocals of U's diagonal, so that a division is a product and one correction step. Before, blocks were
// staged in LDS by the wave that used them, interchanges were 53 shuffles of the vector one after the other and
// divisions whole. Measured before and after (us): 24 systems of 30..61 blocks of 53 2,460 -> 296, 2,000 of 2..4 268 -> 91;
// solutions are bitwise the same. The product with a correction is the rounded quotient where the diagonal is within
// 2^-300 .. 2^300 and the quotient within 2^-600 .. 2^600 or zero; a block with anything else (a singular one, infinities, NaN) is
// solved again with divisions, each row touched only by the columns that it has.
// One wave per SIMD is enough for a chain, but not the most: small blocks need few registers, and batches of many small systems
// want the other waves (4,000 single blocks of 10 / 20 11 / 16 us, with one wave 20 / 25, 1,500 chains of 2..11 of 10 33 and 49).
template <int NC>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1)))
btd_solve_kernel(const int *nblocks, int bs, const double *factors, const long *voff, const double *lval, const long *loff,
                 const int *piv, const long *poff, const double *rhs, double *x, const long *xoff) {
  __shared__ double diag[2][64], inverse[2][64];
  __shared__ int order[2][64];
  const int sys = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int nb = nblocks[sys];
  const long nb2 = (long)bs * bs;
  const double *D = factors + voff[sys];
  const bool act = lane < bs;
  const int rl = act ? lane : 0;
  if (threadIdx.x >= 64) {
    const int *P = piv + poff[sys];
    for (int i = nb - 1; i >= 0; --i) {
      const int p = act ? (P[(long)i * bs + lane] - 1) & 63 : lane;
      const double u = act ? D[i * nb2 + lane * bs + lane] : 1.;
      int from = lane;
      for (int j = 0; j < bs; ++j) {
        const int q = __builtin_amdgcn_readlane(p, j);
        if (q != j) {
          const int a = __builtin_amdgcn_readlane(from, j), b = __builtin_amdgcn_readlane(from, q);
          from = lane == j ? b : lane == q ? a : from;
        }
      }
      order[i & 1][lane] = from;
      diag[i & 1][lane] = u;
      inverse[i & 1][lane] = 1. / u;
      __syncthreads();  // block i is ready, and i + 1 done with
    }
    return;
  }
  const double *L = lval + loff[sys];
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  auto sup = [&](int i) { return D[btd_sup(nb, bs, i) + rl]; };
  double B[2][NC];
  auto load = [&](double(&to)[NC], const double *from) {
#pragma unroll
    for (int c = 0; c < NC; ++c) to[c] = from[min(c, bs - 1) * bs + rl];
  };
  auto column = [&](const double(&of)[NC], int c, bool in) { return in & (c < bs) ? of[c] : 0.; };

  double y = act ? b[lane] : 0.;
  if (act) X[lane] = y;
  auto forward = [&](const double(&of)[NC], int i, double bi) {
    double t = act ? bi : 0.;
#pragma unroll
    for (int c = 0; c < NC; ++c) t = fma(column(of, c, act), -lane_value(y, c), t);
    y = act ? t : 0.;  // (columns beyond the block are zero, and so are their entries: 0 times an infinity is none)
    if (act) X[(long)i * bs + lane] = y;
  };
  if (nb > 1) {
    load(B[0], L + nb2);
    double b0 = b[bs + rl], b1 = 0.;
    for (int i = 1; i < nb; i += 2) {
      const int n1 = min(i + 1, nb - 1), n2 = min(i + 2, nb - 1);
      load(B[1], L + n1 * nb2);
      b1 = b[(long)n1 * bs + rl];
      forward(B[0], i, b0);
      if (i + 1 == nb) break;
      load(B[0], L + n2 * nb2);
      b0 = b[(long)n2 * bs + rl];
      forward(B[1], i + 1, b1);
    }
  }
  double xn = 0.;
  auto backward = [&](const double(&of)[NC], int i, double yi, double s) {
    __syncthreads();
    const int from = order[i & 1][lane];
    const double u = diag[i & 1][lane], v = inverse[i & 1][lane];
    double r = i == nb - 1 ? yi : fma(-s, xn, yi);
    r = act ? r : 0.;
    r = __shfl(r, from, 64);
    const double r0 = r;
    int ln = lane;
    asm volatile("" : "+v"(ln));  // opaque: the comparisons below are not kept (and spilled) over the blocks
#pragma unroll
    for (int j = 0; j < NC; ++j) r = fma(-column(of, j, ln > j), lane_value(r, j), r);
#pragma unroll
    for (int j = NC - 1; j >= 0; --j) {
      const double q = quotient(r, u, v);
      r = ln == j ? q : r;
      r = fma(-column(of, j, ln < j), lane_value(q, j), r);
    }
    // not what divisions give, or entries that the substitutions would not have touched
    if (__any(act && (extreme<300>(u) || (r != 0. && extreme<600>(r))))) {
      const double *Di = D + i * nb2 + rl;
      r = r0;
#pragma unroll 1
      for (int j = 0; j < bs; ++j) {
        const double d = Di[j * bs], q = lane_value(r, j);
        if (act && lane > j) r = fma(-d, q, r);
      }
#pragma unroll 1
      for (int j = bs - 1; j >= 0; --j) {
        if (lane == j) r /= u;
        const double d = Di[j * bs], q = lane_value(r, j);
        if (act && lane < j) r = fma(-d, q, r);
      }
    }
    xn = r;
    if (act) X[(long)i * bs + lane] = r;
  };
  load(B[0], D + (nb - 1) * nb2);
  double y0 = y, y1 = 0., s0 = 0., s1 = 0.;
  for (int i = nb - 1; i >= 0; i -= 2) {
    const int n1 = max(i - 1, 0), n2 = max(i - 2, 0);
    load(B[1], D + n1 * nb2);
    y1 = X[(long)n1 * bs + rl];
    s1 = sup(n1);
    backward(B[0], i, y0, s0);
    if (i == 0) break;
    load(B[0], D + n2 * nb2);
    y0 = X[(long)n2 * bs + rl];
    s0 = sup(n2);
    backward(B[1], i - 1, y1, s1);
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

// One wave's share of a product with a block: what it loads (d: the columns 4 k + q, e: those beyond the groups of four, for
// wave 0; a, c: the vectors that form the next product's vector a - c * (this product)), and the arithmetic.
template <typename T, int N>
struct Product {
  static constexpr int K = N / 4, E = N % 4;
  struct Ahead {
    T d[K > 0 ? K : 1], e[E > 0 ? E : 1];
    double a, c;
  };
  const T *DI;  // the lane's row of the system's inverses
  int q, lane;
  double v;  // the vector, lane = row
  __device__ __forceinline__ void columns(Ahead &B, int blk) const {
    const T *D = DI + (long)blk * (N * N);
#pragma unroll
    for (int k = 0; k < E; ++k) B.e[k] = D[(4 * K + k) * N];
    D += q * N;
#pragma unroll
    for (int k = 0; k < K; ++k) B.d[k] = D[4 * k * N];
  }
  __device__ __forceinline__ void multiply(const Ahead &B, double *out) const {
    double acc = 0.;
#pragma unroll
    for (int k = 0; k < K; ++k) acc = fma((double)B.d[k], lane_value(v, 4 * k + q), acc);
    if (E > 0 && q == 0) {
#pragma unroll
      for (int k = 0; k < E; ++k) acc = fma((double)B.e[k], lane_value(v, 4 * K + k), acc);
    }
    out[lane] = acc;
  }
  __device__ __forceinline__ double sum(const double (*p)[64]) const {
    return (p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane]);
  }
};

template <typename T, int N>
__global__ void __launch_bounds__(512) btd_twist_solve_kernel(const int *nblocks, const double *values, const long *voff,
                                                              const T *dinv, const long *doff, const double *rhs,
                                                              double *x, const long *xoff) {
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
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  const double *sub = values + voff[sys] + (long)nb * (N * N);
  const double *sup = sub + (long)(nb - 1) * N;

  // Every product loads the same number of words without a branch (clamped where there is nothing to load), so that a
  // wait counts the loads it needs and leaves the later products' in flight. y_i is kept in X.
  using Ahead = typename Product<T, N>::Ahead;
  Product<T, N> w{dinv + doff[sys] + rl, q, lane};
  double &v = w.v;
  if (nb == 1) {
    Ahead B;
    v = b[rl];
    w.columns(B, 0);
    w.multiply(B, part[0][0][q]);
    __syncthreads();
    if (q == 0 && act) X[lane] = w.sum(part[0][0]);
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
    w.columns(B, i);
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
    w.multiply(B, part[g & 1][chain][q]);
    // Loads that do not depend on this product go before the barrier. The addend has to be here by then: x may be rhs, and
    // behind the barrier other waves write what it was read from.
    const double a = s == len ? last : B.a, c = B.c;
    asm volatile("" ::"v"(B.a));
    operands(B, s + kAhead<T>);
    __syncthreads();
    if (g == L - 1) {
#pragma clang fp contract(off)
      const double tt = m > 0 ? ct * w.sum(part[g & 1][0]) : 0., tb = cb * w.sum(part[g & 1][1]);
      last = v;
      v = bm - tt - tb;
    } else if ((unsigned)s <= (unsigned)(2 * len)) {
      const bool in = s < len;
      const double mv = w.sum(part[g & 1][chain]);
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

// The same solve with one wave per chain, for small blocks and for many systems: a wave has all columns of a block, so a product
// needs no exchange, and the chains of a system meet at the middle block only. What bounds it is a product's chain of broadcasts
// and multiply-adds where systems are few, and the reads of the inverses where they are many; loads are issued two products
// ahead (one: 300 chains of 10..40 blocks of 10 24 us instead of 21; three take too many registers). Eight waves per
// system and this (us; before both, two waves per system that waited for their loads: third figure), chains of 10..40 blocks:
//   systems            FP64 4               10               20               32              40
//       1 of 60   26 / 19 / 31     32 / 24 / 56     37 / 37 / 64     50 / 54 / 83   59 / 65 / 109
//     300         24 / 16 / 24     35 / 21 / 42     42 / 35 / 57     58 / 51 / 82   69 / 61 / 113
//   1,000         40 / 20 / 26     65 / 34 / 59     77 / 56 / 81   106 / 90 / 106 158 / 152 / 181
//   4,000       114 / 56 / 65   189 / 100 / 148  269 / 222 / 247  404 / 397 / 440 548 / 553 / 646
//   systems            FP32 4               10               20               32              40
//       1 of 60   26 / 19 / 30     30 / 25 / 52     32 / 34 / 61     36 / 42 / 80   42 / 50 / 105
//     300         24 / 16 / 24     28 / 21 / 40     29 / 28 / 48     36 / 36 / 73   44 / 48 / 104
//   1,000         37 / 18 / 25     47 / 24 / 44     49 / 36 / 68     64 / 44 / 84   78 / 61 / 119
//   4,000        102 / 38 / 48    140 / 65 / 112   137 / 83 / 135  207 / 171 / 222 260 / 265 / 344
// (48: 4,000 chains 695 / 769 us FP64, 332 / 361 us FP32.) Bitwise the same.
constexpr int kWaveSolve = 40;  // its largest block
template <typename T>
constexpr int kWaveSolveAlways = sizeof(T) == 8 ? 20 : 16;  // the largest that it takes whatever the number of systems

template <typename T, int N>
__global__ void __launch_bounds__(128) btd_wave_solve_kernel(const int *nblocks, const double *values, const long *voff,
                                                             const T *dinv, const long *doff, const double *rhs, double *x,
                                                             const long *xoff) {
  __shared__ double part[2][64];
  const int lane = threadIdx.x & 63;
  const int chain = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool top = chain == 0;
  const int sys = blockIdx.x;
  const int nb = __builtin_amdgcn_readfirstlane(nblocks[sys]);
  if (!top && nb == 1) return;
  const bool act = lane < N;
  const int rl = act ? lane : 0;
  const int m = (nb - 1) / 2;
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  const double *sub = values + voff[sys] + (long)nb * (N * N);
  const double *sup = sub + (long)(nb - 1) * N;
  const T *DI = dinv + doff[sys] + rl;
  struct Ahead {
    T d[N];
    double a, c;
  };
  double v;
  auto columns = [&](Ahead &B, int i) {
    const T *D = DI + (long)i * (N * N);
#pragma unroll
    for (int k = 0; k < N; ++k) B.d[k] = D[k * N];
  };
  auto multiply = [&](const Ahead &B) {
    constexpr int K4 = N / 4 * 4;
    double p[4] = {0., 0., 0., 0.};
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int j = k < K4 ? k & 3 : 0;
      p[j] = fma((double)B.d[k], lane_value(v, k), p[j]);
    }
    return (p[0] + p[1]) + (p[2] + p[3]);
  };
  if (nb == 1) {
    Ahead B;
    v = b[rl];
    columns(B, 0);
    v = multiply(B);
    if (act) X[lane] = v;
    return;
  }
  // (products, places and loads as in the kernel above)
  const int L = nb - 1 - m;
  const int len = top ? m : L, off = L - len;
  const int first = top ? 0 : nb - 1, dir = top ? 1 : -1;
  auto block = [&](int s) { return first + dir * max(len - abs(len - s), 0); };
  auto at = [&](int i) { return (unsigned)(i * N + rl); };
  const double bm = b[at(m)], ct = m > 0 ? sub[at(m - 1)] : 0., cb = sup[at(m)];
  double last = 0.;
  v = b[at(block(0))];
  if (len > 0 && act) X[at(block(0))] = v;
  auto operands = [&](Ahead &B, int s) {
    const int i = block(s), j = block(s + 1);
    columns(B, i);
    B.c = (top == (s < len) ? sub : sup)[at(min(min(i, j), nb - 2))];
  };
  auto addend = [&](Ahead &B, int s) { B.a = (s < len ? b : X)[at(block(s + 1))]; };
  constexpr int A = 2;
  Ahead buf[A];
#pragma unroll
  for (int k = 0; k < A; ++k) {
    operands(buf[k], max(k - off, 0));
    addend(buf[k], max(k - off, 0));
  }
  auto product = [&](Ahead &B, int g) {
    const int s = g - off;
    const double mv = multiply(B);
    const double a = s == len ? last : B.a, c = B.c;
    asm volatile("" ::"v"(B.a));
    operands(B, s + A);
    if (g == L - 1) {
#pragma clang fp contract(off)
      part[chain][lane] = mv;
      __syncthreads();
      const double tt = m > 0 ? ct * part[0][lane] : 0., tb = cb * part[1][lane];
      last = v;
      v = bm - tt - tb;
    } else if ((unsigned)s <= (unsigned)(2 * len)) {
      const bool in = s < len;
      v = fma(-c, mv, a);
      if (act) X[at(block(in ? s + 1 : s))] = in ? v : mv;
    }
    addend(B, s + A);
  };
  for (int g = 0; g <= 2 * L; g += A) {
#pragma unroll
    for (int k = 0; k < A; ++k) {
      if (g + k > 2 * L) break;
      product(buf[k], g + k);
    }
  }
}

// The same solve with the two chains of a system on two compute units, for few systems of long chains: inwards and outwards one
// workgroup of four waves per chain (blockIdx.x = 2 system + chain), in between the middle block. Both chains of a system
// on one compute unit are bound by its cache fills (45 KB a product at 53); three launches cost about 8 us more.
// Measured (53x53, us, FP64 / FP32): one chain of 126 blocks 150 -> 100 / 108 -> 82, 48 chains of 62..254 312 -> 215 / 232 -> 176,
// 128 chains 397 -> 263 / 238 -> 184. Bitwise the same.
template <typename T, int N>
__global__ void __launch_bounds__(256) btd_chain_solve_kernel(const int *nblocks, const double *values, const long *voff,
                                                              const T *dinv, const long *doff, const double *rhs,
                                                              double *x, const long *xoff, int inwards) {
  __shared__ double part[2][4][64];
  const int sys = blockIdx.x >> 1;
  const bool top = (blockIdx.x & 1) == 0;
  const int lane = threadIdx.x & 63;
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = __builtin_amdgcn_readfirstlane(nblocks[sys]);
  const int m = (nb - 1) / 2, len = top ? m : nb - 1 - m;
  if (len == 0) return;
  const bool act = lane < N;
  const int rl = act ? lane : 0;
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  const double *sub = values + voff[sys] + (long)nb * (N * N);
  const double *sup = sub + (long)(nb - 1) * N;
  Product<T, N> w{dinv + doff[sys] + rl, q, lane};
  const int first = top ? 0 : nb - 1, dir = top ? 1 : -1;
  auto block = [&](int s) { return first + dir * max(len - abs(len - s), 0); };
  auto at = [&](int i) { return (unsigned)(i * N + rl); };
  auto coupling = [&](int s) { return (top == (s < len) ? sub : sup)[at(min(min(block(s), block(s + 1)), nb - 2))]; };
  const double *from = inwards ? b : X;
  const int s0 = inwards ? 0 : len + 1, s1 = inwards ? len - 1 : 2 * len + 1;  // products s0 .. s1 - 1
  if (inwards) {
    w.v = b[at(block(0))];
    if (act) X[at(block(0))] = w.v;  // every wave writes, and later reads, its own
  } else {
    w.v = fma(-coupling(len), X[at(m)], X[at(block(s0))]);
  }
  typename Product<T, N>::Ahead buf[kAhead<T>];
#pragma unroll
  for (int k = 0; k < kAhead<T>; ++k) {
    w.columns(buf[k], block(s0 + k));
    buf[k].c = coupling(s0 + k);
    buf[k].a = from[at(block(s0 + k + 1))];
  }
  auto product = [&](typename Product<T, N>::Ahead &B, int s) {
    w.multiply(B, part[s & 1][q]);
    const double a = B.a, c = B.c;
    asm volatile("" ::"v"(B.a));  // as above: x may be rhs
    w.columns(B, block(s + kAhead<T>));
    B.c = coupling(s + kAhead<T>);
    __syncthreads();
    const double mv = w.sum(part[s & 1]);
    w.v = fma(-c, mv, a);
    if (inwards ? act : act && q == 0) X[at(block(inwards ? s + 1 : s))] = inwards ? w.v : mv;
    B.a = from[at(block(s + kAhead<T> + 1))];
  };
  for (int s = s0; s < s1; s += kAhead<T>) {
#pragma unroll
    for (int k = 0; k < kAhead<T>; ++k) {
      if (s + k >= s1) break;
      product(buf[k], s + k);
    }
  }
}

template <typename T, int N>
__global__ void __launch_bounds__(512) btd_middle_solve_kernel(const int *nblocks, const double *values, const long *voff,
                                                               const T *dinv, const long *doff, const double *rhs,
                                                               double *x, const long *xoff) {
  __shared__ double part[2][2][4][64];
  const int sys = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chain = wave >> 2, q = wave & 3;
  const int nb = __builtin_amdgcn_readfirstlane(nblocks[sys]);
  const int m = (nb - 1) / 2;
  const bool act = lane < N, below = nb > 1;
  const int rl = act ? lane : 0;
  const double *b = rhs + xoff[sys];
  double *X = x + xoff[sys];
  const double *sub = values + voff[sys] + (long)nb * (N * N);
  const double *sup = sub + (long)(nb - 1) * N;
  auto at = [&](int i) { return (unsigned)(i * N + rl); };
  Product<T, N> w{dinv + doff[sys] + rl, q, lane};
  typename Product<T, N>::Ahead A, B;
  const int near = chain == 0 ? max(m - 1, 0) : min(m + 1, nb - 1);
  w.columns(A, near);
  w.columns(B, m);
  const double bm = b[at(m)], ct = m > 0 ? sub[at(m - 1)] : 0., cb = below ? sup[at(m)] : 0.;
  w.v = X[at(near)];
  w.multiply(A, part[0][chain][q]);
  asm volatile("" ::"v"(bm));
  __syncthreads();
  {
#pragma clang fp contract(off)
    const double tt = m > 0 ? ct * w.sum(part[0][0]) : 0., tb = below ? cb * w.sum(part[0][1]) : 0.;
    w.v = bm - tt - tb;
  }
  w.multiply(B, part[1][chain][q]);
  __syncthreads();
  if (wave == 0 && act) X[at(m)] = w.sum(part[1][0]);
}

template <typename T>
using InvSolve = void (*)(const int *, const double *, const long *, const T *, const long *, const double *, double *,
                          const long *);
template <typename T, int... I>
InvSolve<T> inv_solve_kernel(int bs, std::integer_sequence<int, I...>) {
  constexpr InvSolve<T> tab[] = {&btd_twist_solve_kernel<T, kWaveSolveAlways<T> + I + 1>...};
  return tab[bs - kWaveSolveAlways<T> - 1];
}
template <typename T, int... I>
InvSolve<T> wave_solve_kernel(int bs, std::integer_sequence<int, I...>) {
  constexpr InvSolve<T> tab[] = {&btd_wave_solve_kernel<T, I + 1>...};
  return tab[bs - 1];
}

}  // namespace

template <int... I>
static auto factor_kernel(int c, std::integer_sequence<int, I...>) {
  constexpr decltype(&btd_factor_kernel<1>) tab[] = {&btd_factor_kernel<I + 1>...};
  return tab[c - 1];
}

int launch_btd_factor(int nsys, const int *nblocks, int bs, double *values, const long *voff, double *l_values,
                      const long *loff, int *pivots, const long *poff, hipStream_t st) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  const auto kern = factor_kernel((bs + 7) / 8, std::make_integer_sequence<int, 8>{});
  hipLaunchKernelGGL(kern, dim3(nsys), dim3(64 * kLuWaves), 0, st, nblocks, bs, values, voff, l_values, loff, pivots,
                     poff);
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "btd factor launch failed");
  return GF_OK;
}

template <int... I>
static auto solve_kernel(int c, std::integer_sequence<int, I...>) {
  constexpr decltype(&btd_solve_kernel<8>) tab[] = {&btd_solve_kernel<8 * (I + 1)>...};
  return tab[c - 1];
}

int launch_btd_solve(int nsys, const int *nblocks, int bs, const double *values, const long *voff,
                     const double *l_values, const long *loff, const int *pivots, const long *poff, const double *rhs,
                     double *x, const long *xoff, hipStream_t st) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  const auto kern = solve_kernel((bs + 7) / 8, std::make_integer_sequence<int, 8>{});
  hipLaunchKernelGGL(kern, dim3(nsys), dim3(128), 0, st, nblocks, bs, values, voff, l_values, loff, pivots, poff, rhs, x,
                     xoff);
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "btd solve launch failed");
  return GF_OK;
}

template <typename T>
using ChainSolve = void (*)(const int *, const double *, const long *, const T *, const long *, const double *, double *,
                            const long *, int);
template <typename T, int... I>
static ChainSolve<T> chain_solve_kernel(int bs, std::integer_sequence<int, I...>) {
  constexpr ChainSolve<T> tab[] = {&btd_chain_solve_kernel<T, I + 1>...};
  return tab[bs - 1];
}
template <typename T, int... I>
static InvSolve<T> middle_solve_kernel(int bs, std::integer_sequence<int, I...>) {
  constexpr InvSolve<T> tab[] = {&btd_middle_solve_kernel<T, I + 1>...};
  return tab[bs - 1];
}

template <typename T>
int launch_btd_inv_solve(int nsys, const int *nblocks, int bs, const double *values, const long *voff,
                         const T *dinv, const long *doff, const double *rhs, double *x, const long *xoff,
                         hipStream_t st, long blocks) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  constexpr auto sizes = std::make_integer_sequence<int, 64>{};
  // Where the caller knows the number of blocks: a compute unit per chain while there are enough of them (256; 192 systems
  // of 53: 433 against 431 us, 512: 966 against 987), and chains long enough for the two launches more (one workgroup per
  // system against this, one system of 10 blocks of 10: 8 / 11 us, of 40: 22 / 21, of 40 of 53: 51 / 38).
  if (nsys <= 128 && blocks >= 40L * nsys) {
    const auto chain = chain_solve_kernel<T>(bs, sizes);
    hipLaunchKernelGGL(chain, dim3(2 * nsys), dim3(256), 0, st, nblocks, values, voff, dinv, doff, rhs, x, xoff, 1);
    hipLaunchKernelGGL(middle_solve_kernel<T>(bs, sizes), dim3(nsys), dim3(512), 0, st, nblocks, values, voff, dinv, doff,
                       rhs, x, xoff);
    hipLaunchKernelGGL(chain, dim3(2 * nsys), dim3(256), 0, st, nblocks, values, voff, dinv, doff, rhs, x, xoff, 0);
  } else if (bs <= kWaveSolveAlways<T> || (bs <= kWaveSolve && nsys >= (sizeof(T) == 8 ? 300 : 600))) {
    hipLaunchKernelGGL(wave_solve_kernel<T>(bs, std::make_integer_sequence<int, kWaveSolve>{}), dim3(nsys), dim3(128), 0, st,
                       nblocks, values, voff, dinv, doff, rhs, x, xoff);
  } else {
    const auto kern = inv_solve_kernel<T>(bs, std::make_integer_sequence<int, 64 - kWaveSolveAlways<T>>{});
    hipLaunchKernelGGL(kern, dim3(nsys), dim3(512), 0, st, nblocks, values, voff, dinv, doff, rhs, x, xoff);
  }
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "btd inverse solve launch failed");
  return GF_OK;
}

template int launch_btd_inv_solve<double>(int, const int *, int, const double *, const long *, const double *,
                                          const long *, const double *, double *, const long *, hipStream_t, long);
template int launch_btd_inv_solve<float>(int, const int *, int, const double *, const long *, const float *,
                                         const long *, const double *, double *, const long *, hipStream_t, long);

}  // namespace gfa
