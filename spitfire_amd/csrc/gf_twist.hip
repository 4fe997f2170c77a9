// Twisted block factorisation with explicit inverses of the Schur-updated diagonal blocks (the factor half of
// the batched flamelet and reactor linear algebra), blocks of 1..64 unknowns, FP64 or FP32 inverses.
//
// Row i of a system is diag(sub_{i-1}) x_{i-1} + V_i x_i + diag(sup_i) x_{i+1} = b_i; with m = (n - 1) / 2
//   top chain:     D_0 = V_0,          D_i = V_i - diag(sub_{i-1}) D_{i-1}^{-1} diag(sup_{i-1}),  i = 1 .. m-1
//   bottom chain:  E_{n-1} = V_{n-1},  E_i = V_i - diag(sup_i) E_{i+1}^{-1} diag(sub_i),          i = n-2 .. m+1
//   middle:        C_m = V_m - diag(sub_{m-1}) D_{m-1}^{-1} diag(sup_{m-1}) - diag(sup_m) E_{m+1}^{-1} diag(sub_m)
// and block i of dinv receives D_i^{-1} (i < m), C_m^{-1} (i = m) or E_i^{-1} (i > m), column-major. The top half
// is the reference's forward block Thomas recurrence (btddod_matrix_kernels.cpp:19-80); the bottom half running
// at the same time halves the serial chain.
//
// Inverse of one block: blocked in-place Gauss-Jordan elimination with partial (row) pivoting, eight pivot columns
// (a panel) at a time, on the matrix cores. What bounds it is the serial chain of pivots, so the work between two
// pivots is kept small: one wave factors a panel with lane = row and the panel's eight columns in registers (a
// pivot is a wave-wide search, a reciprocal and seven fused multiply-adds), and the rank-8 update of every
// other column is two 16x16x4 MFMAs per 16x16 tile, spread over the chain's NT = ceil(N / 16) waves.
//   - Rows are never interchanged: the pivot of column k is the unused row p with the largest |entry|, and the
//     exchange is done in place at (p, k); the permutation is undone when the inverse is written to LDS, from where
//     the next Schur update and the store read it in order.
//   - Row scaling is deferred: row r is sig_r times its stored values, sig_p = 1/d from the step that pivots it. One
//     pivot (row p, column k, stored value d) is
//         rows r != p:  g_r = x_r[k] / d,  x_r[c] -= g_r x_p[c] (c != k),  x_r[k] = -g_r
//         row p:        x_p[k] = 1,  sig_p = 1 / d
//   - A panel of pivots (p_j, k_j) changes every other column c by x[c] += H x_P[c], x_P the old pivot rows and H_rj the
//     panel's own new entry x_r[k_j], less one at r = p_j (both are -A_rK A_PK^{-1} there, up to the deferred scale). The
//     wave that factors the panel keeps its columns less that one (so that H does not lose its last digits to it) and hands
//     back nothing else.
// What bounds it: a panel's eight pivots take about 2,800 cycles of its wave (50 instructions a pivot at one per four
// cycles and more, the lane shifts, scalar broadcasts and the reciprocal one after another), the hand-over to the tile
// waves, their first two MFMAs and the way back 1,100, a block's exchange and Schur update 4,000; FP64 MFMAs run on
// the vector FP64 units, so they do not overlap with a panel on the same SIMD. Before, every pivot was broadcast row
// by row through scalar registers to one or two waves, with a barrier a pivot. Measured before and after (53x53, us):
//   systems                     FP64             FP32
//   one chain of 126 blocks     2,248 -> 1,026   1,663 ->   732
//   256 chains of 62..254       4,807 -> 2,090   3,547 -> 1,508
//   512 chains                  6,455 -> 4,050   4,546 -> 2,911
//   1,024 chains               11,555 -> 7,071   8,106 -> 5,117
//   1,024 / 4,000 blocks       53 / 238 -> 46 / 172   45 / 155 -> 37 / 144
#include "gf_internal.h"
#include "gf_wave.h"
#include "../../include/griffon_amd.h"

namespace gfa {

namespace {

using wave::lane_value;

template <typename T>
using Vec4 = T __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Vec4<double> mfma4(double a, double b, Vec4<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Vec4<float> mfma4(float a, float b, Vec4<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Pivot search. The key of an unused row orders like |f|, up to the low bits of the mantissa that the lane number
// replaces (14 fraction bits are compared in FP64, 17 in FP32): a pivot within 1e-4 of the largest bounds the growth as
// well as the largest does, and one scan of 32-bit keys finds it without a second search among equal high words.
__device__ __forceinline__ unsigned magnitude(double f) { return (unsigned)__double2hiint(f) & 0x7fffffffu; }
__device__ __forceinline__ unsigned magnitude(float f) { return (unsigned)__float_as_int(f) & 0x7fffffffu; }
template <typename T>
__device__ __forceinline__ unsigned pivot_key(T f, bool used, int lane) {
  return used ? 0u : (magnitude(f) & ~63u) | (unsigned)(63 - lane);
}
// step k = 0 .. 5 of the wave-wide maximum of the keys, complete in lane 63 after step 5
template <int K>
__device__ __forceinline__ unsigned max_step(unsigned v) {
  constexpr int ctrl[6] = {0x111, 0x112, 0x114, 0x118, 0x142, 0x143};  // row_shr 1, 2, 4, 8, row_bcast 15, 31
  constexpr int rows[6] = {0xF, 0xF, 0xF, 0xF, 0xA, 0xC};
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl[K], rows[K], 0xF, false));
}
__device__ __forceinline__ int pivot_of(unsigned scanned) {
  return 63 - (int)((unsigned)__builtin_amdgcn_readlane((int)scanned, 63) & 63u);
}

// 1 / x in steps that are spread between other work: the hardware reciprocal, two Newton steps (FP64), and zeros,
// infinities and NaN as a division gives them. About half the dependent chain of the division.
struct Recip64 {
  double x, r, e;
  template <int K>
  __device__ __forceinline__ void step() {
    if constexpr (K == 0) r = __builtin_amdgcn_rcp(x);
    else if constexpr (K == 1 || K == 3) e = fma(-x, r, 1.);
    else if constexpr (K == 2 || K == 4) r = fma(r, e, r);
    else r = __builtin_amdgcn_div_fixup(r, x, 1.);
  }
};
struct Recip32 {
  float x, r;
  template <int K>
  __device__ __forceinline__ void step() {
    if constexpr (K == 0) r = 1.f / x;
  }
};
__device__ __forceinline__ Recip64 recip_of(double x) { return Recip64{x, 0., 0.}; }
__device__ __forceinline__ Recip32 recip_of(float x) { return Recip32{x, 0.f}; }

// One chain's LDS. Rows and columns are padded to Np = 8 ceil(N / 8) by an identity, so that every panel is full: the
// padding's pivots are its own ones. M holds the block before each panel's update, a row as [lane group][tile][register]
// (the pivot rows are read from it), and between two blocks the inverse, column-major with stride IS.
template <typename T, int NT>
struct ChainLds {
  static constexpr int R = 16 * NT;
  static constexpr int GS = 4 * NT + 2;  // stride of a lane group, and MS of a row: they spread the banks
  static constexpr int MS = 4 * GS + 2;
  static constexpr int IS = R + 2;
  static constexpr int PS = 10;  // stride of a row of P: spreads the rows over the banks
  alignas(16) T P[R][PS];  // the panel's columns before its elimination, then H: [row][column]
  T sig[R];         // scale of each row: the reciprocal of its pivot
  double cs[4][4 * NT + 1];  // column scales of the next Schur update, column 16 t + 4 k + g at [g][4 t + k]
  int rowj[R];      // which of the panel's pivots a row is, -1 if none
  int prow[R];      // pivot row of each column
  static __host__ __device__ constexpr int words(int np) {  // of M: np rows and one that takes the rows beyond
    return (np + 1) * MS > R * IS ? (np + 1) * MS : R * IS;
  }
};

// The wave that factors a chain's panels, lane = row. Per panel: eight pivots, each found among the unused rows,
//   h_r = -x_r[k] / d (0 at the pivot row),  x_r[c] += h_r x_p[c] for the panel's other columns,  H_r[k] = h_r.
// Only the panel's columns are touched here. A single wave issues at most one instruction every four cycles and the
// search of the next pivot is a chain of dependent lane shifts, so a step updates the next pivot's column first
// and then does one lane shift, one step of the next reciprocal and one of the six other columns at a time, in an
// order that the compiler's scheduler (which otherwise runs the chains one after the other) has to keep.
template <typename T, int NT>
__device__ __forceinline__ void factor_panels(ChainLds<T, NT> &s, int Np, int lane) {
  const int row = NT == 4 || lane < 16 * NT ? lane : 0;
  bool used = lane >= Np;
  T sig = T(1);
  for (int base = 0; base < Np; base += 8) {
    __syncthreads();
    T f[8];
    typedef T V2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const V2 g = *reinterpret_cast<const V2 *>(&s.P[row][j]);
      f[j] = g[0];
      f[j + 1] = g[1];
    }
    int rj = -1;
    unsigned key = pivot_key(f[0], used, lane);
    auto rc = recip_of(f[0]);
    key = max_step<0>(key); rc.template step<0>();
    key = max_step<1>(key); rc.template step<1>();
    key = max_step<2>(key); rc.template step<2>();
    key = max_step<3>(key); rc.template step<3>();
    key = max_step<4>(key); rc.template step<4>();
    key = max_step<5>(key); rc.template step<5>();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = pivot_of(key);  // Np - base - j unused rows remain
      const T ip = lane_value(rc.r, p);
      const bool isp = lane == p;
      const T h = isp ? T(0) : -(f[j] * ip);
      auto update = [&](int c) { f[c & 7] = fma(h, lane_value(f[c & 7], p), f[c & 7]); };
      used = used || isp;
      rj = isp ? j : rj;
      sig = isp ? ip : sig;
      if (j < 7) {
        update(j + 1);
        key = pivot_key(f[(j + 1) & 7], used, lane);
        rc = recip_of(f[(j + 1) & 7]);
        rc.template step<0>();
        __builtin_amdgcn_sched_barrier(0);
        key = max_step<0>(key); rc.template step<1>(); update(j + 2);
        __builtin_amdgcn_sched_barrier(0);
        key = max_step<1>(key); rc.template step<2>(); update(j + 3);
        __builtin_amdgcn_sched_barrier(0);
        key = max_step<2>(key); rc.template step<3>(); update(j + 4);
        __builtin_amdgcn_sched_barrier(0);
        key = max_step<3>(key); rc.template step<4>(); update(j + 5);
        __builtin_amdgcn_sched_barrier(0);
        key = max_step<4>(key); rc.template step<5>(); update(j + 6);
        __builtin_amdgcn_sched_barrier(0);
        key = max_step<5>(key); update(j + 7);
        f[j] = h;
        __builtin_amdgcn_sched_barrier(0);
      } else {
#pragma unroll
        for (int c = 0; c < 7; ++c) update(c);
        f[7] = h;
      }
    }
    if (NT == 4 || lane < 16 * NT) {
#pragma unroll
      for (int j = 0; j < 8; j += 2) *reinterpret_cast<V2 *>(&s.P[lane][j]) = V2{f[j], f[j + 1]};
      s.rowj[lane] = rj;
      if (base + 8 == Np) s.sig[lane] = sig;
      if (rj >= 0) s.prow[base + rj] = lane;
    }
    __syncthreads();
  }
}

// A block row as its NT tile waves hold it: wave w has rows 16 w .. 16 w + 15 of every column. The tile of columns
// 16 ct .. 16 ct + 15 is the transpose of an MFMA accumulator: register q of lane l holds row 16 w + (l & 15), column
// 16 ct + 4 q + (l >> 4), so a panel of eight neighbouring columns is two registers.
template <typename T, int NT>
struct Tiles {
  using S = ChainLds<T, NT>;
  Vec4<T> x[NT];

  // In-place elimination of all columns: afterwards element (row, column) times s.sig[row] is element (kap,
  // s.prow[column]) of the inverse; returns kap, the pivot column of the lane's row. `idle(k)` runs while panel k = 0 or 1
  // is factored. Of a panel's update only the tile that holds the next panel is waited for; the other tiles'
  // MFMAs (operands a0, a1, b0, b1) and the copy to M are issued while the next panel is factored.
  template <class F>
  __device__ __forceinline__ int eliminate(S &s, T *M, int Np, int w, int lane, F idle) {
    const int r16 = lane & 15, grp = lane >> 4, row = 16 * w + r16;
    // row i of the left operand is column 4 q + g of the tile, i = 4 q + g in an FP64 accumulator, 4 g + q in FP32
    constexpr bool f64 = sizeof(T) == 8;
    const T *src = M + (f64 ? (r16 & 3) : (r16 >> 2)) * S::GS + (f64 ? (r16 >> 2) : (r16 & 3));
    T *dst = M + min(row, Np) * S::MS + grp * S::GS;
    int kap = row;
    T a0[NT], a1[NT], b0 = T(0), b1 = T(0), pn0 = T(0), pn1 = T(0);
#pragma unroll
    for (int t = 0; t < NT; ++t) a0[t] = a1[t] = T(0);
    auto update = [&](int t) { x[t] = mfma4(a1[t], b1, mfma4(a0[t], b0, x[t])); };
    auto pending = [&](bool wrapped) {
#pragma unroll
      for (int t = 1; t < NT; ++t) update(t);
      if (NT > 1 && wrapped) {
        x[NT - 1][2] = pn0;
        x[NT - 1][3] = pn1;
      }
    };
    auto rotate = [&] {  // the next column tile moves to register tile 0 (back in place after NT of these)
      const Vec4<T> x0 = x[0];
      const T c0 = a0[0], c1 = a1[0];
#pragma unroll
      for (int t = 0; t + 1 < NT; ++t) {
        x[t] = x[t + 1];
        a0[t] = a0[t + 1];
        a1[t] = a1[t + 1];
      }
      x[NT - 1] = x0;
      a0[NT - 1] = c0;
      a1[NT - 1] = c1;
    };
    s.P[row][grp] = x[0][0];
    s.P[row][4 + grp] = x[0][1];
    for (int ct = 0; ct < NT; ++ct) {
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        const int base = 16 * ct + 4 * q;
        if (base < Np) {
          __syncthreads();
          if (q > 0 || ct > 0) pending(q == 0);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            typedef T V2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<V2 *>(dst + 4 * t) = V2{x[t][0], x[t][1]};
            *reinterpret_cast<V2 *>(dst + 4 * t + 2) = V2{x[t][2], x[t][3]};
          }
          if (ct == 0) idle(q / 2);
          __syncthreads();
          const int p0 = s.prow[base + grp], p1 = s.prow[base + 4 + grp], rj = s.rowj[row];
          b0 = s.P[row][grp];
          b1 = s.P[row][4 + grp];
          pn0 = b0 + (rj == grp ? T(1) : T(0));
          pn1 = b1 + (rj == 4 + grp ? T(1) : T(0));
          kap = rj >= 0 ? base + rj : kap;
          const T *s0 = src + p0 * S::MS, *s1 = src + p1 * S::MS;
          constexpr int tn = (NT > 1) ? 1 : 0;
          const int first = q == 2 ? tn : 0;  // the tile of the next panel
          a0[first] = s0[4 * first];
          a1[first] = s1[4 * first];
          update(first);
#pragma unroll
          for (int t = 0; t < NT; ++t)
            if (t != first) {
              a0[t] = s0[4 * t];
              a1[t] = s1[4 * t];
            }
          if (first == 0) {
            x[0][q] = pn0;
            x[0][q + 1] = pn1;
          } else {
            rotate();
          }
          s.P[row][grp] = x[0][(q + 2) & 3];
          s.P[row][4 + grp] = x[0][((q + 2) & 3) + 1];
          __builtin_amdgcn_sched_barrier(0);  // the pending MFMAs stay behind the next panel's hand-over
        }
      }
    }
    const bool wrapped = ((Np - 1) & 8) == 8;  // the last panel was its tile's last: already rotated
    pending(wrapped);
    if (!wrapped) rotate();
    return kap;
  }

  // the padding's identity: ones on the diagonal beyond the block
  __device__ __forceinline__ void pad(int N, int w, int lane) {
    const int r16 = lane & 15, grp = lane >> 4;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (t == w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[t][k] = (16 * w + r16 >= N && 4 * k + grp == r16) ? T(1) : x[t][k];
      }
  }
};

// Elements (row, column) of a block in memory through a buffer descriptor of its N x N elements: those outside the block
// read as zero and are not written, without a branch or a select per element.
template <typename E>
struct Window {
  __amdgpu_buffer_rsrc_t rsrc;
  int at, step;  // byte offset of (row, group's column), bytes of one column
  __device__ __forceinline__ Window(const E *base, int N, int row, int grp)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<E *>(base), 0, N * N * (int)sizeof(E), 0x00020000)),
        at(row < N ? (grp * N + row) * (int)sizeof(E) : (1 << 30)), step(N * (int)sizeof(E)) {}
  __device__ __forceinline__ E load(int c) const {
    if constexpr (sizeof(E) == 8) return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(rsrc, at + c * step, 0, 0));
    else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rsrc, at + c * step, 0, 0));
  }
  __device__ __forceinline__ void store(int c, E v) const {
    typedef unsigned U2 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(E) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), rsrc, at + c * step, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc, at + c * step, 0, 0);
  }
};

// One workgroup of 2 (NT + 1) waves per system: for the top chain NT tile waves and the wave that factors its panels, then
// the same for the bottom chain. Both chains run max(len) inverses so that every wave passes the same barriers: the
// shorter chain starts with one inverse of the identity, which it discards. The middle block is inverted by the top
// chain alone, which reads the bottom chain's last inverse from LDS. While a block's first two panels are factored, the
// tile waves store the inverse before it and load the values of the block after it.
template <typename T, int NT>
__global__ void __launch_bounds__(128 * (NT + 1)) __attribute__((amdgpu_waves_per_eu(NT == 1 ? 8 : NT == 2 ? 5 : NT == 3 ? 4 : 2)))
twist_factor_kernel(int nsys, const int *nblocks, int n, const double *values, const long *voff, T *dinv, const long *doff) {
  using S = ChainLds<T, NT>;
  extern __shared__ char m_raw[];
  __shared__ S lds[2];
  // Two one-block systems share a workgroup, the second (256 further on, so that the workgroups that are left without
  // work are spread evenly over the XCDs and compute units) in the bottom chain's place.
  const int other = blockIdx.x ^ 256;
  const bool paired = other < nsys && nblocks[blockIdx.x] == 1 && nblocks[other] == 1;
  if (paired && (blockIdx.x & 256)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: kept in scalar registers
  const bool top = wave <= NT;
  const bool lead = top || paired;  // the chain that inverts a middle block
  const int sys = paired && !top ? other : blockIdx.x;
  const int w = top ? wave : wave - (NT + 1);
  S &s = lds[top ? 0 : 1];
  int N = n;
  const int Np = (n + 7) & ~7;
  T *M = reinterpret_cast<T *>(m_raw) + (top ? 0 : S::words(Np));
  const T *E = reinterpret_cast<const T *>(m_raw) + S::words(Np);  // the bottom chain's inverse
  const long NB2 = (long)n * n;
  const int nb = __builtin_amdgcn_readfirstlane(nblocks[sys]);
  const int m = (nb - 1) / 2;
  const double *V = values + voff[sys];
  const double *sub = V + nb * NB2;
  const double *sup = sub + (long)(nb - 1) * n;
  T *Dg = dinv + doff[sys];
  const int len = top ? m : nb - 1 - m;
  const int iters = nb - 1 - m;  // >= m
  // block t of the chain: its index, the index of the next one (the top chain's last is the middle block), whether there
  // is a next one, and whether that has this one's Schur term (not after the leading identity)
  auto index = [&](int t) { return t == iters ? m : (top ? t - (iters - len) : nb - 1 - (t - (iters - len))); };
  auto more = [&](int t) { return t < iters && (t + 1 < iters || lead); };
  auto join = [&](int t) { return t >= iters - len; };

  if (w == NT) {  // panels
    if (lane < 16 * NT) s.prow[lane] = lane;  // columns beyond the padding keep their place
    for (int t = 0; t <= iters; ++t) {
      if (t == iters && !lead) return;  // the barriers of the middle inverse wait only on the waves still running
      double csv = 0.;
      if (more(t) && join(t)) {
        const int in = index(t + 1);
        csv = (top ? sup + (long)(in - 1) * N : sub + (long)in * N)[min(lane, N - 1)];
      }
      factor_panels<T, NT>(s, Np, lane);
      if (lane < 16 * NT) s.cs[lane & 3][lane >> 2] = lane < N ? csv : 0.;
      __syncthreads();
      __syncthreads();
    }
    return;
  }

  const int r16 = lane & 15, grp = lane >> 4, row = 16 * w + r16;
  Tiles<T, NT> b;
  {
    const Window<double> v(V + (top ? 0 : nb - 1) * NB2, N, row, grp);
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        b.x[u][k] = len < iters ? (row == 16 * u + 4 * k + grp ? T(1) : T(0)) : (T)v.load(16 * u + 4 * k);
    b.pad(N, w, lane);
  }
  T d[NT][4];
  bool keep = false;  // d holds the inverse of block index(t - 1), not stored yet
  for (int t = 0; t <= iters; ++t) {
    // opaque to the compiler, so that the element offsets are formed again for each block instead of being kept in
    // (and spilled from) registers through the elimination
    asm volatile("" : "+s"(N));
    if (t == iters && !lead) {
      if (keep) {
        const Window<T> o(Dg + index(t - 1) * NB2, N, row, grp);
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) o.store(16 * u + 4 * k, d[u][k]);
      }
      return;
    }
    const bool nxt = more(t);
    double v[NT][4], r = 0.;
    const int kap = b.eliminate(s, M, Np, w, lane, [&](int k) {
      if (k == 0 && keep) {
        const Window<T> o(Dg + index(t - 1) * NB2, N, row, grp);
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) o.store(16 * u + 4 * k, d[u][k]);
      }
      if (k == (Np > 8 ? 1 : 0) && nxt) {  // not used before the block's inverse is done
        const int in = index(t + 1);
        const Window<double> vi(V + in * NB2, N, row, grp);
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) v[u][k] = vi.load(16 * u + 4 * k);
        r = (top ? sub + (long)(in > 0 ? in - 1 : 0) * N : sup + (long)in * N)[min(row, N - 1)];
      }
    });
    __syncthreads();  // M becomes the inverse
    {
      const T sig = s.sig[row];
      T *to = M + kap;
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) to[s.prow[16 * u + 4 * k + grp] * S::IS] = b.x[u][k] * sig;
    }
    __syncthreads();
    const int nat = grp * S::IS + row;
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k) d[u][k] = M[nat + (16 * u + 4 * k) * S::IS];
    keep = t >= iters - len || t == iters;
    if (nxt) {
      r = join(t) && row < N ? r : 0.;
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) b.x[u][k] = (T)(v[u][k] - r * s.cs[grp][4 * u + k] * (double)d[u][k]);
      if (t + 1 == iters) {  // the top chain: the bottom chain's term of the middle block
        const double rm = row < N ? sup[(long)m * N + row] : 0.;
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int c = 16 * u + 4 * k + grp;
            const double cm = sub[(long)m * N + min(c, N - 1)];
            b.x[u][k] = (T)((double)b.x[u][k] - (c < N ? rm * cm : 0.) * (double)E[nat + (16 * u + 4 * k) * S::IS]);
          }
      }
      b.pad(N, w, lane);
    }
  }
  const Window<T> o(Dg + m * NB2, N, row, grp);
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int k = 0; k < 4; ++k) o.store(16 * u + 4 * k, d[u][k]);
}

template <typename T, int NT>
int launch_nt(int nsys, const int *nblocks, int bs, const double *values, const long *voff, T *dinv,
              const long *doff, hipStream_t st) {
  auto kern = twist_factor_kernel<T, NT>;
  const size_t lds = 2 * sizeof(T) * ChainLds<T, NT>::words((bs + 7) & ~7);
  if (lds + 2 * sizeof(ChainLds<T, NT>) > 65536 &&
      hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(GF_ERR_UNSUPPORTED, "block too large for LDS");
  hipLaunchKernelGGL(kern, dim3(nsys), dim3(128 * (NT + 1)), lds, st, nsys, nblocks, bs, values, voff, dinv, doff);
  return hipGetLastError() == hipSuccess ? GF_OK : fail(GF_ERR_HIP, "btd inverse factor launch failed");
}

}  // namespace

template <typename T>
int launch_btd_inv_factor(int nsys, const int *nblocks, int bs, const double *values, const long *voff, T *dinv,
                          const long *doff, hipStream_t st) {
  if (nsys <= 0) return GF_OK;
  if (bs < 1 || bs > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  // Blocks below 12 in batches of at least six systems per compute unit: one wave per chain without barriers is faster
  // there when the systems are single blocks (4,000 blocks of 10: 12 against 20 us FP64, 9 against 16 us FP32) and
  // about even on chains (3,000 chains of 30-99 blocks of 6: 303 against 347 us, of 10: 702 against 640 us); with fewer
  // systems or larger blocks the kernel above wins (1,024 chains of 13: 289 against 491 us).
  if (bs <= kSmallFactor && nsys >= 1536)
    return launch_btd_inv_factor_small<T>(nsys, nblocks, bs, values, voff, dinv, doff, st);
  switch ((bs + 15) / 16) {
    case 1: return launch_nt<T, 1>(nsys, nblocks, bs, values, voff, dinv, doff, st);
    case 2: return launch_nt<T, 2>(nsys, nblocks, bs, values, voff, dinv, doff, st);
    case 3: return launch_nt<T, 3>(nsys, nblocks, bs, values, voff, dinv, doff, st);
    default: return launch_nt<T, 4>(nsys, nblocks, bs, values, voff, dinv, doff, st);
  }
}

template int launch_btd_inv_factor<double>(int, const int *, int, const double *, const long *, double *, const long *,
                                           hipStream_t);
template int launch_btd_inv_factor<float>(int, const int *, int, const double *, const long *, float *, const long *,
                                          hipStream_t);

}  // namespace gfa
