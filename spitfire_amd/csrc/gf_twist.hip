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
// Inverse of one block: in-place Gauss-Jordan elimination with partial (row) pivoting, eight pivot columns (a panel) at a
// time, on the matrix cores. What bounds it is the serial chain of pivots, so the work between two
// pivots is kept small: one wave factors a panel with lane = row and the panel's eight columns in registers (a
// pivot is a wave-wide search, a reciprocal and at most seven fused multiply-adds), and the rank-8 update of the
// columns is two 16x16x4 MFMAs per 16x16 tile, spread over the chain's NT = ceil(N / 16) tile waves.
//   - Rows are never interchanged: the pivot of column k is the unused row p with the largest |entry|, and the
//     exchange is done in place at (p, k); the order of rows and columns that this leaves is carried to the next block.
//   - Row scaling is deferred: row r is sig_r times its stored values, sig_p = 1/d from the step that pivots it. One
//     pivot (row p, column k, stored value d) is
//         rows r != p:  g_r = -x_r[k] / d,  x_r[c] += g_r x_p[c] (c != k),  x_r[k] = g_r
//         row p:        x_p[k] = 1,  sig_p = 1 / d
//   - A panel of pivots (p_j, k_j) adds g_rj u_j[c], j = 0 .. 7 to column c of row r, where u_j is row p_j as it is when it is
//     pivoted: u_j[c] = x_pj[c] + g_{pj,0} u_0[c] + .. + g_{pj,j-1} u_{j-1}[c]. The panel's own columns are columns like the
//     others, starting from g_rj (1 at row p_j), with u_i = 0 up to their own pivot.
//   - An MFMA accumulates its four products in ascending order with one rounding each, and u_j is formed in the same
//     order, so every entry passes through the same fused multiply-adds as in an elimination pivot by pivot: the
//     inverses are bitwise those of gf_twist_small.hip, whatever the panel and tile sizes.
// What bounds it: a panel's eight pivots take about 3,400 cycles of its wave (the lane shifts of the search, the scalar
// broadcasts and the division one after another), forming the u_j, the first two MFMAs and the two hand-overs 1,900, the
// change to the next block 2,000. FP64 MFMAs run on the vector FP64 units, so they do not overlap with a panel on the same
// SIMD. Before, every pivot was broadcast row by row through scalar registers to one or two waves, with a barrier a
// pivot. Measured before and after (53x53, us):
//   systems                     FP64             FP32
//   one chain of 126 blocks     2,248 -> 1,140   1,663 ->   854
//   256 chains of 62..254       4,807 -> 2,386   3,547 -> 1,818
//   512 chains                  6,455 -> 4,580   4,546 -> 3,520
//   1,024 chains               11,555 -> 8,046   8,106 -> 6,184
//   1,024 single blocks            53 ->    50      45 ->    42  (more of them: many_singles)
// (The panel's multipliers instead of the u_j, H = -A_rK A_PK^{-1}, save the substitution, 1,026 us for the chain, but round
// differently.)
#include "gf_internal.h"
#include "gf_wave.h"
#include "../../include/griffon_amd.h"

#include <climits>

namespace gfa {

namespace {

using wave::lane_value;
using wave::max_step;
using wave::recip_of;

template <typename T>
using Vec4 = T __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Vec4<double> mfma4(double a, double b, Vec4<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Vec4<float> mfma4(float a, float b, Vec4<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Pivot search: the first unused row with the largest |f|, on the bit patterns. A row's key is the word of its entry that
// holds the exponent under its mask, which is 0 once the row is used.
__device__ __forceinline__ unsigned key_of(double f, unsigned mask) { return (unsigned)__double2hiint(f) & mask; }
__device__ __forceinline__ unsigned key_of(float f, unsigned mask) { return (unsigned)__float_as_int(f) & mask; }
template <typename T>
__device__ __forceinline__ int pivot_of(unsigned scanned, unsigned key, T f, unsigned mask) {
  const unsigned top = (unsigned)__builtin_amdgcn_readlane((int)scanned, 63);
  unsigned long long hit = __ballot(key == top);
  if constexpr (sizeof(T) == 8) {
    if (hit & (hit - 1)) {  // rare: the low words decide (or all are zero, and used rows have that key as well)
      const bool in = (key == top) & (mask != 0u);
      const unsigned lo = in ? (unsigned)__double2loint(f) : 0u;
      const unsigned most = wave::dpp_wave_max_u32(lo);
      hit = __ballot(in & (lo == most));
    }
  } else {
    if (top == 0u) hit = __ballot(mask != 0u);
  }
  return __builtin_ctzll(hit);
}

// One chain's LDS. Panels and tiles are whole ones: pivots go up to Np = 8 ceil(N / 8), rows and columns to 16 NT. What the rows
// and columns beyond the block hold is arbitrary (V has no entries for them: a row beyond reads the next column's, a column
// beyond words that nothing has written), and never gets into the block: rows beyond are not searched and are never pivots, the
// steps beyond N have multipliers and pivot rows of zero, and an MFMA's output depends on its own row and column only.
// Two more arrays are in dynamic LDS: M, the block before each panel's update, a row as
// [lane group][tile][register] (the pivot rows are read from it), and V, the values of the chain's next block, column-major.
template <typename T, int NT>
struct ChainLds {
  static constexpr int R = 16 * NT;
  static constexpr int GS = 4 * NT;      // stride of a lane group, and MS of a row, which spreads the banks
  static constexpr int MS = 4 * GS + 2;
  static constexpr int PS = 10;  // stride of a row of P and G: spreads the rows over the banks
  static constexpr int CS = 4 * NT + 2;
  alignas(16) T P[R][PS];  // the panel's columns before its elimination: [row][column]
  alignas(16) T G[R][PS];  // multipliers of the panel's pivots: [row][pivot]
  double cs[4][CS];        // column scales of the next Schur update, column 16 t + 4 k + g at [g][4 t + k]
  double rs[R];            // its row scales
  T sig[R];                // scale of each row: the reciprocal of its pivot
  alignas(16) int prow[R];  // pivot row of each column
  int rowid[R];            // the row and the column of the inverse that a row and a column hold, N for those beyond it
  alignas(16) int colid[4][CS + 2];
  static __host__ __device__ constexpr int m_words(int np) { return (np + 1) * MS; }  // a row more, for those beyond
  static __host__ __device__ constexpr int v_words(int n) { return (n + 1) * n + 1; }
};

// The wave that factors a chain's panels, lane = row. Per panel: eight pivots, each found among the unused rows, the
// multipliers g_r = -x_r[k] / d (0 at the pivot row), and x_r[c] += g_r x_p[c] for the panel's later columns c. Only these
// are touched here. A single wave issues at most one instruction every four cycles and the
// search of the next pivot is a chain of dependent lane shifts, so a step updates the next pivot's column first
// and then does one lane shift, one step of the next reciprocal and one of the other columns at a time, in an
// order that the compiler's scheduler (which otherwise runs the chains one after the other) has to keep.
// Columns beyond the block (left <= j) are not pivoted. Returns the pivot column of the lane's row.
template <bool PART, typename T>
__device__ __forceinline__ void panel_pivots(T (&f)[8], T (&g)[8], unsigned &mask, T &sig, int &rj, int left, int lane) {
  unsigned key = key_of(f[0], mask), most = key;
  auto rc = recip_of(f[0]);
  most = max_step<0>(most); rc.template step<0>();
  most = max_step<1>(most); rc.template step<1>();
  most = max_step<2>(most); rc.template step<2>();
  most = max_step<3>(most); rc.template step<3>();
  most = max_step<4>(most); rc.template step<4>();
  most = max_step<5>(most); rc.template step<5>();
  rc.template step<6>();
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (PART && j > 0 && left <= j) {
      g[j] = T(0);
      continue;
    }
    const int p = pivot_of(most, key, f[j], mask);  // left - j unused rows remain
    const bool isp = lane == p;
    T h = f[j] * -lane_value(rc.r, p);
    asm("" : "+v"(h));  // (a select, not a branch around the product)
    h = isp ? T(-0.) : h;
    g[j] = h;
    auto update = [&](int c) {
      if (c < 8) f[c] = fma(h, lane_value(f[c], p), f[c]);
    };
    mask = isp ? 0u : mask;
    rj = isp ? j : rj;
    sig = isp ? rc.r : sig;
    if (j < 7) {
      update(j + 1);
      most = key = key_of(f[(j + 1) & 7], mask);
      rc = recip_of(f[(j + 1) & 7]);
      rc.template step<0>();
      __builtin_amdgcn_sched_barrier(0);
      most = max_step<0>(most); rc.template step<1>(); update(j + 2);
      __builtin_amdgcn_sched_barrier(0);
      most = max_step<1>(most); rc.template step<2>(); update(j + 3);
      __builtin_amdgcn_sched_barrier(0);
      most = max_step<2>(most); rc.template step<3>(); update(j + 4);
      __builtin_amdgcn_sched_barrier(0);
      most = max_step<3>(most); rc.template step<4>(); update(j + 5);
      __builtin_amdgcn_sched_barrier(0);
      most = max_step<4>(most); rc.template step<5>(); update(j + 6);
      __builtin_amdgcn_sched_barrier(0);
      most = max_step<5>(most); rc.template step<6>(); update(j + 7);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <typename T, int NT>
__device__ __forceinline__ int factor_panels(ChainLds<T, NT> &s, int N, int Np, int lane) {
  const int row = NT == 4 || lane < 16 * NT ? lane : 0;
  unsigned mask = lane < N ? 0x7fffffffu : 0u;
  T sig = T(1);
  int kap = lane;
  for (int base = 0; base < Np; base += 8) {
    __syncthreads();
    T f[8], g[8];
    typedef T V2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const V2 v = *reinterpret_cast<const V2 *>(&s.P[row][j]);
      f[j] = v[0];
      f[j + 1] = v[1];
    }
    int rj = -1;
    if (base + 8 <= N) panel_pivots<false>(f, g, mask, sig, rj, 8, lane);
    else panel_pivots<true>(f, g, mask, sig, rj, N - base, lane);
    if (NT == 4 || lane < 16 * NT) {
#pragma unroll
      for (int j = 0; j < 8; j += 2) *reinterpret_cast<V2 *>(&s.G[lane][j]) = V2{g[j], g[j + 1]};
      if (base + 8 == Np) s.sig[lane] = sig;
      if (rj >= 0) s.prow[base + rj] = lane;
    }
    __syncthreads();
    kap = rj >= 0 ? base + rj : kap;
  }
  return kap;
}

// a[i] of lane group k becomes a[k] of lane group i: the four registers' 16-lane rows transposed
__device__ __forceinline__ void swap_halves(int &a, int &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap_rows(int &a, int &b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
template <typename T>
__device__ __forceinline__ void transpose4(T &a, T &b, T &c, T &d) {
  constexpr int W = sizeof(T) / 4;
  typedef int Words __attribute__((ext_vector_type(W)));
  int v[4][W];
  auto get = [&](int i, T x) {
    if constexpr (W == 1) v[i][0] = __builtin_bit_cast(int, x);
    else {
      const Words q = __builtin_bit_cast(Words, x);
      v[i][0] = q[0];
      v[i][W - 1] = q[W - 1];
    }
  };
  auto put = [&](int i) {
    if constexpr (W == 1) return __builtin_bit_cast(T, v[i][0]);
    else return __builtin_bit_cast(T, Words{v[i][0], v[i][W - 1]});
  };
  get(0, a); get(1, b); get(2, c); get(3, d);
#pragma unroll
  for (int k = 0; k < W; ++k) {
    swap_halves(v[0][k], v[2][k]);
    swap_halves(v[1][k], v[3][k]);
    swap_rows(v[0][k], v[1][k]);
    swap_rows(v[2][k], v[3][k]);
  }
  a = put(0); b = put(1); c = put(2); d = put(3);
}
// the value of lane L of each 16-lane row, in all lanes of that row
template <int L, typename T>
__device__ __forceinline__ T row_lane(T v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + L, 0xF, 0xF, true);
}

// A block row as its NT tile waves hold it: wave w has rows 16 w .. 16 w + 15 of every column. The tile of columns
// 16 ct .. 16 ct + 15 is the transpose of an MFMA accumulator: register q of lane l holds row 16 w + (l & 15), column
// 16 ct + 4 q + (l >> 4), so a panel of eight neighbouring columns is two registers.
template <typename T, int NT>
struct Tiles {
  using S = ChainLds<T, NT>;
  Vec4<T> x[NT];
  T a[2][4];  // left operands by tile: pivots 0 .. 3 and 4 .. 7 of a panel
  T b0, b1;

  // Left operands of all tiles for the panel at `base` (lane group g: the rows of pivots g and 4 + g, as each is when it
  // is pivoted), with lane = column of the NT tiles.
  __device__ __forceinline__ void pivot_rows(const S &s, const T *M, int base, int N, int lane) {
    const int n = lane & 15;
    // lane n of each 16 holds the n-th multiplier of the pivot rows 1 .. 5, and of the rows 6 and 7
    const int ja = n < 1 ? 1 : n < 3 ? 2 : n < 6 ? 3 : n < 10 ? 4 : 5, jb = n < 6 ? 6 : 7;
    const int pa = s.prow[base + ja], pb = s.prow[base + jb];
    typedef int I4 __attribute__((ext_vector_type(4)));
    const I4 p0 = *reinterpret_cast<const I4 *>(&s.prow[base]), p1 = *reinterpret_cast<const I4 *>(&s.prow[base + 4]);
    // row i of the left operand is column 4 q + g of the tile, i = 4 q + g in an FP64 accumulator, 4 g + q in FP32
    constexpr bool f64 = sizeof(T) == 8;
    const int g = f64 ? (n & 3) : (n >> 2), k = f64 ? (n >> 2) : (n & 3);
    // column c of the panel starts from its multipliers at pivot c
    int c = (lane & 48) + 4 * k + g - base;
    c = (unsigned)c < 8u ? c : -1;
    asm volatile("" : "+v"(c));  // opaque: its comparisons are not kept (and spilled) over the blocks for each panel
    const T *src = c >= 0 ? &s.G[0][c] : M + g * S::GS + 4 * min(lane >> 4, NT - 1) + k;
    const int stride = c >= 0 ? S::PS : S::MS;
    const T la = s.G[pa][n - ja * (ja - 1) / 2], lb = s.G[pb][n < 6 ? n : n - 6];
    T u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = src[(j < 4 ? p0[j & 3] : p1[j & 3]) * stride];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = c < j ? u[j] : T(0);
#define GF_ROW(J, I, L, AT) u[J] = fma(row_lane<AT>(L), u[I], u[J]);
    GF_ROW(1, 0, la, 0)
    GF_ROW(2, 0, la, 1) GF_ROW(2, 1, la, 2)
    GF_ROW(3, 0, la, 3) GF_ROW(3, 1, la, 4) GF_ROW(3, 2, la, 5)
    GF_ROW(4, 0, la, 6) GF_ROW(4, 1, la, 7) GF_ROW(4, 2, la, 8) GF_ROW(4, 3, la, 9)
    GF_ROW(5, 0, la, 10) GF_ROW(5, 1, la, 11) GF_ROW(5, 2, la, 12) GF_ROW(5, 3, la, 13) GF_ROW(5, 4, la, 14)
    GF_ROW(6, 0, lb, 0) GF_ROW(6, 1, lb, 1) GF_ROW(6, 2, lb, 2) GF_ROW(6, 3, lb, 3) GF_ROW(6, 4, lb, 4) GF_ROW(6, 5, lb, 5)
    GF_ROW(7, 0, lb, 6) GF_ROW(7, 1, lb, 7) GF_ROW(7, 2, lb, 8) GF_ROW(7, 3, lb, 9) GF_ROW(7, 4, lb, 10)
    GF_ROW(7, 5, lb, 11) GF_ROW(7, 6, lb, 12)
#undef GF_ROW
    if (base + 8 > N) {
#pragma unroll
      for (int j = 1; j < 8; ++j) u[j] = base + j < N ? u[j] : T(0);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      transpose4(u[4 * h], u[4 * h + 1], u[4 * h + 2], u[4 * h + 3]);
#pragma unroll
      for (int t = 0; t < 4; ++t) a[h][t] = u[4 * h + t];
    }
  }

  __device__ __forceinline__ void update(int t) { x[t] = mfma4(a[1][t], b1, mfma4(a[0][t], b0, x[t])); }

  // what is left of a panel's update: every tile but the one that was waited for
  __device__ __forceinline__ void pending(int done) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (t != done) update(t);
  }

  // In-place elimination of all columns. On entry tile 0 is complete, and `enter` completes the other ones
  // while the first panel is factored; on return tile 0 is complete up to its rows' scale s.sig, and pending(0) does the
  // others. `idle` runs while the second panel is factored (the first, if there is one tile only). Of a panel's update only
  // the tile that holds the next panel is waited for; the other tiles' MFMAs and the copy to M are issued while the
  // next panel is factored.
  template <class Enter, class Idle>
  __device__ __forceinline__ void eliminate(S &s, T *M, int N, int Np, int w, int lane, Enter enter, Idle idle) {
    const int r16 = lane & 15, grp = lane >> 4, row = 16 * w + r16;
    T *dst = M + min(row, Np) * S::MS + grp * S::GS;
    s.P[row][grp] = x[0][0];
    s.P[row][4 + grp] = x[0][1];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        const int base = 16 * ct + 4 * q;
        if (ct + 1 < NT || base < Np) {
          __syncthreads();
          if (q == 0 && ct == 0) enter();
          else pending(ct);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            typedef T V2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<V2 *>(dst + 4 * t) = V2{x[t][0], x[t][1]};
            *reinterpret_cast<V2 *>(dst + 4 * t + 2) = V2{x[t][2], x[t][3]};
          }
          if (ct == 0 && q == (NT == 1 ? 0 : 2)) idle();
          __syncthreads();
          b0 = s.G[row][grp];
          b1 = s.G[row][4 + grp];
          x[ct][q] = s.prow[base + grp] == row ? T(1) : b0;
          x[ct][q + 1] = s.prow[base + 4 + grp] == row ? T(1) : b1;
          pivot_rows(s, M, base, N, lane);
          const bool last = ct + 1 == NT && base + 8 == Np;
          if (last) {
            update(0);
          } else {
            const int next = q == 2 ? (ct + 1 < NT ? ct + 1 : 0) : ct;
            update(next);
            s.P[row][grp] = x[next][(q + 2) & 3];
            s.P[row][4 + grp] = x[next][((q + 2) & 3) + 1];
          }
          __builtin_amdgcn_sched_barrier(0);  // the pending MFMAs stay behind the next panel's hand-over
        }
      }
  }
};

// Elements of a block in memory through a buffer descriptor of its N x N elements: those outside the block read as zero
// and are not written, without a branch or a select per element.
template <typename E>
struct Window {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ Window(const E *base, int N)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<E *>(base), 0, N * N * (int)sizeof(E), 0x00020000)) {}
  __device__ __forceinline__ E load(int e) const {
    if constexpr (sizeof(E) == 8) return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(rsrc, e * 8, 0, 0));
    else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rsrc, e * 4, 0, 0));
  }
  __device__ __forceinline__ void store(int e, E v) const {
    typedef unsigned U2 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(E) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), rsrc, e * 8, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc, e * 4, 0, 0);
  }
};

// One workgroup of 2 (NT + 1) waves per system: for the top chain NT tile waves and the wave that factors its panels, then
// the same for the bottom chain. Both chains run max(len) inverses so that every wave passes the same barriers: the
// shorter chain starts with one inverse of the identity, which it discards. The middle block is inverted by the top
// chain alone, which reads the bottom chain's term from its V. A block keeps the order of rows and columns that the inverse
// before it left (the panel wave tracks it), so the inverse never moves between lanes; the next block's values, which the
// tile waves bring to LDS while the second panel is factored, are read in that order. Only register tile 0 of the Schur
// update, which holds the next panel, is waited for: the others and the store follow while that panel is factored.
template <typename T, int NT>
__global__ void __launch_bounds__(128 * (NT + 1)) __attribute__((amdgpu_waves_per_eu(NT == 1 ? 6 : NT == 2 ? 5 : NT == 3 ? 4 : 2)))
twist_factor_kernel(int nsys, const int *nblocks, int n, const double *values, const long *voff, T *dinv, const long *doff,
                    int least) {
  using S = ChainLds<T, NT>;
  extern __shared__ double v_raw[];
  __shared__ S lds[2];
  if (nblocks[blockIdx.x] < least) return;  // (systems of fewer blocks are another kernel's)
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
  double *Vb = v_raw + S::v_words(n);  // the bottom chain's
  double *Vl = top ? v_raw : Vb;
  T *M = reinterpret_cast<T *>(v_raw + ((2 * S::v_words(n) + 1) & ~1)) + (top ? 0 : S::m_words(Np));
  const long NB2 = (long)n * n;
  const int nb = __builtin_amdgcn_readfirstlane(nblocks[sys]);
  const int m = (nb - 1) / 2;
  const double *V = values + voff[sys];
  const double *sub = V + nb * NB2;
  const double *sup = sub + (long)(nb - 1) * n;
  T *Dg = dinv + doff[sys];
  const int len = top ? m : nb - 1 - m;
  const int iters = nb - 1 - m;  // >= m
  // block t of the chain: its index, the index of the next one (both chains' last is the middle block), and whether that
  // has this one's Schur term (not after the leading identity)
  auto index = [&](int t) { return t == iters ? m : (top ? t - (iters - len) : nb - 1 - (t - (iters - len))); };
  auto join = [&](int t) { return t >= iters - len; };

  if (w == NT) {  // panels
    __builtin_amdgcn_s_setprio(3);
    int rowid = lane, colid = lane;
    if (lane < 16 * NT) s.prow[lane] = lane;  // columns beyond the padding keep their place
    for (int t = 0; t <= iters; ++t) {
      if (t == iters && !lead) return;  // the barriers of the middle inverse wait only on the waves still running
      double rsv = 0., csv = 0.;
      if (t < iters && join(t) && lane < N) {
        const int in = index(t + 1);
        rsv = (top ? sub + (long)(in - 1) * N : sup + (long)in * N)[lane];
        csv = (top ? sup + (long)(in - 1) * N : sub + (long)in * N)[lane];
      }
      const int kap = factor_panels<T, NT>(s, N, Np, lane);
      const int p = s.prow[lane < 16 * NT ? lane : 0];
      const int rn = __shfl(colid, kap), cn = lane < 16 * NT ? __shfl(rowid, p) : lane;
      rowid = rn;
      colid = cn;
      const double rl = __shfl(rsv, rowid), cl = __shfl(csv, colid);
      if (lane < 16 * NT) {
        s.rowid[lane] = min(rowid, N);
        s.colid[lane & 3][lane >> 2] = min(colid, N);
        s.rs[lane] = rl;
        s.cs[lane & 3][lane >> 2] = cl;
      }
      __syncthreads();
      if (t + 1 == iters) __syncthreads();
    }
    return;
  }

  const int r16 = lane & 15, grp = lane >> 4, row = 16 * w + r16;
  Tiles<T, NT> b;
  {
    const Window<double> v(V + (top ? 0 : nb - 1) * NB2, N);
    const int at = row < N ? grp * N + row : 1 << 27;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        b.x[u][k] = len < iters ? (row == 16 * u + 4 * k + grp ? T(1) : T(0)) : (T)v.load(at + (16 * u + 4 * k) * N);
    }
  }
  int rid = 0;
  T sig = T(1);
  double r = 0.;
  bool keep = false;
  // tile u of the inverse of block index(t): its values d and places e, and the same tile of the block after it
  auto schur = [&](int t, int u, int (&e)[4], Vec4<T> &d) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      e[k] = s.colid[grp][4 * u + k] * N + rid;
      d[k] = b.x[u][k] * sig;
    }
    if (t < iters) {
#pragma unroll
      for (int k = 0; k < 4; ++k) b.x[u][k] = (T)(Vl[e[k]] - r * s.cs[grp][4 * u + k] * (double)d[k]);
      if (t + 1 == iters) {
#pragma unroll
        for (int k = 0; k < 4; ++k) b.x[u][k] = (T)((double)b.x[u][k] - Vb[e[k]]);
      }
    }
  };
  auto store = [&](int t, const int (&e)[4], const Vec4<T> &d) {
    if (keep && rid < N) {
      const Window<T> o(Dg + index(t) * NB2, N);
#pragma unroll
      for (int k = 0; k < 4; ++k) o.store(e[k], d[k]);
    }
  };
  int e0[4];
  Vec4<T> d0;
  auto complete = [&](int t) {  // the other tiles
    b.pending(0);
    store(t, e0, d0);
#pragma unroll
    for (int u = 1; u < NT; ++u) {
      int e[4];
      Vec4<T> d;
      schur(t, u, e, d);
      store(t, e, d);
    }
  };
  for (int t = 0; t <= iters; ++t) {
    // opaque to the compiler, so that the element offsets are formed again for each block instead of being kept in
    // (and spilled from) registers through the elimination
    asm volatile("" : "+s"(N));
    if (t == iters && !lead) return;
    b.eliminate(
        s, M, N, Np, w, lane,
        [&] {
          if (t > 0) complete(t - 1);
        },
        [&] {
          if (t < iters && (t + 1 < iters || lead)) {
            const Window<double> v(V + index(t + 1) * NB2, N);
            const int e = w * 64 + lane;
            double q[4 * NT];
#pragma unroll
            for (int k = 0; k < 4 * NT; ++k) q[k] = v.load(e + 64 * NT * k);
#pragma unroll
            for (int k = 0; k < 4 * NT; ++k) Vl[min(e + 64 * NT * k, N * N)] = q[k];
          }
        });
    __syncthreads();  // the order of the inverse, the scales
    rid = s.rowid[row];
    r = s.rs[row];
    sig = s.sig[row];
    keep = join(t) || t == iters;
    if (t + 1 == iters) {
      if (!lead) {  // the bottom chain's term of the middle block, and its last store
        b.pending(0);
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int c = s.colid[grp][4 * u + k];
            const T x = b.x[u][k] * sig;
            if (rid < N && c < N) {
              Vl[c * N + rid] = r * (double)x * s.cs[grp][4 * u + k];
              Dg[index(t) * NB2 + c * N + rid] = x;
            }
          }
      }
      __syncthreads();
      if (!lead) return;
    }
    schur(t, 0, e0, d0);
  }
  complete(iters);
}

template <typename T, int NT>
int launch_nt(int nsys, const int *nblocks, int bs, const double *values, const long *voff, T *dinv,
              const long *doff, int least, hipStream_t st) {
  auto kern = twist_factor_kernel<T, NT>;
  using S = ChainLds<T, NT>;
  const size_t lds = sizeof(double) * ((2 * S::v_words(bs) + 1) & ~1) + 2 * sizeof(T) * S::m_words((bs + 7) & ~7);
  if (lds + 2 * sizeof(S) > 65536 &&
      hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(GF_ERR_UNSUPPORTED, "block too large for LDS");
  hipLaunchKernelGGL(kern, dim3(nsys), dim3(128 * (NT + 1)), lds, st, nsys, nblocks, bs, values, voff, dinv, doff,
                     least);
  return hipGetLastError() == hipSuccess ? GF_OK : fail(GF_ERR_HIP, "btd inverse factor launch failed");
}

// From how many systems on the one-block systems of a batch have a launch of their own, one wave each, ahead of the panels' (how
// many there are is known on the device only; panels take the rest). A wave takes time with the block's size, panels with the
// tiles that it is padded to, and of these fewer fit a compute unit with each tile. Single blocks, panels and one wave (us):
//                     FP64 17         20         27         32         33         48         53         64
//   1,536 systems   19 -> 16   21 -> 19   26 -> 29   27 -> 38   44 -> 39   68 -> 73   74 -> 87  89 -> 117
//   2,048 systems   22 -> 16   23 -> 19   29 -> 29   30 -> 40   52 -> 40   90 -> 76   97 -> 89 117 -> 120
//   4,000 systems   39 -> 26   41 -> 33   53 -> 51   56 -> 67   93 -> 70 174 -> 131 186 -> 155 226 -> 220
//                     FP32 17         20         28         32         33         48         53         64
//   1,280 systems   15 -> 12   16 -> 14   20 -> 21   20 -> 27   28 -> 26   40 -> 47   60 -> 56   68 -> 70
//   1,536 systems   17 -> 12   17 -> 14   22 -> 21   22 -> 27   34 -> 26   49 -> 48   64 -> 58   73 -> 72
//   4,000 systems   33 -> 19   34 -> 23   48 -> 39   52 -> 50   76 -> 49  100 -> 85 168 -> 102 189 -> 131
// Batches of chains lose the launch, 2 us (1,536 chains of 2..7 blocks of 20: 91 -> 94 us).
template <typename T>
int many_singles(int n) {
  if (sizeof(T) == 4) return n <= 22 ? 1025 : n >= 29 && n <= 32 ? 4000 : 1536;
  if (n <= 20) return 1280;
  if (n >= 28 && n <= 32) return INT_MAX;
  return n >= 23 && n <= 27 ? 3000 : n <= 38 ? 1536 : 1537;  // (three rounds of panels at one workgroup per compute unit)
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
  // systems or larger blocks the kernel above wins (1,024 chains of 13: 289 against 491 us). Blocks of up to 4 would be padding
  // for the most part: one wave whatever the batch (one chain of 126 blocks of 1 / 4 unknowns 30 / 97 against 90 / 117 us FP64, 28 /
  // 85 against 80 / 103 us FP32, 300 chains of 40..99 of 4 92 against 100 us; of 5 120 against 126 and 115 against 108 us).
  if (bs <= 4 || (bs <= kSmallFactor && nsys >= 1536))
    return launch_btd_inv_factor_small<T>(nsys, nblocks, bs, values, voff, dinv, doff, st);
  int least = 1;
  if (bs >= kSingleFrom && nsys >= many_singles<T>(bs)) {
    const int rc = launch_btd_inv_factor_single<T>(nsys, nblocks, bs, values, voff, dinv, doff, st);
    if (rc != GF_OK) return rc;
    least = 2;
  }
  switch ((bs + 15) / 16) {
    case 1: return launch_nt<T, 1>(nsys, nblocks, bs, values, voff, dinv, doff, least, st);
    case 2: return launch_nt<T, 2>(nsys, nblocks, bs, values, voff, dinv, doff, least, st);
    case 3: return launch_nt<T, 3>(nsys, nblocks, bs, values, voff, dinv, doff, least, st);
    default: return launch_nt<T, 4>(nsys, nblocks, bs, values, voff, dinv, doff, least, st);
  }
}

template int launch_btd_inv_factor<double>(int, const int *, int, const double *, const long *, double *, const long *,
                                           hipStream_t);
template int launch_btd_inv_factor<float>(int, const int *, int, const double *, const long *, float *, const long *,
                                          hipStream_t);

}  // namespace gfa
