// Gauss-Jordan inverses of one dense block in registers, every entry by the same sequence of fused multiply-adds whether
// one wave or two share the block: the one-wave-per-chain factor (gf_twist_small.hip) and the reactor batches' block
// inverse (gf_block_inverse.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "gf_wave.h"

namespace gfa {
namespace gj {

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

// ---- the same with the columns split over W waves ----
//
// The single-wave inverse above is a serial chain of N pivot steps, each a few hundred instructions of one
// wave (at N = 53: 52 slot updates of two readlanes and an fma each, plus the pivot search and the reciprocal).
// Splitting the columns of the block over W waves
// divides the update work of a step by W: wave w holds slots w*C .. w*C + C - 1 (C = ceil(N / W)) of every
// lane's row. Step j is pivoted by the wave that holds slot j; it publishes the multipliers g (one per lane;
// the pivot lane's entry carries its scale 1 / d) and the pivot lane through LDS, and after one workgroup
// barrier every wave updates its own slots. The arithmetic of every entry is the one of the single-wave
// routine (same pivot, same g, same fma, same final scaling), so the inverse is bitwise the same.
//
// All waves compute a pivot candidate on their own slot of step j (only the owner publishes it): that work
// sits in the same basic block as the updates of step j - 1, where the compiler can interleave it, and the
// other waves would otherwise wait at the barrier. The multipliers are double-buffered on the step parity
// `ph` (carried across calls), so one barrier per step suffices: the buffer written at step j was last read
// at step j - 2, before every wave passed the barrier of step j - 1.
template <int N>
constexpr int twist_waves() {
  return N >= 12 ? 2 : 1;
}

template <typename T, int N, int W>
__device__ __forceinline__ void split_gj_inverse(T (&x)[(N + W - 1) / W], int &rowid, int &colid, int lane, int w,
                                                 T *gb, int *pb, int &ph) {
  constexpr int C = (N + W - 1) / W;
  bool used = lane >= N;
  T sig = T(1);
  for (int ww = 0; ww < W; ++ww) {
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const int j = ww * C + k;
      if (j < N) {
        {
          const T f = x[k];
          const T rf = T(1) / f;  // every lane's reciprocal, formed beside the pivot search instead of after it
          const int p = wave_first_argmax(fabs(f), !used);  // N - j unused lanes remain, so p >= 0
          const T ipv = lane_value(rf, p);
          if (w == ww) {
            gb[ph * 64 + lane] = lane == p ? ipv : f * ipv;  // g of each row; the pivot lane carries 1 / d
            if (lane == 0) pb[ph] = p;
          }
        }
        __syncthreads();
        const int p = __builtin_amdgcn_readfirstlane(pb[ph]);
        const T gl = gb[ph * 64 + lane];
        ph ^= 1;
        const bool isp = lane == p;
        const T g = isp ? T(0) : gl;
#pragma unroll
        for (int c = 0; c < C; ++c) x[c] = fma(-g, lane_value(x[c], p), x[c]);
        if (w == ww) x[k] = isp ? T(1) : -g;  // the pivot column
        if (isp) sig = gl;
        const int cj = __builtin_amdgcn_readlane(colid, j);
        const int rp = __builtin_amdgcn_readlane(rowid, p);
        if (isp) {
          rowid = cj;
          used = true;
        }
        if (lane == j) colid = rp;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c) x[c] *= sig;
}

}  // namespace gj
}  // namespace gfa
