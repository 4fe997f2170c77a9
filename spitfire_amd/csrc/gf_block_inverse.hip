// Inverses of many independent dense blocks (the Newton and adjoint matrices of a reactor batch, one n x n block per
// reactor): every block is inverted in registers by Gauss-Jordan elimination with partial pivoting, two waves per block
// (one below 12 unknowns). The elimination applies the same operations to every entry in the same order as it always
// has, so a reactor batch's trajectories do not change: its Newton test (residual below 1e-12) sits at rounding level,
// and another rounding of the inverse ends some stages an iteration earlier or later, which moves an igniting batch's
// heat release gradients by 4e-8 relative (measured with the blocked elimination of gf_twist.hip in its place).
// Bound by the serial chain of pivots. Two waves a block, 128 registers a lane: four blocks per compute unit run at
// once, one wave per SIMD for each half.
#include "gf_internal.h"
#include "gf_gj.h"
#include "../../include/griffon_amd.h"

#include <utility>

namespace gfa {

namespace {

template <int N>
__global__ void __launch_bounds__(64) block_inverse_kernel(const double *values, double *inv) {
  const double *V = values + (long)blockIdx.x * N * N;
  double *D = inv + (long)blockIdx.x * N * N;
  const int lane = threadIdx.x;
  double x[N];
  int rowid = lane, colid = lane;
  const int rl = lane < N ? lane : 0;
#pragma unroll
  for (int k = 0; k < N; ++k) x[k] = V[k * N + rl];
  gj::reg_gj_inverse<double, N>(x, rowid, colid, lane);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int c = __builtin_amdgcn_readlane(colid, k);
    if (lane < N) D[c * N + rowid] = x[k];
  }
}

template <int N>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(4)))
block_inverse_split_kernel(const double *values, double *inv) {
  constexpr int C = (N + 1) / 2;
  __shared__ double gb[2 * 64];
  __shared__ int pb[2];
  const double *V = values + (long)blockIdx.x * N * N;
  double *D = inv + (long)blockIdx.x * N * N;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double x[C];
  int rowid = lane, colid = lane, ph = 0;
  const int rl = lane < N ? lane : 0;
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const int s = w * C + k;
    x[k] = V[(s < N ? s : 0) * N + rl];
  }
#pragma unroll
  for (int k = 0; k < C; ++k) x[k] = (lane < N && w * C + k < N) ? x[k] : 0.;
  gj::split_gj_inverse<double, N, 2>(x, rowid, colid, lane, w, gb, pb, ph);
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const int s = w * C + k;
    if (s < N) {
      const int c = __builtin_amdgcn_readlane(colid, s);
      if (lane < N) D[c * N + rowid] = x[k];
    }
  }
}

template <int N>
void launch_block_inverse(int nblk, const double *values, double *inv, hipStream_t st) {
  if constexpr (N < 12)
    hipLaunchKernelGGL(block_inverse_kernel<N>, dim3(nblk), dim3(64), 0, st, values, inv);
  else
    hipLaunchKernelGGL(block_inverse_split_kernel<N>, dim3(nblk), dim3(128), 0, st, values, inv);
}

using Fn = void (*)(int, const double *, double *, hipStream_t);

template <int... I>
Fn block_inverse_fn(int n, std::integer_sequence<int, I...>) {
  constexpr Fn tab[] = {&launch_block_inverse<I + 1>...};
  return tab[n - 1];
}

}  // namespace

}  // namespace gfa

extern "C" int gf_batch_block_inverse(int nblk, int n, const double *values, double *inv, void *stream) {
  using namespace gfa;
  if (nblk <= 0) return GF_OK;
  if (n < 1 || n > 64) return fail(GF_ERR_UNSUPPORTED, "block size must be in 1..64");
  if (!values || !inv) return fail(GF_ERR_ARG, "null argument");
  block_inverse_fn(n, std::make_integer_sequence<int, 64>{})(nblk, values, inv, static_cast<hipStream_t>(stream));
  return hipGetLastError() == hipSuccess ? GF_OK : fail(GF_ERR_HIP, "block inverse launch failed");
}
