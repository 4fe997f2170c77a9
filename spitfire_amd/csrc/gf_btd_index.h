// Offsets within the values of one block-tridiagonal system (griffon's BTDDOD format): nb blocks of bs x bs, then nb - 1
// rows of bs sub-diagonals, then as many of super-diagonals. No device code: checked on the host as well.
#pragma once

#ifdef __HIPCC__
#define GF_INDEX __host__ __device__ constexpr
#else
#define GF_INDEX constexpr
#endif

namespace gfa {

GF_INDEX long btd_values(int nb, int bs) { return (long)bs * ((long)nb * bs + 2l * (nb - 1)); }

// The super-diagonals that couple block i to block i + 1. For kernels that load them ahead, for every block alike: where there
// are none (i < 0, the last block, one block alone), a row of bs values that is in range all the same and is not used.
GF_INDEX long btd_sup(int nb, int bs, int i) {
  const int last = nb - 2, row = i < last ? i : last;
  return nb > 1 ? (long)nb * bs * bs + (long)(nb - 1 + (row > 0 ? row : 0)) * bs : 0;
}

}  // namespace gfa
