// df_tiles.h -- layout of the density-fitting factor B in HBM, and the exchange
// products that read it (df_mfma.hip).
//
// Row Q holds the symmetric n x n matrix B_Q as the 32 x 32 tiles (I, J),
// I >= J, of its lower triangle, tile after tile (I(I+1)/2 + J), each row-major
// and zero past n; the tiles on the diagonal are whole.  Against packed rows
// (src/df.rs:121, n(n+1)/2 a row) that is 1.6 % more at n = 2080 and 4 % at
// n = 800, and every tile is 8 KB that starts 16-byte aligned: the matrix-core
// kernels stage it with wide loads and no index arithmetic, above and below
// the diagonal alike.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "engine.h"

namespace hfg {

constexpr int TL = 32;
__host__ __device__ inline int tiles_of(int n) { return (n + TL - 1) / TL; }
// Doubles of one row Q.
__host__ __device__ inline size_t tiled_size(int n) {
  const size_t t = tiles_of(n);
  return t * (t + 1) / 2 * (TL * TL);
}
__host__ __device__ inline size_t tile_index(int I, int J) {
  return I >= J ? (size_t)I * (I + 1) / 2 + J : (size_t)J * (J + 1) / 2 + I;
}
// Position of element (i, j), i >= j or both in one tile row.
__host__ __device__ inline size_t tiled_at(int i, int j) {
  return tile_index(i / TL, j / TL) * (TL * TL) + (i % TL) * TL + j % TL;
}

// Workspace of the exchange products, kept by the factor's owner and grown to
// the largest call.
struct ExchangeWork {
  struct Buf : DevBuf {
    void grow(size_t b) {
      if (bytes < b) alloc(b);
    }
  };
  Buf c, x, part, sums;
};

// K = 2 sum_Q (B_Q C)(B_Q C)^T of the tiled factor (rank rows of npt doubles) and
// C (n x o, row-major); precision 0 FP64, 1 FP32 operands and accumulation, 2
// each operand split into two BF16 parts, three products in FP32 (the sums over
// the slices of the contraction in FP64).  With gamma (FP64 only), also
// gamma[Q] = 2 tr(B_Q C C^T).  On stream st.
void df_exchange(const double* Bt, size_t npt, int rank, int n, const double* C, int o, int precision, double* K,
                 double* gamma, ExchangeWork& w, hipStream_t st);
// Grows the workspace to what such a call needs, which then allocates nothing.
void df_exchange_reserve(int rank, int n, int o, int precision, bool gamma, ExchangeWork& w);

}  // namespace hfg
