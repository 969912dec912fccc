// la_batch.h -- FP64 linear algebra over many matrices of different sizes in
// one launch: the batched RHF iterations run every molecule's products,
// reductions and purification steps together instead of one library call per
// molecule.  Row-major matrices throughout.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "engine.h"

namespace hfg {

// One product C (M x N, leading dimension ldc) = alpha op(A) op(B) + beta C,
// op(A) M x K, op(B) K x N; skip (optional, device) nonzero skips it.
struct GemmOp {
  const double* A;
  const double* B;
  double* C;
  int M, N, K, lda, ldb, ldc;
  double alpha, beta;
  int ta, tb;
  const int* skip;
};

// 32 x 32 tile of one product per workgroup (grid: N tiles, M tiles, ops): each
// of four waves a 16 x 16 block on the FP64 matrix cores (v_mfma_f64_16x16x4:
// operands row or column l % 16, contraction index l / 16; result column l % 16,
// rows l / 16 + 4 r).  The products are small (m 25 to a few hundred) and a
// purification step waits for each, so what counts is the latency of one tile's
// chain of k panels: panels 32 wide, the next one on its way to registers during
// the current one's MFMAs, two LDS buffers, one barrier a panel.  Panels are held
// [row][k] with a padding column.  Forty def2-SVP molecules: 18.6 us a launch;
// 67 us with 64 x 64 tiles on the vector units, 16-wide panels loaded after the
// barrier.
// Out-of-range tiles of the smaller products of a launch exit at once.
constexpr int GT = 32, GP = GT + 1;
__global__ __launch_bounds__(256) inline void k_gemm_batched(const GemmOp* __restrict__ ops) {
  typedef double d4 __attribute__((ext_vector_type(4)));
  const GemmOp& op = ops[blockIdx.z];
  if (op.skip && *op.skip) return;
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  const int M = op.M, N = op.N, K = op.K, lda = op.lda, ldb = op.ldb;
  if (m0 >= M || n0 >= N) return;
  __shared__ double As[2][GT * GP], Bs[2][GT * GP];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, lo = t & 31, hi = t >> 5;
  const double* __restrict__ A = op.A;
  const double* __restrict__ B = op.B;
  const bool ta = op.ta, tb = op.tb;
  double va[4], vb[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int x = hi + 8 * r;  // consecutive lanes along the stored rows
      const int am = m0 + (ta ? lo : x), ak = k0 + (ta ? x : lo);
      va[r] = am < M && ak < K ? A[ta ? (size_t)ak * lda + am : (size_t)am * lda + ak] : 0.0;
      const int bn = n0 + (tb ? x : lo), bk = k0 + (tb ? lo : x);
      vb[r] = bn < N && bk < K ? B[tb ? (size_t)bn * ldb + bk : (size_t)bk * ldb + bn] : 0.0;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int x = hi + 8 * r;
      As[buf][ta ? lo * GP + x : x * GP + lo] = va[r];
      Bs[buf][tb ? x * GP + lo : lo * GP + x] = vb[r];
    }
  };
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  const int am = 16 * (w >> 1) + (lane & 15), bn = 16 * (w & 1) + (lane & 15), g = lane >> 4;
  load(0);
  store(0);
  if (K > GT) load(GT);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < K; k0 += GT, buf ^= 1) {
    if (k0 + GT < K) {
      store(buf ^ 1);
      if (k0 + 2 * GT < K) load(k0 + 2 * GT);
    }
    const double *a = As[buf] + am * GP + g, *b = Bs[buf] + bn * GP + g;
#pragma unroll
    for (int kk = 0; kk < GT; kk += 4) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kk], b[kk], acc, 0, 0, 0);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int gm = m0 + 16 * (w >> 1) + g + 4 * r, gn = n0 + bn;
    if (gm >= M || gn >= N) continue;
    double* c = op.C + (size_t)gm * op.ldc + gn;
    *c = op.beta == 0.0 ? op.alpha * acc[r] : op.alpha * acc[r] + op.beta * *c;
  }
}

// A fixed list of products run together: built on the host and uploaded once
// (when the set of molecules changes), then launched any number of times.
struct GemmList {
  std::vector<GemmOp> ops;
  DevBuf d_ops;
  int mt = 0, nt = 0, count = 0;
  void clear() { ops.clear(); }
  void add(bool ta, bool tb, int M, int N, int K, double alpha, const double* A, int lda, const double* B, int ldb,
           double beta, double* C, int ldc, const int* skip = nullptr) {
    ops.push_back(GemmOp{A, B, C, M, N, K, lda, ldb, ldc, alpha, beta, ta ? 1 : 0, tb ? 1 : 0, skip});
  }
  // Copies the list to the device (synchronously: the host list may change next).
  void upload(hipStream_t s) {
    count = (int)ops.size();
    mt = nt = 0;
    for (const GemmOp& o : ops) {
      mt = std::max(mt, (o.M + GT - 1) / GT);
      nt = std::max(nt, (o.N + GT - 1) / GT);
    }
    if (!count) return;
    if (d_ops.bytes < ops.size() * sizeof(GemmOp)) {
      HIP_CHECK(hipStreamSynchronize(s));  // a previous launch may still read the old array
      d_ops.alloc(std::max<size_t>(ops.size(), 64) * sizeof(GemmOp));
    }
    HIP_CHECK(hipMemcpyAsync(d_ops.p, ops.data(), ops.size() * sizeof(GemmOp), hipMemcpyHostToDevice, s));
    HIP_CHECK(hipStreamSynchronize(s));
  }
  void launch(hipStream_t s) const {
    for (int z0 = 0; z0 < count; z0 += 65535) {
      const unsigned nz = (unsigned)std::min(65535, count - z0);
      hipLaunchKernelGGL(k_gemm_batched, dim3(nt, mt, nz), dim3(256), 0, s, d_ops.as<GemmOp>() + z0);
    }
    HIP_CHECK(hipGetLastError());
  }
};

}  // namespace hfg
