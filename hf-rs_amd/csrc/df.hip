// df.hip -- Coulomb-metric density fitting on the GPU: metric (P|Q), the
// 3-index tensor (P|mu nu), the whitened factor B = X^T (P|mu nu) with
// X = U_kept lambda^{-1/2} of the metric (canonical orthogonaliser, cutoff
// 1e-10), DF-J/K, and the DF-RHF driver.
//
// Follows src/df.rs:16-174 (metric_orthogonalizer, coulomb_metric,
// three_center_integrals, DfTensor::build, coulomb_exchange_rhf) and
// run_factorized_rhf (src/hf_variants/ri_df_hf.rs:160-263).  The integrals are
// the generated Head-Gordon-Pople blocks with the auxiliary shell paired with
// the exponent-0 unit function (src/df.rs:30-40).  B is kept as the tiles of its
// rows' lower triangles (df_tiles.h), formed one chunk of tile rows at a time;
// DF-J is two passes over B (HBM-bound), DF-K the matrix-core products of
// df_mfma.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <future>
#include <map>
#include <memory>
#include <numeric>
#include <string>
#include <type_traits>

#include "../../include/hfg.h"
#include "cholesky.h"
#include "df_tiles.h"
#include "engine.h"
#include "la_device.h"
#include "rhf.h"
#include "scf_host.h"

namespace hfg {

// Where a 3-index block's elements go.
struct Scatter3 {
  long long off;
  int aux_bra;        // 1: block is (P 1|a b), else (a b|P 1)
  int na, nb, np;     // component counts (kernel orientation of the orbital pair)
  int mu0, nu0, p0;   // AO offsets of first / second orbital shell and aux shell
};

// Block element -> T[P][tiled_at(i, j) - c0] of a chunk of tile rows [I0, I1)
// (cols doubles a row, c0 its first tile's position), i >= j; on the tiles of
// the diagonal the transposed element as well.  A block of one shell with
// itself writes only its a >= b elements, and elements of other tile rows
// belong to another chunk, so every entry is written once.
__global__ void k_scatter3(const Scatter3* __restrict__ d, int ntask, const double* __restrict__ blk,
                           const double* __restrict__ so, const double* __restrict__ sx, double* __restrict__ T,
                           int I0, int I1, size_t c0, size_t cols) {
  const int t = blockIdx.x;
  if (t >= ntask) return;
  const Scatter3 s = d[t];
  const int tot = s.na * s.nb * s.np;
  const bool diag = s.mu0 == s.nu0;
  for (int e = threadIdx.x; e < tot; e += blockDim.x) {
    int a, b, p;
    if (s.aux_bra) {
      p = e / (s.na * s.nb);
      const int r = e - p * s.na * s.nb;
      a = r / s.nb;
      b = r - a * s.nb;
    } else {
      a = e / (s.nb * s.np);
      const int r = e - a * s.nb * s.np;
      b = r / s.np;
      p = r - b * s.np;
    }
    if (diag && a < b) continue;
    const int mu = s.mu0 + a, nu = s.nu0 + b, P = s.p0 + p;
    const int i = mu > nu ? mu : nu, j = mu > nu ? nu : mu;
    if (i / TL < I0 || i / TL >= I1) continue;
    const double v = blk[s.off + e] * so[mu] * so[nu] * sx[P];
    double* row = T + (size_t)P * cols;
    row[tiled_at(i, j) - c0] = v;
    if (i / TL == j / TL) row[tiled_at(j, i) - c0] = v;
  }
}

// Position x of the tiled layout -> its (i, j); i or j past n: padding.
__device__ __forceinline__ void tiled_ij(size_t x, int& i, int& j) {
  const int t = (int)(x / (TL * TL)), r = (int)(x % (TL * TL));
  int I = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (I * (I + 1) / 2 > t) --I;
  while ((I + 1) * (I + 2) / 2 <= t) ++I;
  i = I * TL + r / TL;
  j = (t - I * (I + 1) / 2) * TL + r % TL;
}

// Symmetric n x n -> tiled, doubled off the diagonal tiles: sum_ij X_ij Y_ij =
// sum_x tiled2(X)_x tiled(Y)_x for symmetric X, Y.
__global__ void k_tile_sym2(const double* __restrict__ X, int n, size_t npt, double* __restrict__ Xt) {
  const size_t x = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= npt) return;
  int i, j;
  tiled_ij(x, i, j);
  Xt[x] = (i < n && j < n) ? (i / TL == j / TL ? 1.0 : 2.0) * X[(size_t)i * n + j] : 0.0;
}

// d[Q] = sum_j B[Q][j] v[j] over the nc columns of rows Q (row stride ld), four
// rows a workgroup so that each load of v serves four rows; 16-byte loads
// where rows and v are 16-byte aligned; per row a fixed-order sum (strided
// lanes, then a tree over the workgroup).  B P of DF-J (the transposed GEMV).
constexpr int RD_ROWS = 4, RD_NT = 512;
__global__ __launch_bounds__(RD_NT) void k_rowdot(const double* __restrict__ B, size_t ld, size_t nc, int rows,
                                                  const double* __restrict__ v, double* __restrict__ d) {
  __shared__ double red[RD_ROWS][RD_NT];
  const int q0 = blockIdx.x * RD_ROWS, t = threadIdx.x;
  double s[RD_ROWS];
  const double* row[RD_ROWS];
#pragma unroll
  for (int r = 0; r < RD_ROWS; ++r) {
    s[r] = 0.0;
    row[r] = B + (size_t)(q0 + r < rows ? q0 + r : q0) * ld;  // a missing row repeats the first, unused
  }
  const bool vec = (ld % 2 == 0) && ((uintptr_t)B % 16 == 0) && ((uintptr_t)v % 16 == 0);
  if (vec) {
    const size_t n2 = nc / 2;
    const double2* v2 = (const double2*)v;
    for (size_t x = t; x < n2; x += RD_NT) {
      const double2 b = v2[x];
#pragma unroll
      for (int r = 0; r < RD_ROWS; ++r) {
        const double2 a = ((const double2*)row[r])[x];
        s[r] = fma(a.x, b.x, s[r]);
        s[r] = fma(a.y, b.y, s[r]);
      }
    }
    if ((nc & 1) && t == 0)
#pragma unroll
      for (int r = 0; r < RD_ROWS; ++r) s[r] = fma(row[r][nc - 1], v[nc - 1], s[r]);
  } else {
    for (size_t x = t; x < nc; x += RD_NT) {
      const double b = v[x];
#pragma unroll
      for (int r = 0; r < RD_ROWS; ++r) s[r] = fma(row[r][x], b, s[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < RD_ROWS; ++r) red[r][t] = s[r];
  __syncthreads();
  for (int h = RD_NT / 2; h > 0; h >>= 1) {
    if (t < h)
#pragma unroll
      for (int r = 0; r < RD_ROWS; ++r) red[r][t] += red[r][t + h];
    __syncthreads();
  }
  if (t < RD_ROWS && q0 + t < rows) d[q0 + t] = red[t][0];
}

// Tiled -> symmetric n x n.
__global__ void k_untile_sym(const double* __restrict__ Xt, int n, double* __restrict__ X) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n * n) return;
  const int i = (int)(idx / n), j = (int)(idx - (size_t)i * n);
  X[idx] = Xt[i > j ? tiled_at(i, j) : tiled_at(j, i)];
}

// Tasks i < cnt of one (orbital pair class, auxiliary class) product,
// t = t0 + i = (orbital pair io, auxiliary shell ix) with ix fastest: the
// block task (kernel orientation) and its scatter record, at output offset
// i * NT.  Generated on the device: the product has ~1e8 entries for
// (H2O)32/cc-pVDZ with def2-universal-JKFIT, far too many to build and sort
// on the host.
__global__ void k_expand3(const int* __restrict__ opair, const int* __restrict__ oao_a, const int* __restrict__ oao_b,
                          const int* __restrict__ xsh, const int* __restrict__ xao, int nx, long long t0, int cnt,
                          int NT, int aux_bra, int norb_pairs, int na, int nb, int np, BlockTask* __restrict__ tasks,
                          Scatter3* __restrict__ sc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  const long long t = t0 + i;
  const int io = (int)(t / nx), ix = (int)(t - (long long)io * nx);
  const int op = opair[io], xp = norb_pairs + xsh[ix];
  const long long off = (long long)i * NT;
  tasks[i] = BlockTask{aux_bra ? xp : op, aux_bra ? op : xp, off};
  sc[i] = Scatter3{off, aux_bra, na, nb, np, oao_a[io], oao_b[io], xao[ix]};
}

// Metric block (P 1|Q 1) -> V[P][Q] and V[Q][P].
struct ScatterM {
  long long off;
  int np, nq, p0, q0;
};

__global__ void k_scatter_metric(const ScatterM* __restrict__ d, int ntask, const double* __restrict__ blk,
                                 const double* __restrict__ sx, double* __restrict__ V, int naux) {
  const int t = blockIdx.x;
  if (t >= ntask) return;
  const ScatterM s = d[t];
  for (int e = threadIdx.x; e < s.np * s.nq; e += blockDim.x) {
    const int i = e / s.nq, j = e - i * s.nq;
    const int P = s.p0 + i, Q = s.q0 + j;
    const double v = blk[s.off + e] * sx[P] * sx[Q];
    V[(size_t)P * naux + Q] = v;
    V[(size_t)Q * naux + P] = v;
  }
}

__global__ void k_axpby_fock(const double* H, const double* J, const double* K, double* F, size_t nn) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nn) F[i] = H[i] + J[i] - 0.5 * K[i];
}

struct DfEngine {
  hipStream_t stream = nullptr;
  std::unique_ptr<Blas> bl;
  int n = 0, naux = 0, rank = 0;
  std::vector<Shell> orb, aux;
  size_t npt = 0;  // doubles of one row of the tiled B
  DevBuf d_B;
  // kept between calls: P, its tiled form and the tiled J, d = B P, and the
  // exchange products' workspace
  DevBuf d_P, d_tj, d_q;
  DevBuf d_io;  // J, K and C of a call with host buffers
  ExchangeWork xwork;
  static constexpr size_t T_CHUNK = 8ull << 30;  // bytes of one column chunk of the 3-index tensor
  // HFG_DF_CHUNK: smaller ones (one tile row at least)
  static size_t chunk_bytes() {
    const char* e = std::getenv("HFG_DF_CHUNK");
    return e ? std::min<size_t>(T_CHUNK, std::strtoull(e, nullptr, 10)) : T_CHUNK;
  }

  DfEngine(const hfg_basis_view& basis, const hfg_basis_view& auxv, double cutoff) {
    if (!(cutoff > 0) || !std::isfinite(cutoff))
      throw HfgError{HFG_INVALID_INPUT, "DF metric cutoff must be finite and positive"};
    orb = group_shells(basis);
    aux = group_shells(auxv);
    n = basis.n_functions;
    naux = auxv.n_functions;
    npt = tiled_size(n);
    for (auto& s : orb)
      if (s.L > 3) throw HfgError{HFG_UNSUPPORTED, "density fitting compiled for orbital shells up to f"};
    for (auto& s : aux)
      if (s.L > 4) throw HfgError{HFG_UNSUPPORTED, "density fitting compiled for auxiliary shells up to g"};
    // HBM footprint: B at naux n(n+1)/2 doubles (and the padding of its last
    // tile row), and the 3-index tensor one chunk at a time.  Where twice
    // naux n^2 doubles fit easily so do these; beyond, they are checked.
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    const double metric = 8.0 * 2.0 * (double)naux * naux;
    const double half = 8.0 * (double)naux * ((double)n * (n + 1) / 2);
    if (4.0 * half + metric > 0.4 * (double)free_b && half + (double)T_CHUNK + metric > 0.8 * (double)free_b)
      throw HfgError{HFG_DEVICE, "DF factor B does not fit in the free device memory"};
    HIP_CHECK(hipStreamCreate(&stream));
    bl.reset(new Blas(stream));
    build(cutoff);
  }
  // Factors of the pivoted Cholesky decomposition of the AO ERIs
  // (src/cholesky.rs:44-192, cholesky.hip) in place of the fitted B, for
  // CD-HF: n_aux = rank = the number of Cholesky vectors.
  DfEngine(const hfg_basis_view& basis, double threshold, double budget, CholeskyInfo& info) {
    orb = group_shells(basis);
    n = basis.n_functions;
    npt = tiled_size(n);
    for (auto& s : orb)
      if (s.L > 2) throw HfgError{HFG_UNSUPPORTED, "Cholesky factors compiled for orbital shells up to d"};
    HIP_CHECK(hipStreamCreate(&stream));
    try {
      bl.reset(new Blas(stream));
      cholesky_factors(orb, n, stream, *bl, threshold, budget, d_B, rank, info);
    } catch (...) {
      bl.reset();
      (void)hipStreamDestroy(stream);
      stream = nullptr;
      throw;
    }
    naux = rank;
  }
  ~DfEngine() {
    bl.reset();
    if (stream) (void)hipStreamDestroy(stream);
  }

  void build(double cutoff) {
    // pair table: orbital pairs (a >= b) then auxiliary pairs (P, unit)
    std::vector<PairInfo> pairs;
    PrimPairHost pp;
    build_pairs(orb, pairs, pp);
    const int norb_pairs = (int)pairs.size();
    for (size_t p = 0; p < aux.size(); ++p) {
      PairInfo pi;
      std::memset(&pi, 0, sizeof pi);
      pi.p0 = (int)pp.size();
      append_aux_pair(aux[p], pp);
      pi.p1 = (int)pp.size();
      pi.ao_a = aux[p].ao;
      pi.ao_b = 0;
      pi.sh_a = (int)p;
      pi.sh_b = -1;
      pi.la = aux[p].L;
      pi.lb = 0;
      pairs.push_back(pi);
    }
    const size_t np = pp.size();
    DevBuf d_pp, d_pairs, d_boys, d_so, d_sx;
    d_pp.alloc(9 * np * sizeof(double));
    const std::vector<double>* cols[9] = {&pp.p, &pp.Px, &pp.Py, &pp.Pz, &pp.PAx, &pp.PAy, &pp.PAz, &pp.K, &pp.H};
    for (int c = 0; c < 9; ++c)
      HIP_CHECK(hipMemcpyAsync(d_pp.as<double>() + c * np, cols[c]->data(), np * 8, hipMemcpyHostToDevice, stream));
    std::vector<PairDev> pd(pairs.size());
    for (size_t i = 0; i < pairs.size(); ++i) {
      std::memset(&pd[i], 0, sizeof(PairDev));
      pd[i].p0 = pairs[i].p0;
      pd[i].p1 = pairs[i].p1;
      for (int k = 0; k < 3; ++k) pd[i].AB[k] = pairs[i].AB[k];
    }
    d_pairs.alloc(pd.size() * sizeof(PairDev));
    HIP_CHECK(hipMemcpyAsync(d_pairs.p, pd.data(), pd.size() * sizeof(PairDev), hipMemcpyHostToDevice, stream));
    auto tab = boys_table();
    d_boys.alloc(tab.size() * 8);
    HIP_CHECK(hipMemcpyAsync(d_boys.p, tab.data(), tab.size() * 8, hipMemcpyHostToDevice, stream));
    std::vector<double> so(n), sx(naux);
    for (auto& s : orb)
      for (size_t c = 0; c < s.scale.size(); ++c) so[s.ao + c] = s.scale[c];
    for (auto& s : aux)
      for (size_t c = 0; c < s.scale.size(); ++c) sx[s.ao + c] = s.scale[c];
    d_so.alloc(n * 8);
    d_sx.alloc(naux * 8);
    HIP_CHECK(hipMemcpyAsync(d_so.p, so.data(), n * 8, hipMemcpyHostToDevice, stream));
    HIP_CHECK(hipMemcpyAsync(d_sx.p, sx.data(), naux * 8, hipMemcpyHostToDevice, stream));
    const PrimPairs view{d_pp.as<double>(),          d_pp.as<double>() + np,     d_pp.as<double>() + 2 * np,
                         d_pp.as<double>() + 3 * np, d_pp.as<double>() + 4 * np, d_pp.as<double>() + 5 * np,
                         d_pp.as<double>() + 6 * np, d_pp.as<double>() + 7 * np, d_pp.as<double>() + 8 * np};
    auto nc = [](int L) { return (L + 1) * (L + 2) / 2; };

    // Run block tasks grouped by class in bounded batches, then scatter.
    auto run_blocks = [&](std::vector<BlockTask>& tasks, std::vector<int>& cls, auto&& scatter) {
      std::vector<size_t> ord(tasks.size());
      std::iota(ord.begin(), ord.end(), 0);
      std::stable_sort(ord.begin(), ord.end(), [&](size_t x, size_t y) { return cls[x] < cls[y]; });
      const long long budget = 1ll << 26;  // doubles per batch (512 MB)
      size_t i = 0;
      DevBuf dt, dout;
      while (i < ord.size()) {
        std::vector<BlockTask> bt;
        std::vector<int> bc;
        std::vector<size_t> which;
        long long off = 0;
        while (i < ord.size() && off < budget) {
          BlockTask t = tasks[ord[i]];
          const long long sz = t.off;  // size stashed by the caller
          t.off = off;
          bt.push_back(t);
          bc.push_back(cls[ord[i]]);
          which.push_back(ord[i]);
          off += sz;
          ++i;
        }
        dt.alloc(bt.size() * sizeof(BlockTask));
        dout.alloc(std::max<long long>(1, off) * 8);
        HIP_CHECK(hipMemcpyAsync(dt.p, bt.data(), bt.size() * sizeof(BlockTask), hipMemcpyHostToDevice, stream));
        size_t a = 0;
        while (a < bt.size()) {
          size_t b = a;
          while (b < bt.size() && bc[b] == bc[a]) ++b;
          BlockArgs args{dt.as<BlockTask>() + a, (int)(b - a), d_pairs.as<PairDev>(), view, d_boys.as<double>(),
                         dout.as<double>()};
          launch_block_class(bc[a], args, stream);
          a = b;
        }
        scatter(bt, which, dout.as<double>());
        HIP_CHECK(hipStreamSynchronize(stream));
      }
    };

    // Metric (P|Q), Q <= P.
    DevBuf d_V;
    d_V.alloc((size_t)naux * naux * 8);
    {
      std::vector<BlockTask> tasks;
      std::vector<int> cls;
      std::vector<ScatterM> sm;
      for (int p = 0; p < (int)aux.size(); ++p)
        for (int q = 0; q <= p; ++q) {
          int b = norb_pairs + p, k = norb_pairs + q;
          int pb = pair_class(aux[p].L, 0), pk = pair_class(aux[q].L, 0);
          if (pk > pb) {
            std::swap(b, k);
            std::swap(pb, pk);
          }
          const int s0 = b - norb_pairs, s1 = k - norb_pairs;
          const int n0 = nc(aux[s0].L), n1 = nc(aux[s1].L);
          tasks.push_back({b, k, (long long)n0 * n1});
          cls.push_back(quartet_class(pb, pk));
          sm.push_back({0, n0, n1, aux[s0].ao, aux[s1].ao});
        }
      DevBuf dsm;
      run_blocks(tasks, cls, [&](std::vector<BlockTask>& bt, std::vector<size_t>& which, double* blk) {
        std::vector<ScatterM> h(bt.size());
        for (size_t i = 0; i < bt.size(); ++i) {
          h[i] = sm[which[i]];
          h[i].off = bt[i].off;
        }
        dsm.alloc(h.size() * sizeof(ScatterM));
        HIP_CHECK(hipMemcpyAsync(dsm.p, h.data(), h.size() * sizeof(ScatterM), hipMemcpyHostToDevice, stream));
        hipLaunchKernelGGL(k_scatter_metric, dim3(h.size()), dim3(64), 0, stream, dsm.as<ScatterM>(), (int)h.size(),
                           blk, d_sx.as<double>(), d_V.as<double>(), naux);
        HIP_CHECK(hipGetLastError());
      });
    }
    // X = U_kept lambda^{-1/2} (src/matrix.rs:329-346 with cutoff)
    Dev dw;
    dw.alloc(naux);
    Eigh eig;
    eig.run(*bl, d_V.as<double>(), dw.p, naux);
    std::vector<double> w(naux);
    download(w.data(), dw.p, naux, stream);
    if (w[0] < -cutoff) throw HfgError{HFG_INTEGRAL, "metric has a negative eigenvalue"};
    int first = 0;
    while (first < naux && w[first] < cutoff) ++first;
    rank = naux - first;
    if (rank <= 0) throw HfgError{HFG_INTEGRAL, "metric has zero retained rank"};
    // rows of d_V's row-major view are eigenvectors; X^T rows = kept vectors / sqrt(lambda)
    std::vector<double> U((size_t)naux * naux);
    download(U.data(), d_V.as<double>(), (size_t)naux * naux, stream);
    std::vector<double> Xt((size_t)rank * naux);
    for (int r = 0; r < rank; ++r)
      for (int c = 0; c < naux; ++c) Xt[(size_t)r * naux + c] = U[(size_t)(first + r) * naux + c] / std::sqrt(w[first + r]);
    DevBuf d_Xt;
    d_Xt.alloc(Xt.size() * 8);
    HIP_CHECK(hipMemcpyAsync(d_Xt.p, Xt.data(), Xt.size() * 8, hipMemcpyHostToDevice, stream));
    d_V.free();

    // 3-index tensor (P|mu nu): every orbital pair against every auxiliary
    // shell (src/df.rs:60-78), one (pair class, auxiliary class) product at a
    // time, in batches of at most `budget` block doubles, then B = X^T T.  The
    // tensor is formed one chunk of tile rows [I0, I1) at a time -- the tiles
    // I0(I0+1)/2 .. I1(I1+1)/2 - 1 of every row -- and each chunk's columns of B
    // follow from one GEMM, so the tensor never exists whole.  A shell pair
    // whose functions lie in two chunks is evaluated for both.
    const int nt = tiles_of(n);
    const double chunk_max = (double)chunk_bytes();
    auto tiles_before = [](int I) { return (size_t)I * (I + 1) / 2; };
    std::vector<std::pair<int, int>> rows;  // chunks of tile rows
    for (int I = 0; I < nt;) {
      int e = I + 1;
      while (e < nt && 8.0 * naux * (tiles_before(e + 1) - tiles_before(I)) * (TL * TL) <= chunk_max) ++e;
      rows.push_back({I, e});
      I = e;
    }
    d_B.alloc((size_t)rank * npt * 8);
    DevBuf d_T;
    std::map<int, std::vector<int>> by_xc;  // auxiliary class -> shells
    for (int p = 0; p < (int)aux.size(); ++p) by_xc[pair_class(aux[p].L, 0)].push_back(p);
    const long long budget = 1ll << 26;
    DevBuf d_opair, d_oa, d_ob, d_xsh, d_xao, dt, ds3, dout;
    size_t cap_tasks = 0, cap_out = 0;
    for (const auto& rc : rows) {
      const size_t c0 = tiles_before(rc.first) * (TL * TL), cols = tiles_before(rc.second) * (TL * TL) - c0;
      const size_t tsz = (size_t)naux * cols;
      if (d_T.bytes < tsz * 8) d_T.alloc(tsz * 8);
      hipLaunchKernelGGL(k_zero, dim3((unsigned)((tsz + 255) / 256)), dim3(256), 0, stream, d_T.as<double>(), tsz);
      std::map<int, std::vector<int>> by_oc;  // orbital pair class -> pairs with functions in this chunk
      for (int i = 0; i < norb_pairs; ++i) {
        const PairInfo& pr = pairs[i];
        const int la = pr.ao_a + nc(pr.la) - 1, lb = pr.ao_b + nc(pr.lb) - 1;  // last functions
        if (std::max(la, lb) / TL >= rc.first && std::max(pr.ao_a, pr.ao_b) / TL < rc.second)
          by_oc[pair_class(pr.la, pr.lb)].push_back(i);
      }
      for (auto& oc : by_oc) {
        const std::vector<int>& ol = oc.second;
        std::vector<int> oa(ol.size()), ob(ol.size());
        for (size_t k = 0; k < ol.size(); ++k) {
          oa[k] = pairs[ol[k]].ao_a;
          ob[k] = pairs[ol[k]].ao_b;
        }
        d_opair.alloc(ol.size() * sizeof(int));
        d_oa.alloc(ol.size() * sizeof(int));
        d_ob.alloc(ol.size() * sizeof(int));
        HIP_CHECK(hipMemcpyAsync(d_opair.p, ol.data(), ol.size() * sizeof(int), hipMemcpyHostToDevice, stream));
        HIP_CHECK(hipMemcpyAsync(d_oa.p, oa.data(), ol.size() * sizeof(int), hipMemcpyHostToDevice, stream));
        HIP_CHECK(hipMemcpyAsync(d_ob.p, ob.data(), ol.size() * sizeof(int), hipMemcpyHostToDevice, stream));
        const PairInfo& o0 = pairs[ol[0]];
        for (auto& xc : by_xc) {
          const std::vector<int>& xl = xc.second;
          std::vector<int> xao(xl.size());
          for (size_t k = 0; k < xl.size(); ++k) xao[k] = aux[xl[k]].ao;
          d_xsh.alloc(xl.size() * sizeof(int));
          d_xao.alloc(xl.size() * sizeof(int));
          HIP_CHECK(hipMemcpyAsync(d_xsh.p, xl.data(), xl.size() * sizeof(int), hipMemcpyHostToDevice, stream));
          HIP_CHECK(hipMemcpyAsync(d_xao.p, xao.data(), xl.size() * sizeof(int), hipMemcpyHostToDevice, stream));
          const int pco = oc.first, pcx = xc.first;
          const bool aux_bra = pcx > pco;
          const int cls = aux_bra ? quartet_class(pcx, pco) : quartet_class(pco, pcx);
          const int na = nc(o0.la), nb = nc(o0.lb), np_ = nc(aux[xl[0]].L), NT = na * nb * np_;
          const long long total = (long long)ol.size() * (long long)xl.size();
          const long long chunk = std::max<long long>(1, std::min<long long>(budget / NT, 1ll << 24));
          for (long long t0 = 0; t0 < total; t0 += chunk) {
            const int cnt = (int)std::min(chunk, total - t0);
            if ((size_t)cnt > cap_tasks) {
              dt.alloc((size_t)cnt * sizeof(BlockTask));
              ds3.alloc((size_t)cnt * sizeof(Scatter3));
              cap_tasks = cnt;
            }
            if ((size_t)cnt * NT > cap_out) {
              dout.alloc((size_t)cnt * NT * 8);
              cap_out = (size_t)cnt * NT;
            }
            hipLaunchKernelGGL(k_expand3, dim3((cnt + 255) / 256), dim3(256), 0, stream, d_opair.as<int>(),
                               d_oa.as<int>(), d_ob.as<int>(), d_xsh.as<int>(), d_xao.as<int>(), (int)xl.size(), t0,
                               cnt, NT, aux_bra ? 1 : 0, norb_pairs, na, nb, np_, dt.as<BlockTask>(),
                               ds3.as<Scatter3>());
            HIP_CHECK(hipGetLastError());
            BlockArgs args{dt.as<BlockTask>(), cnt, d_pairs.as<PairDev>(), view, d_boys.as<double>(), dout.as<double>()};
            if (cls < HFG_NCLASS_ALL)
              launch_block_class(cls, args, stream);
            else  // an orbital f-p, f-d or f-f pair (never on the auxiliary side)
              launch_df_f_block(o0.la, o0.lb, aux[xl[0]].L, 0, args, stream);
            hipLaunchKernelGGL(k_scatter3, dim3(cnt), dim3(64), 0, stream, ds3.as<Scatter3>(), cnt, dout.as<double>(),
                               d_so.as<double>(), d_sx.as<double>(), d_T.as<double>(), rc.first, rc.second, c0, cols);
            HIP_CHECK(hipGetLastError());
          }
          // the lists are rewritten for the next product
          HIP_CHECK(hipStreamSynchronize(stream));
        }
      }
      // B[:, chunk] = X^T T_chunk  (rank x naux) (naux x cols)
      bl->gemm(false, false, rank, (int)cols, naux, 1.0, d_Xt.as<double>(), naux, d_T.as<double>(), (int)cols, 0.0,
               d_B.as<double>() + c0, (int)npt);
      HIP_CHECK(hipStreamSynchronize(stream));
    }
  }

  // The workspace of a jk() call (each buffer with a test of its own: an
  // allocation before it may be the one that succeeded).
  void reserve(int o, int precision) {
    if (!d_q.p) d_q.alloc((size_t)rank * 8);
    if (!d_tj.p) d_tj.alloc(2 * npt * 8);
    if (precision != 0 && !d_P.p) d_P.alloc((size_t)n * n * 8);
    df_exchange_reserve(rank, n, o, precision, precision == 0, xwork);
  }

  // J = sum_Q B_Q (B_Q . P), P = 2 C C^T; K = 2 sum_Q (B_Q C)(B_Q C)^T
  // (src/df.rs:143-173), the exchange in the given precision (df_mfma.hip), J in
  // FP64.  dC: n x o device; outputs device n x n.  FP64 exchange gives
  // B_Q . P = 2 sum A_Q . C from its tiles; otherwise it is a pass over B.
  void jk(const double* dC, int o, double* dJ, double* dK, int precision) {
    const size_t nn = (size_t)n * n;
    reserve(o, precision);
    double* dq = d_q.as<double>();
    double* tiled_p = d_tj.as<double>();
    double* tiled_j = tiled_p + npt;
    if (precision == 0) {
      df_exchange(d_B.as<double>(), npt, rank, n, dC, o, 0, dK, dq, xwork, stream);
    } else {
      double* P = d_P.as<double>();
      bl->gemm(false, true, n, n, o, 2.0, dC, o, dC, o, 0.0, P, n);
      hipLaunchKernelGGL(k_tile_sym2, dim3((unsigned)((npt + 255) / 256)), dim3(256), 0, stream, P, n, npt, tiled_p);
      HIP_CHECK(hipGetLastError());
      hipLaunchKernelGGL(k_rowdot, dim3((unsigned)((rank + RD_ROWS - 1) / RD_ROWS)), dim3(RD_NT), 0, stream,
                         d_B.as<double>(), npt, npt, rank, tiled_p, dq);
      HIP_CHECK(hipGetLastError());
      df_exchange(d_B.as<double>(), npt, rank, n, dC, o, precision, dK, nullptr, xwork, stream);
    }
    const double one = 1.0, zero = 0.0;  // column-major view of B: npt x rank
    RB_CHECK(rocblas_dgemv(bl->h, rocblas_operation_none, (rocblas_int)npt, rank, &one, d_B.as<double>(),
                           (rocblas_int)npt, dq, 1, &zero, tiled_j, 1));
    hipLaunchKernelGGL(k_untile_sym, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, stream, tiled_j, n, dJ);
    HIP_CHECK(hipGetLastError());
  }
};

// DF-RHF (src/hf_variants/ri_df_hf.rs:160-263): core-Hamiltonian guess, CDIIS
// from the second iteration, convergence on |dE|, the projected commutator
// residual and max|dP|, then one final Fock build with the new orbitals.
// make_engine builds the factors (DF: metric, 3-index and B; CD-HF: the
// Cholesky vectors) while the one-electron matrices are formed on a second
// host thread.
static int df_rhf(const hfg_basis_view* basis, const std::function<DfEngine*()>& make_engine, const double* zxyz,
                  int natom, int charge, const hfg_dfhf_options* opt, hfg_dfhf_result* res, double* p_out,
                  double* f_out, double* j_out, double* k_out) {
  using clk = std::chrono::steady_clock;
  const auto t0 = clk::now();
  std::memset(res, 0, sizeof *res);
  if (natom <= 0 || opt->max_iter <= 0 || !(opt->energy_tol > 0) || !(opt->residual_tol > 0) ||
      !(opt->density_tol > 0))
    throw HfgError{HFG_INVALID_INPUT, "DF-HF requires finite geometry and positive convergence controls"};
  if (opt->k_precision < 0 || opt->k_precision > 2 || !(opt->switch_residual > 0))
    throw HfgError{HFG_INVALID_INPUT, "DF-HF k_precision must be 0, 1 or 2 and switch_residual positive"};
  std::vector<std::array<double, 4>> atoms(natom);
  double el = -charge;
  for (int a = 0; a < natom; ++a) {
    for (int k = 0; k < 4; ++k) atoms[a][k] = zxyz[4 * a + k];
    el += atoms[a][0];
  }
  if (!(el > 0) || std::fabs(el - std::round(el)) > 1e-8 || ((long)std::lround(el)) % 2)
    throw HfgError{HFG_INVALID_INPUT, "DF-RHF requires a positive even electron count"};
  const std::vector<Shell> sh1 = group_shells(*basis);
  std::unique_ptr<DfEngine> df_p(make_engine());
  DfEngine& df = *df_p;
  const int n = df.n, no = (int)std::lround(el) / 2;
  if (n != basis->n_functions) throw HfgError{HFG_INVALID_INPUT, "DF tensor and basis differ in size"};
  hipStream_t st = df.stream;
  Blas& bl = *df.bl;
  const size_t nn = (size_t)n * n;
  double enuc = 0;
  for (int i = 0; i < natom; ++i)
    for (int j = i + 1; j < natom; ++j) {
      const double dx = atoms[i][1] - atoms[j][1], dy = atoms[i][2] - atoms[j][2], dz = atoms[i][3] - atoms[j][3];
      enuc += atoms[i][0] * atoms[j][0] / std::sqrt(dx * dx + dy * dy + dz * dz);
    }
  Dev dS, dH, dX, dTmp, dTmp2, dF, dP, dPn, dJ, dK, dC, dCo, dCn, dW, dErr, dFu;
  for (Dev* d : {&dS, &dH, &dTmp, &dTmp2, &dF, &dP, &dPn, &dJ, &dK, &dErr, &dFu}) d->alloc(nn);
  one_electron_device(sh1, n, atoms, dS.p, nullptr, nullptr, dH.p, st);  // S, H = T + V
  // canonical orthogonaliser of S (cutoff 1e-8, Cartesian)
  Eigh eig;
  int m;
  {
    Dev dw;
    dw.alloc(n);
    HIP_CHECK(hipMemcpyAsync(dTmp.p, dS.p, nn * 8, hipMemcpyDeviceToDevice, st));
    eig.run(bl, dTmp.p, dw.p, n);
    std::vector<double> w(n), U(nn);
    download(w.data(), dw.p, n, st);
    download(U.data(), dTmp.p, nn, st);
    if (w[0] < -1e-8) throw HfgError{HFG_INTEGRAL, "overlap has negative eigenvalue"};
    int first = 0;
    while (first < n && w[first] < 1e-8) ++first;
    m = n - first;
    if (no > m) throw HfgError{HFG_INVALID_INPUT, "factorized RHF occupied count exceeds overlap rank"};
    std::vector<double> X((size_t)n * m);
    for (int c = 0; c < m; ++c)
      for (int r = 0; r < n; ++r) X[(size_t)r * m + c] = U[(size_t)(first + c) * n + r] / std::sqrt(w[first + c]);
    dX.alloc((size_t)n * m);
    upload(dX.p, X.data(), (size_t)n * m, st);
  }
  dC.alloc((size_t)n * m);
  dCo.alloc((size_t)n * no);
  dCn.alloc((size_t)n * m);
  dW.alloc(m);
  const int tb = 256;
  auto grid = [&](size_t c) { return dim3((unsigned)((c + tb - 1) / tb)); };
  // C = X eigvecs(X^T F X); C_occ; P = 2 C_occ C_occ^T
  auto diag = [&](const double* F, double* C, double* P) {
    bl.gemm(false, false, n, m, n, 1.0, F, n, dX.p, m, 0.0, dTmp.p, m);
    bl.gemm(true, false, m, m, n, 1.0, dX.p, m, dTmp.p, m, 0.0, dTmp2.p, m);
    eig.run(bl, dTmp2.p, dW.p, m);
    bl.gemm(false, true, n, m, m, 1.0, dX.p, m, dTmp2.p, m, 0.0, C, m);
    bl.gemm(false, true, n, n, no, 2.0, C, m, C, m, 0.0, P, n);
  };
  auto occ_copy = [&](const double* C) {
    // C_occ (n x no): the first no columns of C (n x m), a strided device copy
    HIP_CHECK(hipMemcpy2DAsync(dCo.p, (size_t)no * 8, C, (size_t)m * 8, (size_t)no * 8, n, hipMemcpyDeviceToDevice, st));
  };
  double t_fock = 0;
  int builds = 0;
  int kprec = opt->k_precision;  // nonzero until the switch to FP64 builds
  int fp64_builds = 0;
  auto fock = [&](double* F) {
    const auto tf = clk::now();
    df.jk(dCo.p, no, dJ.p, dK.p, kprec);
    if (kprec == 0) ++fp64_builds;
    hipLaunchKernelGGL(k_axpby_fock, grid(nn), dim3(tb), 0, st, dH.p, dJ.p, dK.p, F, nn);
    HIP_CHECK(hipStreamSynchronize(st));
    t_fock += std::chrono::duration<double>(clk::now() - tf).count();
    ++builds;
  };
  auto energy = [&](const double* P, const double* F) { return 0.5 * (bl.dot(nn, P, dH.p) + bl.dot(nn, P, F)); };
  diag(dH.p, dC.p, dP.p);
  occ_copy(dC.p);
  // CDIIS histories on the device (8 slots of n x n Focks and m x m
  // errors); the error inner products are kept per slot pair, so each
  // iteration adds at most 8 dot products; the (k+1)^2 system is solved on
  // the host.
  const int MAXS = 8;
  Dev hF, hE, dCoef;
  hF.alloc(MAXS * nn);
  hE.alloc((size_t)MAXS * (size_t)m * m);
  dCoef.alloc(MAXS);
  hipLaunchKernelGGL(k_zero, grid(MAXS * nn), dim3(tb), 0, st, hF.p, MAXS * nn);
  std::vector<int> order;  // logical order (oldest first) -> slot
  std::map<std::pair<int, int>, double> edot;
  double last = INFINITY;
  const size_t mm2 = (size_t)m * m;
  for (int it = 1; it <= opt->max_iter; ++it) {
    fock(dF.p);
    const double ce = energy(dP.p, dF.p) + enuc;
    // projected commutator X^T (FPS - SPF) X
    bl.gemm(false, false, n, n, n, 1.0, dF.p, n, dP.p, n, 0.0, dTmp.p, n);
    bl.gemm(false, false, n, n, n, 1.0, dTmp.p, n, dS.p, n, 0.0, dTmp2.p, n);
    hipLaunchKernelGGL(k_antisym, grid(nn), dim3(tb), 0, st, dTmp2.p, dErr.p, n);
    bl.gemm(false, false, n, m, n, 1.0, dErr.p, n, dX.p, m, 0.0, dTmp.p, m);
    bl.gemm(true, false, m, m, n, 1.0, dX.p, m, dTmp.p, m, 0.0, dTmp2.p, m);
    const double resid = bl.amax(mm2, dTmp2.p);
    // this iteration's error, kept before diag() reuses dTmp2
    int slot;
    if ((int)order.size() >= MAXS) {
      slot = order.front();
      order.erase(order.begin());
    } else {
      slot = (int)order.size();
    }
    HIP_CHECK(hipMemcpyAsync(hE.p + (size_t)slot * mm2, dTmp2.p, mm2 * 8, hipMemcpyDeviceToDevice, st));
    if (!std::isfinite(ce) || !std::isfinite(resid)) throw HfgError{HFG_INTEGRAL, "DF-HF energy/residual became nonfinite"};
    // the density of F decides convergence only: its eigensolve waits until the
    // energy and the residual have passed (one eigensolve an iteration instead
    // of two: the solver was 60 % of a (H2O)6/cc-pVDZ solve)
    bool done = kprec == 0 && fp64_builds >= 2 && std::fabs(ce - last) <= opt->energy_tol && resid <= opt->residual_tol;
    if (done) {
      diag(dF.p, dCn.p, dPn.p);
      hipLaunchKernelGGL(k_sub, grid(nn), dim3(tb), 0, st, dPn.p, dP.p, dTmp.p, nn);
      done = bl.amax(nn, dTmp.p) <= opt->density_tol;
    }
    if (done) {
      occ_copy(dCn.p);
      fock(dF.p);
      res->total_energy = energy(dPn.p, dF.p) + enuc;
      res->iterations = it;
      res->converged = 1;
      res->n_aux = df.rank;
      res->fock_builds = builds;
      res->seconds_fock = t_fock;
      if (p_out) download(p_out, dPn.p, nn, st);
      if (f_out) download(f_out, dF.p, nn, st);
      if (j_out) download(j_out, dJ.p, nn, st);
      if (k_out) download(k_out, dK.p, nn, st);
      res->seconds_total = std::chrono::duration<double>(clk::now() - t0).count();
      return HFG_OK;
    }
    last = ce;
    if (kprec != 0 && resid < opt->switch_residual) {
      // from here on FP64 builds only; the reduced-precision Focks leave the
      // extrapolation history, this one included
      kprec = 0;
      order.clear();
      edot.clear();
      last = INFINITY;
      diag(dF.p, dC.p, dP.p);
      occ_copy(dC.p);
      continue;
    }
    HIP_CHECK(hipMemcpyAsync(hF.p + (size_t)slot * nn, dF.p, nn * 8, hipMemcpyDeviceToDevice, st));
    for (auto e = edot.begin(); e != edot.end();)
      if (e->first.first == slot || e->first.second == slot)
        e = edot.erase(e);
      else
        ++e;
    order.push_back(slot);
    for (int o : order)
      edot[{std::min(slot, o), std::max(slot, o)}] = bl.dot(mm2, hE.p + (size_t)slot * mm2, hE.p + (size_t)o * mm2);
    const double* fuse = dF.p;
    if (it >= 2 && order.size() >= 2) {
      const int k = (int)order.size();
      std::vector<double> B((size_t)(k + 1) * (k + 1), 0.0), rhs(k + 1, 0.0), c;
      for (int i = 0; i < k; ++i) {
        for (int j = 0; j < k; ++j)
          B[(size_t)i * (k + 1) + j] = edot[{std::min(order[i], order[j]), std::max(order[i], order[j])}];
        B[(size_t)i * (k + 1) + k] = B[(size_t)k * (k + 1) + i] = -1.0;
      }
      rhs[k] = -1.0;
      if (solve_small(B, rhs, k + 1, c)) {
        std::vector<double> cs(MAXS, 0.0);
        for (int i = 0; i < k; ++i) cs[order[i]] = c[i];
        upload(dCoef.p, cs.data(), MAXS, st);
        const double one = 1.0, zero = 0.0;
        RB_CHECK(rocblas_dgemv(bl.h, rocblas_operation_none, (rocblas_int)nn, MAXS, &one, hF.p, (rocblas_int)nn,
                               dCoef.p, 1, &zero, dFu.p, 1));
        fuse = dFu.p;
      }
    }
    diag(fuse, dC.p, dP.p);
    occ_copy(dC.p);
  }
  res->iterations = opt->max_iter;
  res->seconds_total = std::chrono::duration<double>(clk::now() - t0).count();
  throw HfgError{HFG_NOT_CONVERGED, "factorized RHF did not converge"};
}

}  // namespace hfg

using namespace hfg;

static int dferr(int code, const std::string& m) { return set_error(code, m); }

struct hfg_df {
  std::unique_ptr<DfEngine> e;
};

// J and K of host coefficients into host buffers, through the handle's staging
// buffer; device_ms (may be null): device time of the contraction.
static int df_host_jk(hfg_df* df, const double* cocc, int nocc, double* j, double* k, int precision,
                      double* device_ms) {
  if (!df || !cocc || !j || !k || nocc <= 0) return dferr(HFG_INVALID_INPUT, "invalid occupied coefficients for DF J/K");
  if (precision < 0 || precision > 2) return dferr(HFG_INVALID_INPUT, "precision must be 0 (FP64), 1 (FP32) or 2 (BF16x3)");
  try {
    DfEngine& e = *df->e;
    const size_t nn = (size_t)e.n * e.n, no = (size_t)e.n * nocc;
    for (size_t x = 0; x < no; ++x)
      if (!std::isfinite(cocc[x])) return dferr(HFG_INVALID_INPUT, "invalid occupied coefficients for DF J/K");
    if (e.d_io.bytes < (2 * nn + no) * 8) e.d_io.alloc((2 * nn + no) * 8);
    double *dj = e.d_io.as<double>(), *dk = dj + nn, *dc = dk + nn;
    upload(dc, cocc, no, e.stream);
    e.reserve(nocc, precision);  // not between the events
    hipEvent_t ev[2] = {};
    struct Events {
      hipEvent_t* ev;
      ~Events() {
        for (int x = 0; x < 2; ++x)
          if (ev[x]) (void)hipEventDestroy(ev[x]);
      }
    } events{ev};
    if (device_ms) {
      for (hipEvent_t& x : ev) HIP_CHECK(hipEventCreate(&x));
      HIP_CHECK(hipEventRecord(ev[0], e.stream));
    }
    e.jk(dc, nocc, dj, dk, precision);
    if (device_ms) HIP_CHECK(hipEventRecord(ev[1], e.stream));
    download(j, dj, nn, e.stream);
    download(k, dk, nn, e.stream);
    if (device_ms) {
      float ms = 0;
      HIP_CHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
      *device_ms = ms;
    }
    return HFG_OK;
  } catch (HfgError& ex) {
    return dferr(ex.code, ex.msg);
  }
}

extern "C" {

int hfg_df_build(const hfg_basis_view* basis, const hfg_basis_view* aux, double metric_cutoff, hfg_df** out) {
  if (!basis || !aux || !out) return dferr(HFG_INVALID_INPUT, "null argument");
  try {
    auto* h = new hfg_df;
    try {
      h->e.reset(new DfEngine(*basis, *aux, metric_cutoff));
    } catch (...) {
      delete h;
      throw;
    }
    *out = h;
    return HFG_OK;
  } catch (HfgError& e) {
    return dferr(e.code, e.msg);
  } catch (std::exception& e) {
    return dferr(HFG_DEVICE, e.what());
  }
}

void hfg_df_destroy(hfg_df* df) { delete df; }

int hfg_df_info(const hfg_df* df, int64_t* n, int64_t* naux, int64_t* rank) {
  if (!df) return dferr(HFG_INVALID_INPUT, "null handle");
  if (n) *n = df->e->n;
  if (naux) *naux = df->e->naux;
  if (rank) *rank = df->e->rank;
  return HFG_OK;
}

int hfg_df_jk(hfg_df* df, const double* cocc, int nocc, double* j, double* k) {
  return df_host_jk(df, cocc, nocc, j, k, 0, nullptr);
}

int hfg_df_jk_ex(hfg_df* df, const double* cocc, int nocc, double* j, double* k, int precision,
                 double* device_ms) {
  return df_host_jk(df, cocc, nocc, j, k, precision, device_ms);
}

int hfg_df_rhf(const hfg_basis_view* basis, const hfg_basis_view* aux, const double* zxyz, int natom, int charge,
               const hfg_dfhf_options* opt, hfg_dfhf_result* res, double* p_out, double* f_out, double* j_out,
               double* k_out) {
  if (!basis || !aux || !zxyz || !opt || !res) return dferr(HFG_INVALID_INPUT, "null argument");
  try {
    if (!(opt->metric_cutoff > 0)) throw HfgError{HFG_INVALID_INPUT, "DF metric cutoff must be finite and positive"};
    return df_rhf(
        basis, [&] { return new DfEngine(*basis, *aux, opt->metric_cutoff); }, zxyz, natom, charge, opt, res, p_out,
        f_out, j_out, k_out);
  } catch (HfgError& e) {
    return dferr(e.code, e.msg);
  }
}

int hfg_cd_build(const hfg_basis_view* basis, double threshold, double budget_bytes, hfg_df** out, hfg_cd_info* info,
                 int32_t* pivots, int32_t max_pivots) {
  if (!basis || !out) return dferr(HFG_INVALID_INPUT, "null argument");
  try {
    CholeskyInfo ci;
    auto* d = new hfg_df;
    try {
      d->e.reset(new DfEngine(*basis, threshold, budget_bytes, ci));
    } catch (...) {
      delete d;
      throw;
    }
    if (info) {
      info->rank = ci.rank;
      info->max_residual = ci.max_residual;
    }
    if (pivots)
      for (int k = 0; k < ci.rank && k < max_pivots; ++k) pivots[k] = ci.pivots[k];
    *out = d;
    return HFG_OK;
  } catch (HfgError& e) {
    return dferr(e.code, e.msg);
  }
}

int hfg_cd_rhf(const hfg_basis_view* basis, const double* zxyz, int natom, int charge, double delta,
               double budget_bytes, const hfg_dfhf_options* opt, hfg_dfhf_result* res, hfg_cd_info* info,
               double* p_out, double* f_out) {
  if (!basis || !zxyz || !opt || !res) return dferr(HFG_INVALID_INPUT, "null argument");
  try {
    CholeskyInfo ci;
    const int st = df_rhf(
        basis, [&] { return new DfEngine(*basis, delta, budget_bytes, ci); }, zxyz, natom, charge, opt, res, p_out,
        f_out, nullptr, nullptr);
    if (info) {
      info->rank = ci.rank;
      info->max_residual = ci.max_residual;
    }
    return st;
  } catch (HfgError& e) {
    return dferr(e.code, e.msg);
  }
}

}  // extern "C"
