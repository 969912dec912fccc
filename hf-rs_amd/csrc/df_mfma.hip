// df_mfma.hip -- the exchange products of DF-K on the matrix cores, straight
// from the tiled factor: A_Q = B_Q C for every auxiliary row Q, and
// K = 2 sum_Q A_Q A_Q^T = 2 X X^T (coulomb_exchange_rhf's loop over Q,
// src/df.rs:143-173, as one symmetric rank-L update with L = rank n_occ), in
// FP64, in FP32 and with operands split into two BF16 parts.
//
// The tiled factor (df_tiles.h): row Q holds the lower triangle of B_Q in
// 32 x 32 tiles.  Both kernels work on panels of 16-byte chunks: a panel row
// is one matrix row (or column) of a contraction step, CH chunks of 16 bytes
// (2 FP64, 4 FP32 or 8 BF16 values), and a lane's operand is one chunk, read
// from LDS with one 16-byte load: in a group of MFMAs lane l takes row l % 16
// and the chunk of its lane group l / 16, so that FP64 and FP32 chunks feed
// two and four consecutive MFMAs (the order of the contraction index within
// a step is free as long as both operands share it).  Chunks are stored at
// c ^ swz(row), which spreads the 16 rows that one operand reads over all LDS
// banks without padding.
//
// MFMA layouts (lane l): operand row or column l % 16, contraction index from
// l / 16; the FP64 16x16x4 result has column l % 16 and row l / 16 + 4 r in
// register r, the FP32 and BF16 16x16 forms row 4 (l / 16) + r.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "df_tiles.h"
#include "engine.h"

namespace hfg {
namespace {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

template <class To, class From>
__device__ __forceinline__ To as_bits(From x) {
  static_assert(sizeof(To) == sizeof(From), "same size");
  return __builtin_bit_cast(To, x);
}

// FP32 pair -> BF16 pair (round to nearest even) and back
__device__ __forceinline__ unsigned bf16_pair(f2 v) { return as_bits<unsigned>(__builtin_convertvector(v, b2)); }
__device__ __forceinline__ f2 bf16_values(unsigned p) {
  return f2{__uint_as_float(p << 16), __uint_as_float(p & 0xffff0000u)};
}

// The three arithmetics.  CH: 16-byte chunks of a panel row of the A = B C
// step (32 contraction values); acc: accumulator of one 16 x 16 block; X: an
// element of the exchange product's operand; XK: contraction values in its
// 256-byte step; P: a partial sum; SUB: MFMAs of a chunk pair.
struct F64 {
  static constexpr int CH = 16, XK = 32, SUB = 2;
  typedef d4 acc;
  typedef double X, P;
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
struct F32 {
  static constexpr int CH = 8, XK = 64, SUB = 4;
  typedef f4 acc;
  typedef float X, P;
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
// x = hi + lo, hi = bf16(x), lo = bf16(x - hi); hi hi + hi lo + lo hi summed in
// FP32.  Panel rows hold the hi chunks, then the lo chunks; the exchange
// operand alternates 64 hi and the same 64 lo values.
struct BF16x3 {
  static constexpr int CH = 8, XK = 64, SUB = 3;
  typedef f4 acc;
  typedef unsigned short X;
  typedef float P;
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

template <int CH>
__device__ __forceinline__ int swz(int row) {
  return CH == 16 ? row & 15 : (row >> 1) & 7;
}

// Sub-step s of one chunk pair: FP64 and FP32 take one value of each chunk, BF16
// one of the products hi hi, hi lo, lo hi.
__device__ __forceinline__ void mac(F64, int s, d4& acc, u4 a, u4, u4 b, u4) {
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(as_bits<d2>(a)[s], as_bits<d2>(b)[s], acc, 0, 0, 0);
}
__device__ __forceinline__ void mac(F32, int s, f4& acc, u4 a, u4, u4 b, u4) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(as_bits<f4>(a)[s], as_bits<f4>(b)[s], acc, 0, 0, 0);
}
__device__ __forceinline__ void mac(BF16x3, int s, f4& acc, u4 ah, u4 al, u4 bh, u4 bl) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bits<b8>(s == 2 ? al : ah), as_bits<b8>(s == 1 ? bl : bh), acc, 0,
                                                0, 0);
}

// A 256-thread workgroup's four waves over a tile of 64 rows and NB 16-column
// blocks: 2 x 2 waves of 32 rows and NB / 2 blocks (7 chunks read for 10 chunk
// products at NB = 10), 4 x 1 of 16 rows where NB is odd.
template <int NB>
struct Waves {
  static constexpr int M = NB % 2 ? 4 : 2, N = 4 / M, RA = 4 / M, NBW = NB / N;
};
constexpr int ROWS = 64, NT = 256;

// One step over LDS panels of CHP chunks a row (rows of A at ra + 16 x, columns
// of B at cb + 16 b): the chunks of the step, or for BF16 the hi chunks of its
// first half with the lo chunks of its second.
template <class T, int CHP, int RA, int NBW>
__device__ __forceinline__ void step(typename T::acc (&acc)[RA][NBW], const u4* A, const u4* B, int ra, int cb,
                                     int lane) {
  const int rq = lane & 15, g = lane >> 4;
  constexpr bool BF = T::SUB == 3;
  constexpr int GROUPS = BF ? CHP / 8 : CHP / 4;  // groups of four chunks (BF16: of hi chunks)
#pragma unroll
  for (int t = 0; t < GROUPS; ++t) {
    u4 a[RA], al[RA], v[NBW], vl[NBW];
#pragma unroll
    for (int x = 0; x < RA; ++x) {
      const int r = ra + 16 * x + rq;
      a[x] = A[r * CHP + ((4 * t + g) ^ swz<CHP>(r))];
      al[x] = BF ? A[r * CHP + ((CHP / 2 + 4 * t + g) ^ swz<CHP>(r))] : a[x];
    }
#pragma unroll
    for (int b = 0; b < NBW; ++b) {
      const int r = cb + 16 * b + rq;
      v[b] = B[r * CHP + ((4 * t + g) ^ swz<CHP>(r))];
      vl[b] = BF ? B[r * CHP + ((CHP / 2 + 4 * t + g) ^ swz<CHP>(r))] : v[b];
    }
#pragma unroll
    for (int s = 0; s < T::SUB; ++s)
#pragma unroll
      for (int b = 0; b < NBW; ++b)
#pragma unroll
        for (int x = 0; x < RA; ++x) mac(T(), s, acc[x][b], a[x], al[x], v[b], vl[b]);
  }
}

// ---- A = B C

// The pair kp of a panel row's 32 values (FP64 2 kp, 2 kp + 1) -> LDS.
__device__ __forceinline__ void put2(F64, u4* L, int r, int kp, d2 v) { L[r * 16 + (kp ^ swz<16>(r))] = as_bits<u4>(v); }
__device__ __forceinline__ void put2(F32, u4* L, int r, int kp, d2 v) {
  ((f2*)(L + r * 8 + ((kp >> 1) ^ swz<8>(r))))[kp & 1] = f2{(float)v.x, (float)v.y};
}
__device__ __forceinline__ void split2(d2 v, unsigned& h, unsigned& l) {
  const f2 x = {(float)v.x, (float)v.y};
  h = bf16_pair(x);
  const f2 y = bf16_values(h);
  l = bf16_pair(f2{x.x - y.x, x.y - y.y});
}
__device__ __forceinline__ void put2(BF16x3, u4* L, int r, int kp, d2 v) {
  unsigned h, l;
  split2(v, h, l);
  ((unsigned*)(L + r * 8 + ((kp >> 2) ^ swz<8>(r))))[kp & 3] = h;
  ((unsigned*)(L + r * 8 + ((4 + (kp >> 2)) ^ swz<8>(r))))[kp & 3] = l;
}

// C (n x o, FP64) -> panels [column tile it][k tile kb][column < an][CH chunks],
// zero past (n, o): what one workgroup's step reads is one contiguous run.
template <class T>
__global__ __launch_bounds__(256) void k_pack_c(const double* __restrict__ C, int n, int o, int nt, int an, int gy,
                                                u4* __restrict__ out) {
  const int e = blockIdx.x * 256 + threadIdx.x;  // (it, kb, pair of values, column)
  if (e >= gy * nt * an * 16) return;
  const int col = e % an, kp = (e / an) & 15, rest = e / an / 16;
  const int k = rest % nt * TL + 2 * kp, i = (rest / nt) * an + col;
  d2 v = {0.0, 0.0};
  if (i < o) {
    if (k < n) v.x = C[(size_t)k * o + i];
    if (k + 1 < n) v.y = C[(size_t)(k + 1) * o + i];
  }
  u4* row = out + (size_t)(rest * an + col) * T::CH;
  if constexpr (T::CH == 16) {
    row[kp] = as_bits<u4>(v);
  } else if constexpr (T::SUB == 4) {
    ((f2*)row)[kp] = f2{(float)v.x, (float)v.y};
  } else {
    unsigned h, l;
    split2(v, h, l);
    ((unsigned*)row)[kp] = h;
    ((unsigned*)row)[16 + kp] = l;
  }
}

// The exchange operand X (n x L, contraction index k = Q o + i) is stored step by
// step: the n rows' 256 bytes of a step are one run, so that what a workgroup
// reads of a step, and what it writes of a row Q, lies in a few pages.  (Row by
// row, with rows of 5 MB, every panel row was in a page of its own.)
__device__ __forceinline__ void put_x(double* X, int n, int m, long long k, double v) {
  X[((k >> 5) * n + m) * 32 + (k & 31)] = v;
}
__device__ __forceinline__ void put_x(float* X, int n, int m, long long k, float v) {
  X[((k >> 6) * n + m) * 64 + (k & 63)] = v;
}
__device__ __forceinline__ void put_x(unsigned short* X, int n, int m, long long k, float v) {
  const unsigned h = bf16_pair(f2{v, 0.f}) & 0xffffu;
  const unsigned l = bf16_pair(f2{v - __uint_as_float(h << 16), 0.f}) & 0xffffu;
  unsigned short* p = X + ((k >> 6) * n + m) * 128 + (k & 63);
  p[0] = (unsigned short)h;
  p[64] = (unsigned short)l;
}

// A workgroup takes two 32-row blocks -- consecutive (Q, tile row I) pairs, so
// that no row is padding beyond the last tile of a row Q -- against NB x 16
// columns of C.  Step kb multiplies tile (I, kb) of each block, read along its
// rows where kb <= I and as the transpose of tile (kb, I) above the diagonal,
// with the C panel of that tile column.  A block is staged by a pair of waves as
// pairs of consecutive contraction values, converted (and split) once: along
// its rows, one 16-byte load of 64 consecutive pairs a wave; as a transpose,
// two 8-byte loads along two of its rows.
// One LDS buffer and two barriers a step, the next step's panels on their way
// to registers meanwhile: half the LDS of a second buffer lets two workgroups
// share a CU, and while one stages, the other multiplies.  (One 512-thread
// workgroup of 128 rows and two buffers: the two waves of a SIMD move in step
// and the matrix cores idle while both wait, 75 % busy.)
// Measured, n 800, rank 4256, 160 columns: FP64 16.3 ms (53 TFLOP/s of tiles
// computed; the rocBLAS product, the permute and the pass for B . P that it
// replaces 26.3 ms), split BF16 4.3 ms (5 TB/s of B tiles requested; three
// rocBLAS products, the permute and the split 9.6 ms).  n 1200, rank 6384, 240
// columns, FP64: 83.6 ms (57 TFLOP/s; 160-column tiles of packed rows 114 ms).
// n 500, rank 2660, 100 columns, FP32: 1.6 ms (rocBLAS and the permute 3.1 ms).
// The FP64 form is bound by the matrix cores (72 TFLOP/s by themselves, 68
// with the step's LDS traffic), the BF16 form by the traffic of B.
// Output: X[m][Q o + i] (put_x), and with part the sums of A_Q . C over each
// wave's rows of a block (B_Q . P without another pass over B).
// Workgroups are dealt round-robin to the 8 XCDs by linear id; id 8 j + x takes
// item off(x) + j, so that each XCD runs a contiguous run of blocks and the
// two reads of a tile (as itself and transposed) meet in its L2.
template <class T, int NB>
__global__ __launch_bounds__(NT) void k_bc_tiles(const double* __restrict__ Bt, size_t npt, int nt, int rank, int n,
                                                 const u4* __restrict__ Cp, const double* __restrict__ C, int o,
                                                 typename T::X* __restrict__ X, double* __restrict__ part, int gy,
                                                 int total) {
  typedef Waves<NB> W;
  constexpr int CH = T::CH, AN = 16 * NB, RA = W::RA, NBW = W::NBW;
  constexpr int NC = (AN * CH + NT - 1) / NT;  // C chunks a thread stages
  __shared__ u4 lds[(ROWS + AN) * CH];
  u4* lc = lds + ROWS * CH;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int per = total / 8, rem = total % 8, xcd = blockIdx.x % 8;
  const int item = xcd * per + min(xcd, rem) + blockIdx.x / 8;
  const int it = item % gy;
  const int nblk = rank * nt;
  const int f0 = (item / gy) * 2;
  // the block this thread stages, by pairs of waves
  const int fs = min(f0 + (w >> 1), nblk - 1);
  const int qs = fs / nt, is = fs - qs * nt;
  const double* Bq = Bt + (size_t)qs * npt;
  const int h = w & 1;
  constexpr bool even = AN * CH % NT == 0;
  d2 bv[4];
  u4 cv[NC];
  auto load = [&](int kb) {
    const double* tile = Bq + tile_index(is, kb) * (TL * TL);
    if (kb <= is) {
#pragma unroll
      for (int c = 0; c < 4; ++c) bv[c] = ((const d2*)tile)[256 * h + 64 * c + lane];
    } else {
      const double* p = tile + (16 * h + 2 * (lane >> 5)) * TL + (lane & 31);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        bv[c].x = p[4 * c * TL];
        bv[c].y = p[(4 * c + 1) * TL];
      }
    }
    const u4* cp = Cp + ((size_t)it * nt + kb) * AN * CH;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (even || t + NT * c < AN * CH) cv[c] = cp[NT * c + t];
  };
  auto store = [&](int kb) {
    const bool low = kb <= is;
    const int r = 32 * (w >> 1) + (low ? 16 * h + (lane >> 4) : lane & 31), kp = low ? lane & 15 : 8 * h + (lane >> 5);
#pragma unroll
    for (int c = 0; c < 4; ++c) put2(T(), lds, low ? r + 4 * c : r, low ? kp : kp + 2 * c, bv[c]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = t + NT * c, col = e / CH;
      if (even || e < AN * CH) lc[col * CH + ((e % CH) ^ swz<CH>(col))] = cv[c];
    }
  };
  typename T::acc acc[RA][NBW] = {};
  const int wm = w % W::M, wn = w / W::M;
  load(0);
  for (int kb = 0; kb < nt; ++kb) {
    if (kb) __syncthreads();  // every wave has read the last step's panels
    store(kb);
    if (kb + 1 < nt) load(kb + 1);
    __syncthreads();
    step<T, CH>(acc, lds, lc, 16 * RA * wm, 16 * NBW * wn, lane);
  }
  // a wave's rows lie in one block
  const int fb = f0 + 16 * RA * wm / 32;
  if (fb >= nblk) return;
  const int q = fb / nt, m0 = (fb - q * nt) * TL + 16 * RA * wm % 32;
  double sum = 0.0;
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < NBW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * a + T::row(lane, r), i = it * AN + 16 * (NBW * wn + b) + (lane & 15);
        if (m < n && i < o) {
          put_x(X, n, m, (long long)q * o + i, acc[a][b][r]);
          if (part) sum += (double)acc[a][b][r] * C[(size_t)m * o + i];
        }
      }
  if (part) {  // two waves to a block: two halves of its rows, or of the columns
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) sum += __shfl_xor(sum, s, 64);
    if (lane == 0) part[((size_t)fb * gy + it) * 2 + (RA == 2 ? wn : wm & 1)] = sum;
  }
}

// gamma[Q] = alpha * (the np sums of row Q, in order)
__global__ void k_part_reduce(const double* __restrict__ part, int np, int rank, double alpha,
                              double* __restrict__ gamma) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= rank) return;
  double s = 0.0;
  for (int j = 0; j < np; ++j) s += part[(size_t)q * np + j];
  gamma[q] = alpha * s;
}

// Zero the exchange operand's values k in [L, L + w) of its last step.
template <class X>
__global__ void k_zero_tail(X* __restrict__ x, int n, long long L, int w) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < w * n) put_x(x, n, e / w, L + e % w, 0);
}

// Column tile of the A = B C kernel: gy tiles of nb 16-column blocks, the
// least padded width plus one block's worth a tile for what a tile costs
// beside its columns.
void column_tiles(int o, int& nb, int& gy) {
  const int all = (o + 15) / 16;
  int best = INT32_MAX;
  for (int g = (all + 9) / 10; g <= (all + 9) / 10 + 2; ++g) {
    const int b = (all + g - 1) / g;
    if (g * (b + 1) < best) {
      best = g * (b + 1);
      nb = b;
      gy = g;
    }
  }
}

template <class T, int NB>
void launch_bc(int nb, const double* Bt, size_t npt, int nt, int rank, int n, const u4* Cp, const double* C, int o,
               typename T::X* X, double* part, int gy, hipStream_t st) {
  if constexpr (NB > 0) {
    if (nb != NB) {
      launch_bc<T, NB - 1>(nb, Bt, npt, nt, rank, n, Cp, C, o, X, part, gy, st);
      return;
    }
    const long long total = ((long long)rank * nt + 1) / 2 * gy;
    if (total > INT32_MAX) throw HfgError{HFG_UNSUPPORTED, "tiled A = B C: too many tiles for one launch"};
    hipLaunchKernelGGL((k_bc_tiles<T, NB>), dim3((unsigned)total), dim3(NT), 0, st, Bt, npt, nt, rank, n, Cp, C, o, X,
                       part, gy, (int)total);
    HIP_CHECK(hipGetLastError());
  }
}

// ---- K = 2 X X^T

// The exchange product's output tiles: 64 rows against the columns from the
// tile's own first row on (only the upper triangle is computed: 346k elements at
// n = 800 for the 320k needed, where 128 x 128 tiles took 459k), in the fewest column tiles of at most ten 16-column blocks, all within one block
// of each other.
struct SyrkTile {
  int i0, j0, nb;  // first row, first column, 16-column blocks
};
__host__ __device__ inline int syrk_tiles(int n, int r) { return ((n - ROWS * r + 15) / 16 + 9) / 10; }
__device__ inline SyrkTile syrk_tile(int n, int x) {
  for (int r = 0;; ++r) {
    const int c = syrk_tiles(n, r);
    if (x < c) {
      const int all = (n - ROWS * r + 15) / 16, base = all / c, more = all % c;
      return SyrkTile{ROWS * r, ROWS * r + 16 * (base * x + min(x, more)), base + (x < more ? 1 : 0)};
    }
    x -= c;
  }
}

// One tile over steps [k0, k1) of 256 bytes a row, staged as the A = B C kernel
// stages its own.  Measured for the sizes above: FP64 7.9 ms (59 TFLOP/s of
// tiles computed) against 10.9 ms for 128 x 128 tiles, 42.3 against 54.1 ms at
// n 1200; FP32 0.8 ms against 2.6; split BF16 2.2 ms against 6.0 (three rocBLAS
// products of the whole square).
template <class T, int NB>
__device__ __forceinline__ void syrk_body(const typename T::X* __restrict__ X, int n, int i0, int j0, int k0, int k1,
                                          u4* lds, typename T::P* __restrict__ out) {
  typedef Waves<NB> W;
  constexpr int RA = W::RA, NBW = W::NBW, PR = ROWS + 16 * NB;  // panel rows
  constexpr int NC = PR * 16 / NT;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = w % W::M, wn = w / W::M;
  const u4* src[NC];
  u4 v[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int r = (t >> 4) + 16 * c;
    const int row = min(r < ROWS ? i0 + r : j0 + r - ROWS, n - 1);  // rows past n repeat the last: never stored
    src[c] = (const u4*)X + ((size_t)k0 * n + row) * 16 + (t & 15);
  }
  auto load = [&] {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      v[c] = *src[c];
      src[c] += (size_t)n * 16;
    }
  };
  typename T::acc acc[RA][NBW] = {};
  if (k0 < k1) load();
  for (int k = k0; k < k1; ++k) {
    if (k > k0) __syncthreads();
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int r = (t >> 4) + 16 * c;
      lds[r * 16 + ((t & 15) ^ swz<16>(r))] = v[c];
    }
    if (k + 1 < k1) load();
    __syncthreads();
    step<T, 16>(acc, lds, lds + ROWS * 16, 16 * RA * wm, 16 * NBW * wn, lane);
  }
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < NBW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + 16 * (RA * wm + a) + T::row(lane, r), j = j0 + 16 * (NBW * wn + b) + (lane & 15);
        if (i <= j && j < n) out[(size_t)i * n + j] = acc[a][b][r];
      }
}

template <class T, int NB>
__device__ __forceinline__ void syrk_pick(const SyrkTile& tl, const typename T::X* X, int n, int k0, int k1, u4* lds,
                                          typename T::P* out) {
  if constexpr (NB > 0) {
    if (tl.nb != NB)
      syrk_pick<T, NB - 1>(tl, X, n, k0, k1, lds, out);
    else
      syrk_body<T, NB>(X, n, tl.i0, tl.j0, k0, k1, lds, out);
  }
}

// Workgroup (tile, slice): the tiles alone are far too few for 256 CUs, so the
// contraction is cut into S slices (a multiple of 8) whose partial tiles a
// second kernel sums in a fixed order.  Linear id 8 j + x runs on XCD x; it
// takes slice x + 8 (j / tiles), so that every tile of a slice reads the
// slice's panels through one L2.
template <class T>
__global__ __launch_bounds__(NT) void k_syrk(const typename T::X* __restrict__ X, int n, int steps, int S, int tiles,
                                             typename T::P* __restrict__ part) {
  __shared__ u4 lds[(ROWS + 160) * 16];
  const int j = blockIdx.x / 8, s = blockIdx.x % 8 + 8 * (j / tiles);
  const SyrkTile tl = syrk_tile(n, j % tiles);
  const int k0 = (int)((long long)steps * s / S), k1 = (int)((long long)steps * (s + 1) / S);
  syrk_pick<T, 10>(tl, X, n, k0, k1, lds, part + (size_t)s * n * n);
}

// K[i][j] = K[j][i] = alpha sum_s part[s][i][j], i <= j, by 8 x 32 blocks (both
// writes along rows of a 32 x 32 tile's parts); the sums are in FP64 whatever the
// partials are, in order, eight loads on their way at a time: one element a
// thread, since at n = 150 there are 45 blocks of 192 slices (11.5 us; 222 us with
// 32 x 32 blocks and one load at a time).
template <class P>
__global__ __launch_bounds__(256) void k_syrk_reduce(const P* __restrict__ part, int S, int n, double alpha,
                                                     double* __restrict__ K) {
  __shared__ double tile[8][33];
  const int i0 = blockIdx.y * 8, j0 = blockIdx.x * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
  if (i0 >= j0 + 32) return;
  const size_t nn = (size_t)n * n;
  const int i = i0 + y, j = j0 + x;
  double v = 0.0;
  if (i <= j && j < n) {
    const P* p = part + (size_t)i * n + j;
    int s = 0;
    for (; s + 8 <= S; s += 8) {
      P u[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) u[k] = p[(s + k) * nn];
#pragma unroll
      for (int k = 0; k < 8; ++k) v += (double)u[k];
    }
    for (; s < S; ++s) v += (double)p[s * nn];
    v *= alpha;
    K[(size_t)i * n + j] = v;
  }
  tile[y][x] = v;
  __syncthreads();
  const int c = threadIdx.x & 7, r = threadIdx.x >> 3;  // K[j0 + r][i0 + c]
  if (i0 + c < j0 + r && j0 + r < n) K[(size_t)(j0 + r) * n + i0 + c] = tile[c][r];
}

// The launches' shapes, with the workspace for them.
struct Shape {
  int nt, nb = 0, gy = 0, tiles = 0;
  long long L, steps, S;
};
template <class T>
Shape k_reserve(int rank, int n, int o, bool gamma, ExchangeWork& w) {
  Shape h;
  h.nt = tiles_of(n);
  column_tiles(o, h.nb, h.gy);
  h.L = (long long)rank * o;
  h.steps = (h.L + T::XK - 1) / T::XK;
  if (h.steps > INT32_MAX) throw HfgError{HFG_UNSUPPORTED, "DF exchange: contraction index out of range"};
  for (int r = 0; ROWS * r < n; ++r) h.tiles += syrk_tiles(n, r);
  // slices: about six rounds of the chip's 512 workgroups (two a CU), at least
  // four steps each, a multiple of 8
  h.S = (3072 + h.tiles - 1) / h.tiles;
  h.S = std::min(h.S, std::max<long long>(1, h.steps / 4));
  h.S = (h.S + 7) / 8 * 8;
  w.c.grow((size_t)h.gy * h.nt * 16 * h.nb * T::CH * 16);
  w.x.grow((size_t)h.steps * n * 256);
  w.part.grow((size_t)h.S * n * n * sizeof(typename T::P));
  if (gamma) w.sums.grow((size_t)rank * h.nt * 2 * h.gy * 8);
  return h;
}

template <class T>
void k_from_tiles(const double* Bt, size_t npt, int rank, int n, const double* C, int o, double* K, double* gamma,
                  ExchangeWork& w, hipStream_t st) {
  typedef typename T::X X;
  typedef typename T::P P;
  const Shape h = k_reserve<T>(rank, n, o, gamma != nullptr, w);
  const int nt = h.nt, nb = h.nb, gy = h.gy, tiles = h.tiles, an = 16 * nb;
  const long long L = h.L, steps = h.steps, S = h.S;
  double* part = gamma ? w.sums.template as<double>() : nullptr;
  u4* cp = w.c.template as<u4>();
  X* x = w.x.template as<X>();
  hipLaunchKernelGGL(k_pack_c<T>, dim3((unsigned)((gy * nt * an * 16 + 255) / 256)), dim3(256), 0, st, C, n, o, nt, an,
                     gy, cp);
  HIP_CHECK(hipGetLastError());
  if (const int w = (int)(steps * T::XK - L)) {
    hipLaunchKernelGGL(k_zero_tail<X>, dim3((unsigned)((w * n + 255) / 256)), dim3(256), 0, st, x, n, L, w);
    HIP_CHECK(hipGetLastError());
  }
  launch_bc<T, 10>(nb, Bt, npt, nt, rank, n, cp, C, o, x, part, gy, st);
  if (gamma) {
    hipLaunchKernelGGL(k_part_reduce, dim3((unsigned)((rank + 255) / 256)), dim3(256), 0, st, part, nt * 2 * gy, rank,
                       2.0, gamma);
    HIP_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(k_syrk<T>, dim3((unsigned)(tiles * S)), dim3(NT), 0, st, x, n, (int)steps, (int)S, tiles,
                     w.part.template as<P>());
  HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_syrk_reduce<P>, dim3((unsigned)((n + 31) / 32), (unsigned)((n + 7) / 8)), dim3(256), 0, st,
                     w.part.template as<P>(), (int)S, n, 2.0, K);
  HIP_CHECK(hipGetLastError());
}

}  // namespace

void df_exchange_reserve(int rank, int n, int o, int precision, bool gamma, ExchangeWork& w) {
  if (precision == 0)
    k_reserve<F64>(rank, n, o, gamma, w);
  else if (precision == 1)
    k_reserve<F32>(rank, n, o, gamma, w);
  else
    k_reserve<BF16x3>(rank, n, o, gamma, w);
}

void df_exchange(const double* Bt, size_t npt, int rank, int n, const double* C, int o, int precision, double* K,
                 double* gamma, ExchangeWork& w, hipStream_t st) {
  if (precision == 0)
    k_from_tiles<F64>(Bt, npt, rank, n, C, o, K, gamma, w, st);
  else if (precision == 1)
    k_from_tiles<F32>(Bt, npt, rank, n, C, o, K, nullptr, w, st);
  else
    k_from_tiles<BF16x3>(Bt, npt, rank, n, C, o, K, nullptr, w, st);
}

}  // namespace hfg
