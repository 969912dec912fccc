// grad.hip -- analytic RHF nuclear gradient: compute_gradient_from_density
// (src/gradient.rs:287-512) for a density P and an energy-weighted density W.
//
// Two-electron part on the device.  dE2/dX = 1/2 sum over ordered AO
// quadruples of d(mu nu|lam sig)/dX * G, G = P_mn P_ls - 1/4 (P_ml P_ns +
// P_ms P_nl); over unique shell quartets with their degeneracy.  A
// basis-function derivative is d/dA_t phi_a = 2 alpha phi_{a+1_t} - a_t
// phi_{a-1_t} (src/gradient.rs:71-113), so the derivatives of a quartet with
// respect to the centres of three of its shells come from ordinary ERI blocks
// of "raised" shells (L+1, radial coefficients times 2 alpha) and "lowered"
// shells (L-1); the fourth centre follows from translational invariance.  The
// block kernels evaluate those blocks (the fp and fd raised pairs are the extra
// classes of gen/eri_grad.inc); one kernel then contracts every block with G
// and adds the quartet's forces to per-workgroup LDS sums of the atoms' forces.
//
// One-electron terms on the device (onee_dev.hip); the nuclear repulsion
// (src/gradient.rs:220-243) on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <map>
#include <type_traits>
#include <vector>

#include "../../include/hfg.h"
#include "engine.h"
#include "eri_device.h"
#include "la_device.h"
#include "rhf.h"
#include "scf_host.h"
#include "wide_scratch.h"

namespace hfg {
#include "gen/eri_grad.inc"

namespace {

// One thread per block, as the engine's block kernels, each block written
// straight to its place: at up to 2,160 doubles a private copy would only add
// scratch.
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(64) void k_gblock(BlockArgs a) {
  __shared__ double boys[BoysSlice<false>::size];
  load_boys_slice<LA + LB + LC + LD>(a.boys, boys);
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.ntask) return;
  const BlockTask bt = a.tasks[t];
  const PairDev& pb = a.pairs[bt.bra];
  const PairDev& pk = a.pairs[bt.ket];
  eri_block<LA, LB, LC, LD>(a.pp, pb.p0, pb.p1, a.pp, pk.p0, pk.p1 - pk.p0, 1, pb.AB, pk.AB, boys, a.out + bt.off);
}

template <int LA, int LB, int LC, int LD>
void launch_gblock(const BlockArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((k_gblock<LA, LB, LC, LD>), dim3((a.ntask + 63) / 64), dim3(64), 0, s, a);
}

// Rank of a pair class (la >= lb) in the block kernels' order: the orbital
// pairs, the auxiliary f-s and g-s pairs, then the gradient's f-p and f-d.
int pair_rank(int la, int lb) {
  static const int R[5][3] = {{0, -1, -1}, {1, 2, -1}, {3, 4, 5}, {6, 8, 9}, {7, -1, -1}};
  return (la < 0 || la > 4 || lb < 0 || lb > 2) ? -1 : R[la][lb];
}

// Launch of block class (l1 l2 | l3 l4) (kernel orientation, first pair of
// rank >= second).
void launch_any_block(int l1, int l2, int l3, int l4, const BlockArgs& a, hipStream_t s) {
  int idx = 0;
#define X(p, q, r, u)                                              \
  if (p == l1 && q == l2 && r == l3 && u == l4) {                    \
    launch_block_class(idx, a, s);                                   \
    return;                                                          \
  }                                                                  \
  ++idx;
  HFG_FOR_EACH_CLASS_ALL(X)
#undef X
#define X(p, q, r, u)                                          \
  if (p == l1 && q == l2 && r == l3 && u == l4) {              \
    auto launch = [&](hipStream_t on) {                        \
      launch_gblock<p, q, r, u>(a, on);                        \
      HIP_CHECK(hipGetLastError());                            \
    };                                                         \
    if (p + q + r + u == 9) /* (fd|dd) */                      \
      launch_wide(s, launch);                                  \
    else                                                       \
      launch(s);                                               \
    return;                                                    \
  }
  HFG_FOR_EACH_GRAD_CLASS(X)
#undef X
  throw HfgError{HFG_UNSUPPORTED, "no gradient block kernel for class (" + std::to_string(l1) + std::to_string(l2) +
                                      "|" + std::to_string(l3) + std::to_string(l4) + ")"};
}

// Cartesian components in hf-rs order (as the generator's cart()): exponents
// per (L, index) and index per (L, lx, ly).
struct CartTab {
  signed char e[4][10][3];
  signed char idx[4][4][4];
};
constexpr CartTab make_cart() {
  CartTab t{};
  for (int L = 0; L < 4; ++L) {
    int k = 0;
    if (L == 2) {
      const int d[6][3] = {{2, 0, 0}, {0, 2, 0}, {0, 0, 2}, {1, 1, 0}, {1, 0, 1}, {0, 1, 1}};
      for (; k < 6; ++k)
        for (int c = 0; c < 3; ++c) t.e[L][k][c] = (signed char)d[k][c];
    } else {
      for (int lx = L; lx >= 0; --lx)
        for (int ly = L - lx; ly >= 0; --ly, ++k) {
          t.e[L][k][0] = (signed char)lx;
          t.e[L][k][1] = (signed char)ly;
          t.e[L][k][2] = (signed char)(L - lx - ly);
        }
    }
    for (int i = 0; i < k; ++i) t.idx[L][t.e[L][i][0]][t.e[L][i][1]] = (signed char)i;
  }
  return t;
}
const CartTab g_cart = make_cart();

// A shell pair as the gradient's kernels read it: AO offsets and atoms of its
// two shells (kernel orientation), and its four derivative pairs' entries in
// the pair table (raised and lowered first shell, raised and lowered second;
// -1: none).
struct GPair {
  int ao[2], atom[2], d[4];
};

// The quartets of a pair of pair classes (la lb|lc ld) all have the same
// derivative blocks: at most six (raised and lowered A, B and C).
constexpr int MAX_BLK = 6;
struct GBlocks {
  int n;
  int ket[MAX_BLK];    // the derivative pair is the ket's (of C), else the bra's
  int slot[MAX_BLK];   // which of the pair's derivative pairs
  int first[MAX_BLK];  // the block stores the derivative pair first
  int size[MAX_BLK];
  long long base[MAX_BLK];  // of the block's values in the block buffer
  long long task[MAX_BLK];  // and of its tasks in the task buffer
};

// Quartet t of a class: rows are the bra class's pairs, each with the prefix of
// the ket class's pairs (both sorted by Schwarz bound) that passes the test;
// pre[i] .. pre[i + 1] - 1 are row i's.  Writes the quartet's pairs and its block
// tasks.  One thread a quartet: on the host, listing the quartets of C8H18/6-31G
// and copying the lists took 130 of 162 ms; these launches take 0.1 ms, and the
// whole gradient 16.6.
__global__ __launch_bounds__(256) void k_grad_tasks(const int* __restrict__ bra, const int* __restrict__ ket,
                                                    const long long* __restrict__ pre, int rows, long long t0, int nq,
                                                    const GPair* __restrict__ pairs, GBlocks g,
                                                    int2* __restrict__ quartets, BlockTask* __restrict__ tasks) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= nq) return;
  const long long t = t0 + q;
  int lo = 0, hi = rows - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int ij = bra[lo], kl = ket[t - pre[lo]];
  quartets[q] = int2{ij, kl};
  for (int b = 0; b < g.n; ++b) {
    const int dp = pairs[g.ket[b] ? kl : ij].d[g.slot[b]], other = g.ket[b] ? ij : kl;
    tasks[g.task[b] + q] =
        BlockTask{g.first[b] ? dp : other, g.first[b] ? other : dp, g.base[b] + (long long)q * g.size[b]};
  }
}

// One term of a quartet's force: element e of block b times coef contributes,
// with G of the quartet's own element o, to one derivative (x, y or z of A, B
// or C; the entries are grouped by it).
struct GEntry {
  unsigned short o, e;
  short b, coef;
};
struct GContract {
  int dim[4];       // components of A, B, C, D
  int end[9];       // entries up to derivative s (A x, y, z, B x, ...)
  GBlocks blocks;
};

// Forces of every quartet: G = P_mn P_ls - 1/4 (P_ml P_ns + P_ms P_nl) with the
// component factors, each of its elements once into LDS, then the entries, the
// nine sums and d/dD = -(d/dA + d/dB + d/dC).  GL lanes a quartet, chosen by
// the class's entries (9 for (ss|ss), 1,197 for (pp|pp)): a wave per quartet
// had 3 of 64 lanes at work on an (ss|ss) block and formed G again for every
// entry.  The longest lists (17,000 of (dd|dd)) and short launches take a whole
// workgroup a quartet: a wave's walk through them is what a launch then lasts.
// Atoms' forces are summed in LDS per workgroup, then added to grad
// (natom x 3).  w = 1/2 x the quartet's degeneracy.
template <int GL>
__global__ __launch_bounds__(256) void k_grad_contract(const int2* __restrict__ quartets, int nq,
                                                       const GPair* __restrict__ pairs, GContract c,
                                                       const GEntry* __restrict__ entries,
                                                       const double* __restrict__ blk, const double* __restrict__ P,
                                                       const double* __restrict__ scale, int n, int natom,
                                                       double* __restrict__ grad) {
  extern __shared__ double lds[];
  const int nt = c.dim[0] * c.dim[1] * c.dim[2] * c.dim[3];
  double* acc = lds;                                           // natom x 3
  double* G = lds + 3 * natom + (size_t)(threadIdx.x / GL) * nt;  // this group's quartet
  for (int i = threadIdx.x; i < 3 * natom; i += blockDim.x) acc[i] = 0.0;
  const int lane = threadIdx.x % GL, per = 256 / GL;
  const int rounds = (nq + per * gridDim.x - 1) / (per * gridDim.x);
  for (int r = 0; r < rounds; ++r) {
    const int q = (r * gridDim.x + blockIdx.x) * per + threadIdx.x / GL;
    const bool on = q < nq;
    const int2 ids = quartets[on ? q : 0];
    const GPair A = pairs[ids.x], C = pairs[ids.y];
    __syncthreads();  // the last round's G is read, and acc is clear
    if (on)
      for (int o = lane; o < nt; o += GL) {
        int x = o;
        const int d = x % c.dim[3];
        x /= c.dim[3];
        const int cc = x % c.dim[2];
        x /= c.dim[2];
        const int b = x % c.dim[1], a = x / c.dim[1];
        const size_t mu = A.ao[0] + a, nu = A.ao[1] + b, la = C.ao[0] + cc, si = C.ao[1] + d;
        G[o] = (P[mu * n + nu] * P[la * n + si] -
                0.25 * (P[mu * n + la] * P[nu * n + si] + P[mu * n + si] * P[nu * n + la])) *
               scale[mu] * scale[nu] * scale[la] * scale[si];
      }
    __syncthreads();
    double s[9];
    int k = lane;
#pragma unroll
    for (int x = 0; x < 9; ++x) {
      double v = 0.0;
      if (on)
        for (; k < c.end[x]; k += GL) {
          const GEntry e = entries[k];
          v += e.coef * blk[c.blocks.base[e.b] + (long long)q * c.blocks.size[e.b] + e.e] * G[e.o];
        }
#pragma unroll
      for (int o = (GL < 64 ? GL : 64) / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o, GL < 64 ? GL : 64);
      s[x] = v;
    }
    if (on && lane % 64 == 0) {  // each wave's part, where a quartet has four
      double w = 0.5;
      if (A.ao[0] != A.ao[1]) w *= 2.0;
      if (C.ao[0] != C.ao[1]) w *= 2.0;
      if (ids.x != ids.y) w *= 2.0;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        atomicAdd(&acc[3 * A.atom[0] + t], w * s[t]);
        atomicAdd(&acc[3 * A.atom[1] + t], w * s[3 + t]);
        atomicAdd(&acc[3 * C.atom[0] + t], w * s[6 + t]);
        atomicAdd(&acc[3 * C.atom[1] + t], -w * (s[t] + s[3 + t] + s[6 + t]));
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 3 * natom; i += blockDim.x)
    if (acc[i] != 0.0) atomicAdd(&grad[i], acc[i]);
}

Shell raised(const Shell& s) {
  Shell r = s;
  r.L = s.L + 1;
  for (int k = 0; k < s.K; ++k) r.r[k] = s.r[k] * 2.0 * s.e[k];
  return r;
}
Shell lowered(const Shell& s) {
  Shell r = s;
  r.L = s.L - 1;
  return r;
}

// The blocks and force terms of class (L0 L1|L2 L3).  A block's derivative pair
// is stored with the higher L first, and the pair of higher rank first in the
// block.
struct GClass {
  GBlocks blocks = {};
  int key[MAX_BLK][4];  // the blocks' own classes
  GContract c = {};
  std::vector<GEntry> entries;
};
GClass gradient_class(const int (&L)[4]) {
  GClass k;
  std::vector<GEntry> by[9];
  auto add = [&](int X, bool up) {  // raised or lowered shell X (0, 1 or 2)
    const int l = L[X] + (up ? 1 : -1), side = X / 2, Y = X ^ 1;  // Y: X's partner
    if (l < 0) return;
    const int b = k.blocks.n++;
    // X before Y unless its L is now the lower one; first shells stay first at equal L
    const bool x_first = X % 2 ? l > L[Y] : l >= L[Y];
    const int d0 = x_first ? X : Y, d1 = x_first ? Y : X, o0 = side ? 0 : 2, o1 = o0 + 1;
    auto len = [&](int s) { return s == X ? l : L[s]; };
    const bool first = pair_rank(len(d0), len(d1)) >= pair_rank(L[o0], L[o1]);
    const int sh[4] = {first ? d0 : o0, first ? d1 : o1, first ? o0 : d0, first ? o1 : d1};
    int dim[4], size = 1;
    for (int p = 0; p < 4; ++p) {
      k.key[b][p] = len(sh[p]);
      dim[p] = ncart(len(sh[p]));
      size *= dim[p];
    }
    k.blocks.ket[b] = side;
    k.blocks.slot[b] = 2 * (X % 2) + (up ? 0 : 1);
    k.blocks.first[b] = first;
    k.blocks.size[b] = size;
    for (int e = 0; e < size; ++e) {
      int o[4], r = e;
      for (int p = 3; p >= 0; --p) {
        o[sh[p]] = r % dim[p];
        r /= dim[p];
      }
      const signed char* ex = g_cart.e[l][o[X]];
      for (int t = 0; t < 3; ++t) {
        int ee[3] = {ex[0], ex[1], ex[2]};
        if (up && ee[t] == 0) continue;
        const int coef = up ? 1 : -(ee[t] + 1);
        ee[t] += up ? -1 : 1;
        int own[4] = {o[0], o[1], o[2], o[3]};
        own[X] = g_cart.idx[L[X]][ee[0]][ee[1]];
        const int at = ((own[0] * ncart(L[1]) + own[1]) * ncart(L[2]) + own[2]) * ncart(L[3]) + own[3];
        by[3 * X + t].push_back(GEntry{(unsigned short)at, (unsigned short)e, (short)b, (short)coef});
      }
    }
  };
  for (int X = 0; X < 3; ++X)
    for (bool up : {true, false}) add(X, up);
  for (int p = 0; p < 4; ++p) k.c.dim[p] = ncart(L[p]);
  for (int x = 0; x < 9; ++x) {
    k.entries.insert(k.entries.end(), by[x].begin(), by[x].end());
    k.c.end[x] = (int)k.entries.size();
  }
  return k;
}

template <int GL>
void launch_contract(const GContract& c, const int2* quartets, int nq, const GPair* pairs, const GEntry* entries,
                     const double* blk, const double* P, const double* scale, int n, int natom, double* grad,
                     hipStream_t st) {
  const size_t lds = (3 * (size_t)natom + (size_t)(256 / GL) * c.dim[0] * c.dim[1] * c.dim[2] * c.dim[3]) * 8;
  if (lds > 65536) {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    raise_dynamic_lds((const void*)k_grad_contract<GL>, dev, lds);
  }
  const int blocks = std::min(2048, (nq + 256 / GL - 1) / (256 / GL));
  hipLaunchKernelGGL(k_grad_contract<GL>, dim3(blocks), dim3(256), lds, st, quartets, nq, pairs, c, entries, blk, P,
                     scale, n, natom, grad);
  HIP_CHECK(hipGetLastError());
}

// Parts of one device allocation, each from a multiple of 256 bytes, and the host
// side of those that are copied there in one piece.  add and place come before
// reserve (no host side), all before upload.
class Slab {
 public:
  size_t place(size_t bytes) {
    const size_t o = reserve(bytes);
    host_.resize(size_);
    return o;
  }
  void put(size_t o, const void* h, size_t bytes) {
    if (bytes) std::memcpy(host_.data() + o, h, bytes);
  }
  size_t add(const void* h, size_t bytes) {
    const size_t o = place(bytes);
    put(o, h, bytes);
    return o;
  }
  size_t reserve(size_t bytes) {
    const size_t o = size_;
    size_ += (bytes + 255) / 256 * 256;
    return o;
  }
  void upload(hipStream_t st) {
    dev_.alloc(size_);
    if (!host_.empty()) HIP_CHECK(hipMemcpyAsync(dev_.p, host_.data(), host_.size(), hipMemcpyHostToDevice, st));
  }
  template <class T>
  T* at(size_t o) const {
    return (T*)((char*)dev_.p + o);
  }

 private:
  std::vector<char> host_;
  size_t size_ = 0;
  DevBuf dev_;
};

}  // namespace

// Nuclear gradient (natom x 3, host) of the engine's molecule for the device
// density dP and energy-weighted density dW (row-major n x n), on stream st.
// Reads the engine's tables only, so it may run beside builds of other
// molecules.
void rhf_gradient_device(Engine& e, const std::vector<std::array<double, 4>>& atoms, const double* dP,
                         const double* dW, double* grad, hipStream_t st) {
  const int n = e.n, na = (int)atoms.size();
  std::vector<double> g((size_t)3 * na, 0.0);
  for (const Shell& s : e.shells)
    if (s.atom < 0 || s.atom >= na) throw HfgError{HFG_INVALID_INPUT, "basis atom index outside the geometry"};
  // nuclear repulsion (src/gradient.rs:220-243)
  for (int a = 0; a < na; ++a)
    for (int b = 0; b < na; ++b) {
      if (a == b) continue;
      double d[3], r2 = 0;
      for (int k = 0; k < 3; ++k) {
        d[k] = atoms[a][1 + k] - atoms[b][1 + k];
        r2 += d[k] * d[k];
      }
      const double f = atoms[a][0] * atoms[b][0] / (r2 * std::sqrt(r2));
      for (int k = 0; k < 3; ++k) g[3 * a + k] -= f * d[k];
    }
  const std::vector<Shell>& sh = e.shells;
  const std::vector<double>& sc = e.ao_scale;
  // ---- two-electron part on the device
  // pair table: the engine's pairs, then the derivative pairs (raised and
  // lowered first shell, raised and lowered second), each with the higher L
  // first; filled in parallel at offsets fixed in advance
  const size_t npair = e.pairs.size();
  std::vector<GPair> gp(npair);
  std::vector<size_t> off(4 * npair + 1, e.pp.size());
  std::vector<int> slots;  // pair * 4 + slot of the derivative pairs, in table order
  for (size_t i = 0; i < npair; ++i) {
    const PairInfo& p = e.pairs[i];
    GPair& g_ = gp[i];
    g_ = GPair{{p.ao_a, p.ao_b}, {sh[p.sh_a].atom, sh[p.sh_b].atom}, {-1, -1, -1, -1}};
    const size_t prims = (size_t)sh[p.sh_a].K * sh[p.sh_b].K;
    for (int s = 0; s < 4; ++s) {
      const bool have = s == 0 || s == 2 || (s == 1 ? p.la : p.lb) > 0;
      if (have) {
        g_.d[s] = (int)(npair + slots.size());
        slots.push_back((int)(4 * i + s));
      }
      off[4 * i + s + 1] = off[4 * i + s] + (have ? prims : 0);
    }
  }
  PrimPairHost pp = e.pp;
  std::vector<double>* grow[9] = {&pp.p, &pp.Px, &pp.Py, &pp.Pz, &pp.PAx, &pp.PAy, &pp.PAz, &pp.K, &pp.H};
  for (auto* c : grow) c->resize(off.back());
  std::vector<PairDev> pd(npair + slots.size());
  for (size_t i = 0; i < npair; ++i) {
    const PairInfo& p = e.pairs[i];
    std::memset(&pd[i], 0, sizeof(PairDev));
    pd[i].p0 = p.p0;
    pd[i].p1 = p.p1;
    for (int k = 0; k < 3; ++k) pd[i].AB[k] = p.AB[k];
  }
#pragma omp parallel for schedule(dynamic, 64)
  for (long x = 0; x < (long)slots.size(); ++x) {
    const PairInfo& p = e.pairs[slots[x] / 4];
    const int s = slots[x] % 4;
    const Shell &A = sh[p.sh_a], &B = sh[p.sh_b];
    const Shell D = s == 0 ? raised(A) : s == 1 ? lowered(A) : s == 2 ? raised(B) : lowered(B);
    const bool d_first = s < 2 ? D.L >= B.L : D.L > A.L;
    const Shell &X = s < 2 ? (d_first ? D : B) : (d_first ? D : A), &Y = s < 2 ? (d_first ? B : D) : (d_first ? A : D);
    PrimPairHost one;
    append_pair(X, Y, one);
    const size_t at = off[slots[x]];
    const std::vector<double>* from[9] = {&one.p, &one.Px, &one.Py, &one.Pz, &one.PAx, &one.PAy, &one.PAz, &one.K, &one.H};
    for (int c = 0; c < 9; ++c) std::copy(from[c]->begin(), from[c]->end(), grow[c]->begin() + at);
    PairDev& d = pd[npair + x];
    std::memset(&d, 0, sizeof d);
    d.p0 = (int)at;
    d.p1 = (int)(at + one.size());
    for (int k = 0; k < 3; ++k) d.AB[k] = X.c[k] - Y.c[k];
  }
  const size_t npp = pp.size();
  // one allocation and one copy for the tables (a small molecule's call is a few
  // dozen launches of 10 to 50 us: sixteen copies and eleven allocations showed)
  Slab tables;
  const size_t o_pp = tables.place(9 * npp * sizeof(double));
  for (int c = 0; c < 9; ++c) tables.put(o_pp + c * npp * sizeof(double), grow[c]->data(), npp * sizeof(double));
  const size_t o_pd = tables.add(pd.data(), pd.size() * sizeof(PairDev)), o_scale = tables.add(sc.data(), (size_t)n * 8),
               o_grad = tables.place((size_t)3 * na * 8);
  tables.upload(st);
  double* d_grad = tables.at<double>(o_grad);
  const PairDev* d_pd = tables.at<PairDev>(o_pd);
  const double* d_scale = tables.at<double>(o_scale);
  hipLaunchKernelGGL(k_zero, dim3((3 * na + 255) / 256), dim3(256), 0, st, d_grad, (size_t)3 * na);
  // ---- one-electron terms on the device (onee_dev.hip)
  onee_gradient_device(sh, n, atoms, dP, dW, d_grad, st);
  const double* b = tables.at<double>(o_pp);
  const PrimPairs view{b, b + npp, b + 2 * npp, b + 3 * npp, b + 4 * npp, b + 5 * npp, b + 6 * npp, b + 7 * npp,
                       b + 8 * npp};
  // Quartets by pair of pair classes: both classes' pairs sorted by Schwarz
  // bound, so that the ket pairs of a row that pass the test are a prefix (and
  // of one class with itself the rows' earlier pairs).  The lists are written on
  // the device, in batches of at most BUDGET block doubles.
  const size_t lds = (size_t)3 * na * sizeof(double);
  if (lds > 60000) throw HfgError{HFG_UNSUPPORTED, "gradient: too many atoms for the per-workgroup force sums"};
  std::array<std::vector<int>, 6> cls;  // pairs by class, largest bound first
  for (size_t i = 0; i < npair; ++i) cls[pair_class(e.pairs[i].la, e.pairs[i].lb)].push_back((int)i);
  std::vector<int> order;
  std::array<size_t, 6> at = {};
  for (int c = 0; c < 6; ++c) {
    std::stable_sort(cls[c].begin(), cls[c].end(), [&](int x, int y) { return e.Q[x] > e.Q[y]; });
    at[c] = order.size();
    order.insert(order.end(), cls[c].begin(), cls[c].end());
  }
  struct Job {
    int cb, ck;
    size_t pre;  // of its rows' prefix sums
    long long total;
    GClass g;
    size_t entries;
  };
  std::vector<Job> jobs;
  std::vector<long long> pre;
  std::vector<GEntry> entries;
  for (int cb = 0; cb < 6; ++cb)
    for (int ck = 0; ck <= cb; ++ck) {
      if (cls[cb].empty() || cls[ck].empty()) continue;
      Job j{cb, ck, pre.size(), 0, {}, entries.size()};
      size_t hi = cls[ck].size();  // falls with the row's bound
      for (size_t i = 0; i < cls[cb].size(); ++i) {
        pre.push_back(j.total);
        while (hi > 0 && !(e.Q[cls[cb][i]] * e.Q[cls[ck][hi - 1]] > e.screen)) --hi;
        j.total += (long long)(cb == ck ? std::min(hi, i + 1) : hi);
      }
      pre.push_back(j.total);
      if (j.total == 0) continue;
      const PairInfo &x = e.pairs[cls[cb][0]], &y = e.pairs[cls[ck][0]];
      j.g = gradient_class({x.la, x.lb, y.la, y.lb});
      entries.insert(entries.end(), j.g.entries.begin(), j.g.entries.end());
      jobs.push_back(std::move(j));
    }
  Slab lists;
  const size_t o_gp = lists.add(gp.data(), gp.size() * sizeof(GPair)),
               o_order = lists.add(order.data(), order.size() * sizeof(int)),
               o_pre = lists.add(pre.data(), pre.size() * sizeof(long long)),
               o_ent = lists.add(entries.data(), entries.size() * sizeof(GEntry));
  // Rounds of at most 128 MB of blocks (they are read back from the last-level
  // cache): chunks of one class's quartets, as many as fit, so that a small
  // molecule's blocks of one kernel go out in one launch whatever classes they
  // are for (water/6-31G*: 16.8 ms with a round per class).
  constexpr long long BUDGET = 1ll << 24;
  struct Chunk {
    const Job* job;
    long long t0;
    int nq;
    size_t q0;  // its quartets' place in the round
    GBlocks g;
  };
  struct Launch {
    const int* key;
    size_t task0;
    int count;
  };
  struct Round {
    std::vector<Chunk> chunks;
    std::vector<Launch> launches;
    size_t quartets = 0, tasks = 0;
    long long doubles = 0;
  };
  std::vector<Round> rounds(1);
  for (const Job& j : jobs) {
    long long size = 0;
    for (int b = 0; b < j.g.blocks.n; ++b) size += j.g.blocks.size[b];
    for (long long t0 = 0; t0 < j.total;) {
      Round* r = &rounds.back();
      long long room = std::min<long long>((BUDGET - r->doubles) / size, (1 << 19) - (long long)r->quartets);
      if (room <= 0 && !r->chunks.empty()) {
        rounds.emplace_back();
        r = &rounds.back();
        room = std::min<long long>(BUDGET / size, 1 << 19);
      }
      const int nq = (int)std::min(j.total - t0, std::max<long long>(1, room));
      Chunk c{&j, t0, nq, r->quartets, j.g.blocks};
      for (int b = 0; b < c.g.n; ++b) {
        c.g.base[b] = r->doubles;
        r->doubles += (long long)nq * c.g.size[b];
      }
      r->quartets += nq;
      r->chunks.push_back(c);
      t0 += nq;
    }
  }
  size_t cap_q = 0, cap_t = 0, cap_b = 0;
  for (Round& r : rounds) {
    std::map<std::array<int, 4>, std::vector<std::pair<Chunk*, int>>> by_key;
    for (Chunk& c : r.chunks)
      for (int b = 0; b < c.g.n; ++b) {
        const int* k = c.job->g.key[b];
        by_key[{k[0], k[1], k[2], k[3]}].push_back({&c, b});
      }
    for (auto& k : by_key) {
      Launch l{k.second[0].first->job->g.key[k.second[0].second], r.tasks, 0};
      for (auto& cb : k.second) {
        cb.first->g.task[cb.second] = (long long)r.tasks;
        r.tasks += cb.first->nq;
        l.count += cb.first->nq;
      }
      r.launches.push_back(l);
    }
    cap_q = std::max(cap_q, r.quartets);
    cap_t = std::max(cap_t, r.tasks);
    cap_b = std::max(cap_b, (size_t)r.doubles);
  }
  const size_t o_q = lists.reserve(cap_q * sizeof(int2)), o_tasks = lists.reserve(cap_t * sizeof(BlockTask)),
               o_blk = lists.reserve(cap_b * 8);
  lists.upload(st);
  const GPair* d_gp = lists.at<GPair>(o_gp);
  const int* d_order = lists.at<int>(o_order);
  const long long* d_pre = lists.at<long long>(o_pre);
  const GEntry* d_ent = lists.at<GEntry>(o_ent);
  int2* d_q = lists.at<int2>(o_q);
  BlockTask* d_tasks = lists.at<BlockTask>(o_tasks);
  double* d_blk = lists.at<double>(o_blk);
  for (const Round& r : rounds) {
    for (const Chunk& c : r.chunks) {
      hipLaunchKernelGGL(k_grad_tasks, dim3((c.nq + 255) / 256), dim3(256), 0, st,
                         d_order + at[c.job->cb], d_order + at[c.job->ck], d_pre + c.job->pre,
                         (int)cls[c.job->cb].size(), c.t0, c.nq, d_gp, c.g, d_q + c.q0, d_tasks);
      HIP_CHECK(hipGetLastError());
    }
    for (const Launch& l : r.launches) {
      BlockArgs args{d_tasks + l.task0, l.count, d_pd, view, e.d_boys.as<double>(), d_blk};
      launch_any_block(l.key[0], l.key[1], l.key[2], l.key[3], args, st);
    }
    for (const Chunk& c : r.chunks) {
      GContract gc = c.job->g.c;
      gc.blocks = c.g;
      auto contract = [&](auto gl) {
        launch_contract<decltype(gl)::value>(gc, d_q + c.q0, c.nq, d_gp, d_ent + c.job->entries, d_blk, dP,
                                             d_scale, n, na, d_grad, st);
      };
      const size_t terms = c.job->g.entries.size();
      // a workgroup a quartet while that leaves CUs idle, or for lists that keep its
      // 256 lanes busy (and whose G, 10 KB of (dd|dd), limits the quartets on a CU)
      if (terms <= 32)
        contract(std::integral_constant<int, 4>());
      else if (terms <= 256)
        contract(std::integral_constant<int, 16>());
      else if (terms <= 4096 && c.nq > 512)
        contract(std::integral_constant<int, 64>());
      else
        contract(std::integral_constant<int, 256>());
    }
  }
  std::vector<double> g2((size_t)3 * na);
  download(g2.data(), d_grad, g2.size(), st);
  for (size_t x = 0; x < g.size(); ++x) grad[x] = g[x] + g2[x];
}

// The same for host P and W, on the engine's stream.
void rhf_gradient(Engine& e, const std::vector<std::array<double, 4>>& atoms, const double* P, const double* W,
                  double* grad) {
  const size_t nn = (size_t)e.n * e.n;
  DevBuf d;
  d.alloc(2 * nn * sizeof(double));
  HIP_CHECK(hipMemcpyAsync(d.as<double>(), P, nn * 8, hipMemcpyHostToDevice, e.stream));
  HIP_CHECK(hipMemcpyAsync(d.as<double>() + nn, W, nn * 8, hipMemcpyHostToDevice, e.stream));
  rhf_gradient_device(e, atoms, d.as<double>(), d.as<double>() + nn, grad, e.stream);
}

}  // namespace hfg
