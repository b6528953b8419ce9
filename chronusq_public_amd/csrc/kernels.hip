// HIP kernels of the direct J/K build for gfx950 (MI355X): screening and
// quartet-list construction, and the matrix transforms around the ERI
// kernels.
//
// Reference algorithm: GTODirectTPIContraction::directScaffoldNew
// (include/particleintegrals/contract/direct.hpp:1412-2123).  The quartet set,
// its screening and the degeneracy factors follow the reference loop; ERIs
// are evaluated by Rys quadrature in Cartesian form and the density /
// result matrices are carried in the Cartesian AO basis (T X T^T and
// T^T A T around the build), which is the same algebra as transforming every
// integral batch to pure functions.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cart_coef.hpp"
#include "kernels.hpp"
#include "screen.hpp"

namespace cqx {

namespace {

__device__ __forceinline__ void atomic_add(double *p, double v) { unsafeAtomicAdd(p, v); }

// ---------------------------------------------------------------------------
// Screening: quartet candidates (bra i, ket j) after the Schwarz pre-cut,
// tested with the reference's Schwarz x shell-block-norm rule in reference
// labels (direct.hpp:1689-1789); survivors appended to a list with the mask
// of contractions that pass their own separated screen.
// ---------------------------------------------------------------------------
constexpr int kListThreads = 1024;

// Candidates [base, base + 1024) of one list: the block's bra range is found
// once, each thread tests one candidate, survivors are appended block-wide
// (the waves' counts meet in LDS and one thread reserves the block's slots
// with one atomic per list), and the Ka Kb Kc Kd sums of the chunk are
// reduced in LDS to one atomic per list.
__device__ __forceinline__ void list_chunk(const ListLaunch &a, long long base) {
  constexpr int NW = kListThreads / 64;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __shared__ int s_lo, s_hi;
  __shared__ unsigned s_cnt[2][NW];
  __shared__ unsigned long long s_start[2][NW];
  __shared__ double s_ps[2][NW];
  // candidates of the list: counted on the device for a list sized in
  // advance (ncand is then its capacity)
  const long long ncand = a.ncand_dev ? min(*a.ncand_dev - a.cand_base, a.ncand) : a.ncand;
  if (base >= ncand) return;  // uniform across the block
  const long long t = base + threadIdx.x;
  bool pass = false;
  unsigned mask = 0;
  int bi = 0, kj = 0;
  double qq = 0.0, kk4 = 0.0;
  // the block's candidates span bra indices [s_lo, s_hi]: two searches per
  // block, then each thread searches that (usually short) range
  if (threadIdx.x == 0 || threadIdx.x == blockDim.x - 1) {
    const long long tt =
        a.cand_base + (threadIdx.x == 0 ? base : min(base + (long long)blockDim.x, ncand) - 1);
    int lo = 0, hi = a.nbra - 1;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (a.cand_off[mid] <= tt) lo = mid; else hi = mid - 1;
    }
    if (threadIdx.x == 0) s_lo = lo; else s_hi = lo;
  }
  __syncthreads();
  const int blo = s_lo, bhi = s_hi;
  if (t < ncand) {
    // bra index: last i with cand_off[i] <= t (absolute candidate index)
    const long long ta = a.cand_base + t;
    int lo = blo, hi = bhi;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (a.cand_off[mid] <= ta) lo = mid; else hi = mid - 1;
    }
    bi = lo;
    kj = a.ket_lo[bi] + (int)(ta - a.cand_off[lo]);
    const PairScr P = a.bra[bi], Q = a.ket[kj];
    qq = P.Q * Q.Q;
    kk4 = (double)P.kk * (double)Q.kk;
    const double *pb = a.bra_pn + (size_t)bi * (a.nmat + 1), *pk = a.ket_pn + (size_t)kj * (a.nmat + 1);
    const ScreenArgs sa{a.Bg, a.Bm, a.mol_boff, a.mol_ns, a.nmat, a.thresh, a.screen};
    pass = screen_candidate(sa, P, Q, pb, pk, qq, mask);
  }
  // precision split on the Schwarz product (the FP32 list when below cut32)
  const bool lo32 = pass && a.cut32 > 0.0 && qq < a.cut32;
  const bool hi64 = pass && !lo32;
  double p64 = hi64 ? kk4 : 0.0, p32 = lo32 ? kk4 : 0.0;
  for (int off = 32; off > 0; off >>= 1) {
    p64 += __shfl_xor(p64, off);
    p32 += __shfl_xor(p32, off);
  }
  const unsigned long long bal[2] = {__ballot(hi64), __ballot(lo32)};
  if (lane == 0) {
    s_cnt[0][wv] = (unsigned)__popcll(bal[0]);
    s_cnt[1][wv] = (unsigned)__popcll(bal[1]);
    s_ps[0][wv] = p64;
    s_ps[1][wv] = p32;
  }
  __syncthreads();
  if (threadIdx.x < 2) {  // thread l reserves list l's slots for the whole block
    const int l = threadIdx.x;
    unsigned long long tot = 0;
    double ps = 0.0;
    for (int w = 0; w < NW; ++w) {
      tot += s_cnt[l][w];
      ps += s_ps[l][w];
    }
    unsigned long long st = 0;
    if (tot) {
      st = atomicAdd(l == 0 ? a.count : a.count32, tot);
      atomic_add(l == 0 ? a.prim_sum : a.prim_sum32, ps);
    }
    for (int w = 0; w < NW; ++w) {
      s_start[l][w] = st;
      st += s_cnt[l][w];
    }
  }
  __syncthreads();
  const bool take[2] = {hi64, lo32};
  for (int l = 0; l < 2; ++l) {
    if (!take[l]) continue;
    const unsigned long long slot = s_start[l][wv] + __popcll(bal[l] & ((1ull << lane) - 1ull));
    if ((long long)slot < (l == 0 ? a.cap : a.cap32)) {
      Quartet qv;
      qv.bra = (uint32_t)bi;
      qv.ket_mask = (uint32_t)kj | (mask << 24);
      (l == 0 ? a.out : a.out32)[slot] = qv;
    }
  }
  __syncthreads();  // the LDS above is rewritten by the next chunk
}

// Every list of a batch in one launch: list k covers the 1024-aligned
// chunks [start[k], start[k + 1]) of a common chunk space, so a chunk never
// spans two lists.
__global__ __launch_bounds__(kListThreads) void quartet_lists_kernel(const ListLaunch *lists, const long long *start,
                                                                     int nlist, long long nchunk) {
  __shared__ int s_k;
  for (long long c = blockIdx.x; c < nchunk; c += gridDim.x) {
    if (threadIdx.x == 0) {
      int lo = 0, hi = nlist - 1;  // last k with start[k] <= c
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= c) lo = mid; else hi = mid - 1;
      }
      s_k = lo;
    }
    __syncthreads();
    const int k = s_k;
    __syncthreads();
    list_chunk(lists[k], (c - start[k]) * kListThreads);
  }
}

// Tile lists: one block of kTileListWaves waves per chunk of kTileChunk
// sub-blocks of one list, each wave taking its sub-blocks one after the
// other.  Lane l tests candidate (i, j) = (l / 8, l % 8) of a sub-block
// with the quartet lists' screen; the survivors of each precision make the
// sub-block's tile (a bitmap and the masks) at the sub-block's own slot.
// The block's counts meet in LDS and take one atomic per counter.
constexpr int kTileListWaves = 4;
__global__ __launch_bounds__(64 * kTileListWaves) void tile_lists_kernel(const TileListLaunch *lists,
                                                                         const long long *start, int nlist,
                                                                         long long nchunk) {
  __shared__ unsigned long long s_cnt[kTileListWaves][3];
  __shared__ double s_ps[kTileListWaves][2];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (long long ch = blockIdx.x; ch < nchunk; ch += gridDim.x) {
    const long long t0 = ch * kTileChunk;
    int lo = 0, hi = nlist - 1;  // the chunk's list: last k with start[k] <= t0
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (start[mid] <= t0) lo = mid; else hi = mid - 1;
    }
    const TileListLaunch &a = lists[lo];
    const long long base = t0 - start[lo];
    unsigned long long ncand = 0, nq64 = 0, nq32 = 0;  // lane 0's running sums
    double ps64 = 0.0, ps32 = 0.0;
    for (int u = wv; u < kTileChunk; u += kTileListWaves) {
      const long long slot = base + u;
      const SubBlock sb = a.sub[slot];
      const int b0 = a.bmem[sb.bra_m0];
      const int mol = a.bra[b0].mol;
      // Schwarz pre-cut of the whole sub-block (uniform across the wave);
      // an empty sub-block has no candidates
      const bool live = sb.nb > 0 && !(a.screen && sb.qq * a.molmax[mol] < a.thresh);
      const int i = lane >> 3, j = lane & 7;
      const bool cand = live && i < sb.nb && j < sb.nk && (!sb.diag || i >= j);
      bool pass = false;
      unsigned mask = 0;
      double qq = 0.0, kk4 = 0.0;
      if (cand) {
        const int bi = a.bmem[sb.bra_m0 + i], kj = a.kmem[sb.ket_m0 + j];
        const PairScr P = a.bra[bi], Q = a.ket[kj];
        qq = P.Q * Q.Q;
        kk4 = (double)P.kk * (double)Q.kk;
        const ScreenArgs sa{a.Bg, a.Bm, a.mol_boff, a.mol_ns, a.nmat, a.thresh, a.screen};
        pass = screen_candidate(sa, P, Q, a.bra_pn + (size_t)bi * (a.nmat + 1),
                                a.ket_pn + (size_t)kj * (a.nmat + 1), qq, mask);
      }
      const bool lo32 = pass && a.cut32 > 0.0 && qq < a.cut32;
      const bool hi64 = pass && !lo32;
      const unsigned long long cbits = __ballot(cand);
      for (int l = 0; l < (a.out32 ? 2 : 1); ++l) {
        const bool take = l == 0 ? hi64 : lo32;
        const unsigned long long bits = __ballot(take);
        double ps = take ? kk4 : 0.0;
        for (int off = 32; off > 0; off >>= 1) ps += __shfl_xor(ps, off);
        Tile *T = (l == 0 ? a.out : a.out32) + slot;
        if (bits) T->mask[lane] = (unsigned char)(take ? mask : 0u);
        if (lane == 0) {
          T->bra_m0 = sb.bra_m0;
          T->ket_m0 = sb.ket_m0;
          T->nb = sb.nb;
          T->nk = sb.nk;
          T->pad = 0u;
          T->bits = bits;  // written for every sub-block: an empty tile is skipped
          T->pad2 = 0ull;
          if (l == 0) {
            nq64 += (unsigned long long)__popcll(bits);
            ps64 += ps;
          } else {
            nq32 += (unsigned long long)__popcll(bits);
            ps32 += ps;
          }
        }
      }
      if (lane == 0) ncand += (unsigned long long)__popcll(cbits);
    }
    if (lane == 0) {
      s_cnt[wv][0] = ncand;
      s_cnt[wv][1] = nq64;
      s_cnt[wv][2] = nq32;
      s_ps[wv][0] = ps64;
      s_ps[wv][1] = ps32;
    }
    __syncthreads();
    if (threadIdx.x < 5) {
      const int k = threadIdx.x;
      if (k < 3) {
        unsigned long long v = 0;
        for (int w = 0; w < kTileListWaves; ++w) v += s_cnt[w][k];
        unsigned long long *dst = k == 0 ? a.ncand : k == 1 ? a.nquart : a.nquart32;
        if (v && dst) atomicAdd(dst, v);
      } else {
        double v = 0.0;
        for (int w = 0; w < kTileListWaves; ++w) v += s_ps[w][k - 3];
        double *dst = k == 3 ? a.prim_sum : a.prim_sum32;
        if (v != 0.0 && dst) atomic_add(dst, v);
      }
    }
    __syncthreads();  // the LDS above is rewritten by the next chunk
  }
}

__global__ void to_cart_kernel(CartMap M, const double *X, int cplx, double *Pre, double *Pim,
                               int ps) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)M.nbc * M.nbc) return;
  const int i = (int)(t % M.nbc), j = (int)(t / M.nbc);
  const int si = M.cart_shell[i], ci = M.cart_comp[i];
  const int sj = M.cart_shell[j], cj = M.cart_comp[j];
  double re = 0.0, im = 0.0;
  for (int mu = 0; mu < nfunc(M, si); ++mu) {
    const double ti = tcoef(M, si, ci, mu);
    if (ti == 0.0) continue;
    for (int nu = 0; nu < nfunc(M, sj); ++nu) {
      const double tj = tcoef(M, sj, cj, nu);
      if (tj == 0.0) continue;
      const size_t idx = (M.sh_bf[si] - M.bf0 + mu) + (size_t)(M.sh_bf[sj] - M.bf0 + nu) * M.nb;
      if (cplx) {
        re += ti * tj * X[2 * idx];
        im += ti * tj * X[2 * idx + 1];
      } else {
        re += ti * tj * X[idx];
      }
    }
  }
  Pre[t * ps] = re;
  if (Pim) Pim[t * ps] = im;
}

// blockIdx.y: matrix of a batch of equal real ones, sa / sx doubles apart
__global__ void from_cart_kernel(CartMap M, const double *A, int her, double *AX, size_t sa, size_t sx) {
  A += blockIdx.y * sa;
  AX += blockIdx.y * sx;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)M.nb * M.nb) return;
  const int mu = (int)(t % M.nb), nu = (int)(t / M.nb);
  const int sm = M.bf_shell[mu], cm = M.bf_comp[mu];
  const int sn = M.bf_shell[nu], cn = M.bf_comp[nu];
  const int ncm = ncart_f(M.sh_l[sm]), ncn = ncart_f(M.sh_l[sn]);
  double a = 0.0, b = 0.0;
  for (int i = 0; i < ncm; ++i) {
    const double ti = tcoef(M, sm, i, cm);
    if (ti == 0.0) continue;
    for (int j = 0; j < ncn; ++j) {
      const double tj = tcoef(M, sn, j, cn);
      if (tj == 0.0) continue;
      a += ti * tj * A[(M.sh_bfc[sm] - M.bfc0 + i) + (size_t)(M.sh_bfc[sn] - M.bfc0 + j) * M.nbc];
      b += ti * tj * A[(M.sh_bfc[sn] - M.bfc0 + j) + (size_t)(M.sh_bfc[sm] - M.bfc0 + i) * M.nbc];
    }
  }
  AX[t] += her ? 0.5 * (a + b) : 0.5 * a;  // 1/2 (A + A^H), direct.hpp:2040-2049; 1/2 A, :2051-2062
}

__global__ void zero_kernel(double *p, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.0;
}

inline unsigned nblocks(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

hipError_t launch_tile_lists(const TileListLaunch *lists, const long long *start, int nlist, long long nsub,
                             hipStream_t s) {
  if (nsub <= 0 || nlist <= 0) return hipSuccess;
  if (nsub % kTileChunk) return hipErrorInvalidValue;  // lists are padded to whole chunks
  const long long nchunk = nsub / kTileChunk;
  const long long blocks = std::min<long long>(nchunk, 1ll << 20);
  hipLaunchKernelGGL(tile_lists_kernel, dim3((unsigned)blocks), dim3(64 * kTileListWaves), 0, s, lists, start,
                     nlist, nchunk);
  return hipGetLastError();
}

hipError_t launch_quartet_lists(const ListLaunch *lists, const long long *start, int nlist, long long nchunk,
                                hipStream_t s) {
  if (nlist <= 0 || nchunk <= 0) return hipSuccess;
  const long long blocks = nchunk < 65536 ? nchunk : 65536;
  hipLaunchKernelGGL(quartet_lists_kernel, dim3((unsigned)blocks), dim3(kListThreads), 0, s, lists, start, nlist,
                     nchunk);
  return hipGetLastError();
}

hipError_t launch_to_cart(const CartMap &m, const double *X, int is_complex, double *pre,
                          double *pim, int ps, hipStream_t s) {
  hipLaunchKernelGGL(to_cart_kernel, dim3(nblocks((long long)m.nbc * m.nbc, 256)), dim3(256), 0,
                     s, m, X, is_complex, pre, pim, ps);
  return hipGetLastError();
}

hipError_t launch_from_cart_many(const CartMap &m, const double *a, size_t sa, int her, double *AX, size_t sx,
                                 size_t n, hipStream_t s) {
  for (size_t k = 0; k < n; k += 65535) {
    const unsigned ny = (unsigned)std::min<size_t>(65535, n - k);
    hipLaunchKernelGGL(from_cart_kernel, dim3(nblocks((long long)m.nb * m.nb, 256), ny), dim3(256), 0, s, m, a + k * sa,
                       her, AX + k * sx, sa, sx);
  }
  return hipGetLastError();
}

hipError_t launch_zero(double *p, size_t n, hipStream_t s) {
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(zero_kernel, dim3(nblocks((long long)n, 256)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace cqx
