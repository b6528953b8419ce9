// Front and back of a build on the device: block norms, Cartesian planes,
// pair norms and pair-order Coulomb planes, candidate counts, and the
// transforms of the accumulators back.
//
// Each step is one launch over every molecule, contraction and class of the
// build.  Launched per molecule, contraction, class and class pair, as
// before, they were some 110 launches of 2-5 us in front of and behind the
// ERI launches of a one-molecule J/K build and several hundred for a batch.
// They are latency, a few microseconds each at any size: with the saved
// waits and copies water / 6-31G(d) went
// 0.75 -> 0.44 ms, 32 molecules / cc-pVDZ 36.2 -> 34.0, (H2O)7 / cc-pVDZ
// 1.84 -> 1.65.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cart_coef.hpp"
#include "front.hpp"

namespace cqx {

namespace {

// molecule whose range of the given prefix field holds t
template <long long MolInfo::*F>
__device__ __forceinline__ int mol_of(const FrontArgs &a, long long t) {
  int lo = 0, hi = a.nmol - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.mol[mid].*F <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ const double *x_of(const FrontArgs &a, int m, int j) {
  return a.nmol == 1 ? a.xs[j] : a.x[(size_t)m * a.nmat + j];
}
__device__ __forceinline__ double *ax_of(const FrontArgs &a, int m, int j) {
  return a.nmol == 1 ? a.axs[j] : a.ax[(size_t)m * a.nmat + j];
}
__device__ __forceinline__ const MolPlanes &planes_of(const FrontArgs &a, int m) {
  return a.nmol == 1 ? a.m0 : a.mols[m];
}

__global__ void zero_ranges_kernel(ZeroRanges z) {
  const int r = blockIdx.y;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < z.n[r]; t += step) z.p[r][t] = 0.0;
}

// ShellBlockNorm (direct.hpp:73-105): B(s1, s2) = max_i sum_j |X(i, j)| over
// the (s1, s2) block, symmetrised for a non-Hermitian X (:1537-1545); the
// global norm is the max over the matrices.
__device__ __forceinline__ double block_norm(const FrontArgs &a, const double *X, const MolInfo &M, int s1, int s2) {
  const int r0 = a.map.sh_bf[M.sh0 + s1] - M.bf0, c0 = a.map.sh_bf[M.sh0 + s2] - M.bf0;
  const int nr = a.sh_nf[M.sh0 + s1], nc = a.sh_nf[M.sh0 + s2];
  double mx = 0.0;
  for (int i = 0; i < nr; ++i) {
    double row = 0.0;
    for (int j = 0; j < nc; ++j) {
      const size_t e = (r0 + i) + (size_t)(c0 + j) * M.nb;
      row += a.cplx ? hypot(X[2 * e], X[2 * e + 1]) : fabs(X[e]);
    }
    mx = fmax(mx, row);
  }
  return mx;
}

__global__ __launch_bounds__(256) void norms_kernel(FrontArgs a, long long n) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  int m = -1;
  double g = 0.0;
  if (t < n) {
    m = mol_of<&MolInfo::boff>(a, t);
    const MolInfo M = a.mol[m];
    const int e = (int)(t - M.boff), s1 = e % M.ns, s2 = e / M.ns;
    for (int j = 0; j < a.nmat; ++j) {
      const double *X = x_of(a, m, j);
      double b = block_norm(a, X, M, s1, s2);
      if (!((a.her >> j) & 1u)) b = fmax(b, block_norm(a, X, M, s2, s1));
      a.Bm[t * a.nmat + j] = b;
      g = fmax(g, b);
    }
    a.Bg[t] = g;
  }
  // the molecule's largest: non-negative doubles order as their bit patterns
  unsigned long long bits = (unsigned long long)__double_as_longlong(g);
  const int m0 = __builtin_amdgcn_readfirstlane(m);
  if (__ballot(m != m0 && m >= 0) == 0ull) {
    for (int o = 32; o > 0; o >>= 1) {
      const unsigned long long v = __shfl_xor(bits, o);
      bits = v > bits ? v : bits;
    }
    if ((threadIdx.x & 63) == 0 && m0 >= 0) atomicMax((unsigned long long *)&a.molmax[m0], bits);
  } else if (m >= 0) {
    atomicMax((unsigned long long *)&a.molmax[m], bits);
  }
}

// blockIdx.y: contraction
__global__ __launch_bounds__(256) void planes_kernel(FrontArgs a, long long n) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  const int j = blockIdx.y, m = mol_of<&MolInfo::nbc2>(a, t);
  const MolInfo M = a.mol[m];
  const long long e = t - M.nbc2;
  const int i = (int)(e % M.nbc), k = (int)(e / M.nbc);
  const int si = a.map.cart_shell[M.bfc0 + i], ci = a.map.cart_comp[M.bfc0 + i];
  const int sk = a.map.cart_shell[M.bfc0 + k], ck = a.map.cart_comp[M.bfc0 + k];
  const double *X = x_of(a, m, j);
  double re = 0.0, im = 0.0;
  for (int mu = 0; mu < nfunc(a.map, si); ++mu) {
    const double ti = tcoef(a.map, si, ci, mu);
    if (ti == 0.0) continue;
    for (int nu = 0; nu < nfunc(a.map, sk); ++nu) {
      const double tk = tcoef(a.map, sk, ck, nu);
      if (tk == 0.0) continue;
      const size_t x = (a.map.sh_bf[si] - M.bf0 + mu) + (size_t)(a.map.sh_bf[sk] - M.bf0 + nu) * M.nb;
      if (a.cplx) {
        re += ti * tk * X[2 * x];
        im += ti * tk * X[2 * x + 1];
      } else {
        re += ti * tk * X[x];
      }
    }
  }
  double *P = const_cast<double *>(planes_of(a, m).kx[a.kind[j]]) + (size_t)e * a.kps[a.kind[j]];
  P[a.re[j]] = re;
  if (a.im[j] >= 0) P[a.im[j]] = im;
}

// (component, pair) t of a class: class, component and pair index
__device__ __forceinline__ bool class_item(const FrontArgs &a, long long t, int &k, int &e, int &i) {
  if (t >= a.cstart[kMaxClass]) return false;
  k = 0;
  while (t >= a.cstart[k + 1]) ++k;
  const long long r = t - a.cstart[k];
  e = (int)(r / a.npair[k]);
  i = (int)(r - (long long)e * a.npair[k]);
  return true;
}
__device__ __forceinline__ int second_ncart(int k) {  // components of the second shell of class k
  int la = 0;
  while ((la + 1) * (la + 2) / 2 <= k) ++la;
  return ncart_f(k - la * (la + 1) / 2);
}

__global__ __launch_bounds__(256) void pairs_kernel(FrontArgs a) {
  int k, e, i;
  if (!class_item(a, (long long)blockIdx.x * 256 + threadIdx.x, k, e, i)) return;
  if (e == 0) {
    const PairScr P = a.scr[k][i];
    const int s1 = (int)(P.s12 & 0xFFFFu), s2 = (int)(P.s12 >> 16);
    const MolInfo M = a.mol[P.mol];
    const size_t b = (size_t)M.boff + s1 + (size_t)s2 * M.ns;
    double *pn = a.pn[k] + (size_t)i * (a.nmat + 1);
    pn[0] = a.Bg[b];
    for (int j = 0; j < a.nmat; ++j) pn[1 + j] = a.Bm[b * a.nmat + j];
  }
  if (!a.jx) return;
  const PairRec &P = a.pairs[k][i];
  const MolPlanes &mp = planes_of(a, P.mol);
  const int nb = second_ncart(k), r = P.bfa + e / nb, c = P.bfb + e % nb;
  const size_t nc_n = (size_t)(a.cstart[k + 1] - a.cstart[k]);
  for (int j = 0; j < a.nj; ++j) {
    const int kd = a.jkind[j];
    const double *x = mp.kx[kd] + a.jidx[j];
    double v = x[((size_t)c + (size_t)r * mp.nbc) * a.kps[kd]];
    if (kd == kJNonHer) v += x[((size_t)r + (size_t)c * mp.nbc) * a.kps[kd]];
    a.jx[a.joff[k] + j * nc_n + (size_t)e * a.npair[k] + i] = v;
  }
}

__global__ __launch_bounds__(256) void pairs_back_kernel(FrontArgs a) {
  int k, e, i;
  if (!class_item(a, (long long)blockIdx.x * 256 + threadIdx.x, k, e, i)) return;
  const PairRec &P = a.pairs[k][i];
  const MolPlanes &mp = planes_of(a, P.mol);
  const int nb = second_ncart(k), r = P.bfa + e / nb, c = P.bfb + e % nb;
  const size_t nc_n = (size_t)(a.cstart[k + 1] - a.cstart[k]);
  for (int j = 0; j < a.nj; ++j) {
    const double v = a.ja[a.joff[k] + j * nc_n + (size_t)e * a.npair[k] + i];
    if (v == 0.0) continue;
    const int kd = a.jkind[j];
    double *o = mp.ka[kd] + a.jidx[j];
    unsafeAtomicAdd(o + ((size_t)r + (size_t)c * mp.nbc) * a.kps[kd], v);
    if (kd == kJNonHer) unsafeAtomicAdd(o + ((size_t)c + (size_t)r * mp.nbc) * a.kps[kd], v);
  }
}

// Candidate kets of every bra pair: the Schwarz pre-cut prefix of its own
// molecule's kets (Q descending), and the inclusive prefix sums over the
// bras -- the same arithmetic the screening of the reference loop implies
// before its per-quartet test (direct.hpp:1689-1789).
__global__ __launch_bounds__(1024) void candidates_kernel(const CandLaunch *table, long long *tot) {
  __shared__ long long s_wave[16];
  __shared__ CandLaunch s_a;
  if (threadIdx.x == 0) s_a = table[blockIdx.x];
  __syncthreads();
  const CandLaunch &a = s_a;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  long long run = 0;
  if (threadIdx.x == 0) a.off[0] = 0;
  for (int base = 0; base < a.nbra; base += 1024) {
    const int i = base + threadIdx.x;
    long long jmax = 0;
    if (i < a.nbra) {
      const int m = a.bra[i].mol;
      const double Q = a.bra[i].Q;
      const int lo = a.seg[m], hi = a.seg[m + 1];
      jmax = hi - lo;
      if (a.screen && jmax > 0) {
        const double bmax = a.molmax[m];
        if (bmax * Q * a.ket[lo].Q < a.thresh) {
          jmax = 0;
        } else {
          // largest prefix with Q_i Q_j bmax >= thresh
          const double need = a.thresh / (bmax * Q);
          int x = lo, y = hi;
          while (x < y) {
            const int mid = (x + y) / 2;
            if (a.ket[mid].Q >= need) x = mid + 1; else y = mid;
          }
          jmax = x - lo;
        }
      }
      if (a.same_class) jmax = min(jmax, (long long)(a.bra_base + i - lo + 1));
      if (jmax < 0) jmax = 0;
      a.klo[i] = lo;
    }
    long long v = jmax;
    for (int o = 1; o < 64; o <<= 1) {
      const long long u = __shfl_up(v, o);
      if (lane >= o) v += u;
    }
    __syncthreads();  // the previous chunk's wave sums have been read
    if (lane == 63) s_wave[wv] = v;
    __syncthreads();
    long long before = run, all = 0;
    for (int w = 0; w < 16; ++w) {
      if (w < wv) before += s_wave[w];
      all += s_wave[w];
    }
    if (i < a.nbra) a.off[i + 1] = before + v;
    run += all;
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = run;
}

// blockIdx.y: contraction, from j0 on
__global__ __launch_bounds__(256) void back_kernel(FrontArgs a, long long first, long long last, int j0) {
  const long long t = first + (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= last) return;
  const int j = j0 + blockIdx.y, m = mol_of<&MolInfo::nb2>(a, t);
  const MolInfo M = a.mol[m];
  const long long e = t - M.nb2;
  const int mu = (int)(e % M.nb), nu = (int)(e / M.nb);
  const int sm = a.map.bf_shell[M.bf0 + mu], cm = a.map.bf_comp[M.bf0 + mu];
  const int sn = a.map.bf_shell[M.bf0 + nu], cn = a.map.bf_comp[M.bf0 + nu];
  const int ncm = ncart_f(a.map.sh_l[sm]), ncn = ncart_f(a.map.sh_l[sn]);
  const int f0 = a.map.sh_bfc[sm] - M.bfc0, g0 = a.map.sh_bfc[sn] - M.bfc0;
  const int kd = a.kind[j], S = a.kps[kd];
  const MolPlanes &mp = planes_of(a, m);
  const double *Are = mp.ka[kd] + a.re[j];
  const double *Aim = a.im[j] >= 0 ? mp.ka[kd] + a.im[j] : nullptr;
  const bool her = (a.her >> j) & 1u;
  double a_re = 0.0, a_im = 0.0, b_re = 0.0, b_im = 0.0;
  for (int i = 0; i < ncm; ++i) {
    const double ti = tcoef(a.map, sm, i, cm);
    if (ti == 0.0) continue;
    for (int k = 0; k < ncn; ++k) {
      const double tk = tcoef(a.map, sn, k, cn);
      if (tk == 0.0) continue;
      const size_t ik = ((f0 + i) + (size_t)(g0 + k) * M.nbc) * S, ki = ((g0 + k) + (size_t)(f0 + i) * M.nbc) * S;
      a_re += ti * tk * Are[ik];
      if (her) b_re += ti * tk * Are[ki];
      if (Aim) {
        a_im += ti * tk * Aim[ik];
        if (her) b_im += ti * tk * Aim[ki];
      }
    }
  }
  double re, im;
  if (her) {  // 1/2 (A + A^H), direct.hpp:2040-2049
    re = 0.5 * (a_re + b_re);
    im = 0.5 * (a_im - b_im);
  } else {    // 1/2 A, direct.hpp:2051-2062
    re = 0.5 * a_re;
    im = 0.5 * a_im;
  }
  double *AX = ax_of(a, m, j);
  if (a.cplx) {
    AX[2 * e] += re;
    AX[2 * e + 1] += im;
  } else {
    AX[e] += re;
  }
}

inline unsigned blocks256(long long n) { return (unsigned)((n + 255) / 256); }

}  // namespace

hipError_t launch_zero_ranges(const ZeroRanges &z, hipStream_t s) {
  if (!z.count) return hipSuccess;
  size_t most = 0;
  for (int k = 0; k < z.count; ++k) most = std::max(most, z.n[k]);
  const unsigned nx = (unsigned)std::min<size_t>((most + 255) / 256, 4096);
  hipLaunchKernelGGL(zero_ranges_kernel, dim3(nx, (unsigned)z.count), dim3(256), 0, s, z);
  return hipGetLastError();
}

hipError_t launch_norms(const FrontArgs &a, long long nblock, hipStream_t s) {
  if (nblock <= 0) return hipSuccess;
  hipLaunchKernelGGL(norms_kernel, dim3(blocks256(nblock)), dim3(256), 0, s, a, nblock);
  return hipGetLastError();
}

hipError_t launch_planes(const FrontArgs &a, long long nbc2, hipStream_t s) {
  if (nbc2 <= 0) return hipSuccess;
  hipLaunchKernelGGL(planes_kernel, dim3(blocks256(nbc2), (unsigned)a.nmat), dim3(256), 0, s, a, nbc2);
  return hipGetLastError();
}

hipError_t launch_pairs(const FrontArgs &a, hipStream_t s) {
  if (a.cstart[kMaxClass] <= 0) return hipSuccess;
  hipLaunchKernelGGL(pairs_kernel, dim3(blocks256(a.cstart[kMaxClass])), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_candidates_all(const CandLaunch *table, int n, long long *tot, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(candidates_kernel, dim3((unsigned)n), dim3(1024), 0, s, table, tot);
  return hipGetLastError();
}

hipError_t launch_pairs_back(const FrontArgs &a, hipStream_t s) {
  if (a.cstart[kMaxClass] <= 0 || !a.nj) return hipSuccess;
  hipLaunchKernelGGL(pairs_back_kernel, dim3(blocks256(a.cstart[kMaxClass])), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_back(const FrontArgs &a, long long first, long long last, int j0, int nj, hipStream_t s) {
  if (last <= first || nj <= 0) return hipSuccess;
  hipLaunchKernelGGL(back_kernel, dim3(blocks256(last - first), (unsigned)nj), dim3(256), 0, s, a, first, last, j0);
  return hipGetLastError();
}

}  // namespace cqx
