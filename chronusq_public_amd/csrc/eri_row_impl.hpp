// Row kernels: screening, ERI evaluation and J/K digestion of one class pair
// in one launch, for the classes whose contracted Cartesian quartet fits a
// lane's registers.
//
// What bounded the quartet-list kernels: their J/K updates went to HBM as
// memory-side atomics (7 to 15 per quartet, executed at about 24 per ns on
// this device whatever the kernel does), and the updates were formed by the
// whole wave from quartets staged in LDS, with as much index arithmetic and
// LDS latency per update as arithmetic.  Here a block takes one bra pair
// (a, b) and a chunk of its kets.  For a fixed bra every exchange update
// falls into the rows K(a, :) and K(b, :), and every density element read
// comes from the rows X(a, :) and X(b, :): both sit in LDS for the whole
// chunk, in columns numbered over the functions of the ket class's two
// angular momenta only.  A lane (or a group of G lanes that split the ket's
// primitive pairs) evaluates a ket and digests it from its registers with
// LDS atomics; the rows go to HBM once per chunk.  J(a, b) is summed over
// the wave; J(c, d) and X(d, c) are kept in the class's pair order, in which
// neighbouring lanes hold neighbouring doubles.
//
// Each block screens its own kets (no quartet list, no host round trip) and
// sorts the survivors by their primitive pairs, so that the lanes of a wave
// run loops of one length.  With two bins (contraction products up to 8 and
// beyond) half of the lanes idled: 6-31G(d) carbon pairs have 1, 3 or 6 in
// the first and 9, 18 or 36 in the second.  Measured with the bins and
// sorted (ms a build): C40H82 / 6-31G(d) 32.7 -> 28.5, mixed 29.2 -> 25.0, 32
// water clusters batched, mixed, 34.0 -> 28.5, (H2O)4 / cc-pVDZ 0.79 -> 0.61,
// non-Hermitian complex (H2O)7 1.63 -> 1.32.
//
// Measured against the quartet-list build (ms a build, two bins): C40H82
// 90.5 -> 36.9, mixed 71.5 -> 30.8; the batch 75 -> 38; GHF (H2O)16 / cc-pVDZ
// 12.8 -> 9.4; (H2O)7 3.2 -> 2.0; (H2O)4 1.38 -> 1.10.  With the later changes
// noted below and the front's C40H82 takes 23.9, mixed 20.5, the batch 20.4,
// GHF 8.6, (H2O)7 1.15, (H2O)4 0.57.  What bounds them now: about half of the
// VALU's cycles at three wavefronts a SIMD (chains of reciprocal square root,
// table read and Horner steps), the LDS 25 to 50 % busy with the table.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "digest.hpp"
#include "eri_bra.hpp"
#include "eri_class.hpp"
#include "eri_row.hpp"
#include "screen.hpp"

namespace cqx {

namespace {

// Sums of N values over the wave, added to out: while a lane holds several
// values it gives half of them to its partner and takes the partner's share of
// the rest, so N values cost about N + 4 exchanges instead of 6 N.  (With six
// each, the J(a, b) sums of C40H82 / 6-31G(d) took 0.28 of 1.29 ms of
// (dp|ss) and 0.14 of 0.45 of (dd|ss).)
template <int N, int O>
__device__ __forceinline__ void wave_sums_add(const double (&v)[N], int base, int most, double *out, int lane) {
  if constexpr (O == 0) {
    if (base < most) unsafeAtomicAdd(out + base, v[0]);
  } else if constexpr (N == 1) {
    double s = v[0];
#pragma unroll
    for (int o = O; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (base < most && (lane & (2 * O - 1)) == 0) unsafeAtomicAdd(out + base, s);
  } else {
    constexpr int H = (N + 1) / 2;
    const bool up = (lane & O) != 0;
    double keep[H];
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const double hi = H + i < N ? v[H + i < N ? H + i : 0] : 0.0;  // (a slot beyond the last adds nothing)
      keep[i] = (up ? hi : v[i]) + __shfl_xor(up ? v[i] : hi, O);
    }
    wave_sums_add<H, O / 2>(keep, base + (up ? H : 0), most, out, lane);
  }
}

// Buckets of the surviving kets by their primitive pairs: exact up to 32,
// then in fours, the last one open.  bucket_most: the most primitive pairs of
// a bucket (of the open one a stand-in: it takes the most lanes anyway).
constexpr int kRowBuckets = 64;
__device__ __forceinline__ int row_bucket(int npp) {
  return npp <= 32 ? max(npp, 1) - 1 : min(32 + (npp - 33) / 4, kRowBuckets - 1);
}
__device__ __forceinline__ int bucket_most(int k) { return k < 32 ? k + 1 : 36 + 4 * (k - 32); }

// sum over the wave, in every lane
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// The four exchange updates of one quartet in row form: with rows Xa = X(a, :)
// and Xb = X(b, :),
//   K(a, c) += I X(b, d)   K(a, d) += I X(b, c)
//   K(b, c) += I X(a, d)   K(b, d) += I X(a, c)
// (direct.hpp:1889-1917, 1961-1998; the 1/2 is applied when the rows are
// flushed).  k: the plane's NA + NB exchange rows of w columns, kets at
// columns c and d; x(r, k, second): element k of row r from ket shell c or d.
template <class K, class X>
__device__ __forceinline__ void digest_rows(const double (&I)[K::NC], const X &x, double *k, int w, int c, int d) {
  {
    double kc[K::NCA][K::NCC], kd[K::NCA][K::NCD];
#pragma unroll
    for (int ia = 0; ia < K::NCA; ++ia) {
#pragma unroll
      for (int ic = 0; ic < K::NCC; ++ic) kc[ia][ic] = 0.0;
#pragma unroll
      for (int id = 0; id < K::NCD; ++id) kd[ia][id] = 0.0;
    }
#pragma unroll
    for (int ib = 0; ib < K::NCB; ++ib) {
      double xc[K::NCC], xd[K::NCD];
#pragma unroll
      for (int ic = 0; ic < K::NCC; ++ic) xc[ic] = x(K::NCA + ib, ic, false);
#pragma unroll
      for (int id = 0; id < K::NCD; ++id) xd[id] = x(K::NCA + ib, id, true);
#pragma unroll
      for (int ia = 0; ia < K::NCA; ++ia)
#pragma unroll
        for (int ic = 0; ic < K::NCC; ++ic)
#pragma unroll
          for (int id = 0; id < K::NCD; ++id) {
            const double v = I[K::oidx(ia, ib, ic, id)];
            kc[ia][ic] = fma(v, xd[id], kc[ia][ic]);
            kd[ia][id] = fma(v, xc[ic], kd[ia][id]);
          }
    }
#pragma unroll
    for (int ia = 0; ia < K::NCA; ++ia) {
#pragma unroll
      for (int ic = 0; ic < K::NCC; ++ic) unsafeAtomicAdd(k + ia * w + c + ic, kc[ia][ic]);
#pragma unroll
      for (int id = 0; id < K::NCD; ++id) unsafeAtomicAdd(k + ia * w + d + id, kd[ia][id]);
    }
  }
#pragma unroll
  for (int ib = 0; ib < K::NCB; ++ib) {
    double kc[K::NCC], kd[K::NCD];
#pragma unroll
    for (int ic = 0; ic < K::NCC; ++ic) kc[ic] = 0.0;
#pragma unroll
    for (int id = 0; id < K::NCD; ++id) kd[id] = 0.0;
#pragma unroll
    for (int ia = 0; ia < K::NCA; ++ia) {
      double xc[K::NCC], xd[K::NCD];
#pragma unroll
      for (int ic = 0; ic < K::NCC; ++ic) xc[ic] = x(ia, ic, false);
#pragma unroll
      for (int id = 0; id < K::NCD; ++id) xd[id] = x(ia, id, true);
#pragma unroll
      for (int ic = 0; ic < K::NCC; ++ic)
#pragma unroll
        for (int id = 0; id < K::NCD; ++id) {
          const double v = I[K::oidx(ia, ib, ic, id)];
          kc[ic] = fma(v, xd[id], kc[ic]);
          kd[id] = fma(v, xc[ic], kd[id]);
        }
    }
    double *row = k + (K::NCA + ib) * w;
#pragma unroll
    for (int ic = 0; ic < K::NCC; ++ic) unsafeAtomicAdd(row + c + ic, kc[ic]);
#pragma unroll
    for (int id = 0; id < K::NCD; ++id) unsafeAtomicAdd(row + d + id, kd[id]);
  }
}

// Work item t of a launch: bra pair t / nchunk, candidate kets
// [t % nchunk, ...) kRowChunk of its molecule's segment.  Dynamic LDS: the
// exchange rows ([plane][NA + NB][width]), then, with XL, the density rows;
// without XL the density is read from its planes in global memory (many
// planes, whose density rows would not fit beside the exchange rows).
// Most threads of a block (256 where a lane takes more than 256 registers),
// and wavefronts per SIMD asked of the compiler: six for the classes that fit
// 80 registers (C40H82 / 6-31G(d), ms a launch: (ss|ss) 2.72 -> 2.27, (ps|ss)
// 3.67 -> 3.40 for the compiler's own five; five for (ps|ps) spill, 1.89 ->
// 2.37).
template <class K>
constexpr int row_threads() {
  return K::NC > 54 ? 256 : 512;
}
template <class K>
constexpr int row_waves() {
  return K::NC <= 3 ? 6 : K::NC <= 9 ? 4 : 1;
}
template <int LA, int LB, int LC, int LD, class R, bool XL>
__global__ __launch_bounds__((row_threads<Cls<LA, LB, LC, LD>>()),
                                        (row_waves<Cls<LA, LB, LC, LD>>())) void eri_row_kernel(RowLaunch a) {
  using K = Cls<LA, LB, LC, LD>;
  const int nthread = blockDim.x;  // see row_block
  constexpr int NROW = K::NCA + K::NCB, NAB = K::NCA * K::NCB, NCD = K::NCC * K::NCD;
  extern __shared__ double s_rows[];
  using Rys = RysRow<K::NR, R, K::NC == 1, XL>;
  __shared__ alignas(16) R s_tab[Rys::kLen];
  __shared__ unsigned s_queue[kRowChunk];  // surviving kets, most primitive pairs first
  __shared__ int s_hist[kRowBuckets];
  __shared__ double s_jab[kRowJ * NAB];
  __shared__ int s_next;
  __shared__ unsigned long long s_tot[2];
  __shared__ double s_psum;
  const int tid = threadIdx.x, lane = tid & 63;
  {
    const R *g = rys_table<R>(Rys::kHalf ? a.rys_half : a.rys, a.rys32_half);
    for (int e = tid; e < Rys::kLen; e += nthread) s_tab[e] = g[Rys::src(e)];
    if (tid == 0) {
      s_tot[0] = s_tot[1] = 0;
      s_psum = 0.0;
    }
  }
  const int w = a.width, rows = a.nk * NROW * w;
  double *s_k = s_rows, *s_x = s_rows + rows;
  const long long nitem = (long long)a.nbra * a.nchunk;
  for (long long item = blockIdx.x; item < nitem; item += gridDim.x) {
    const int i = (int)(item / a.nchunk), ch = (int)(item - (long long)i * a.nchunk);
    const ConstPtr<PairRec> bp = as_const(a.bra + i);
    const int mol = bp->mol;
    const int lo = as_const(a.seg)[mol];
    int hi = as_const(a.seg)[mol + 1];
    if (a.same_class) hi = min(hi, i + 1);
    const int j0 = lo + ch * kRowChunk, j1 = min(hi, j0 + kRowChunk);
    if (j0 >= j1) continue;
    // candidates: the Schwarz pre-cut prefix of the molecule's kets (Q
    // descending), as in candidates_kernel; the precision split is monotonic
    // in the ket index too
    const double Qi = bp->Q;
    double need = 0.0;
    if (a.screen) {
      const double bmax = as_const(a.molmax)[mol];
      if (bmax * Qi * as_const(a.kscr + lo)->Q < a.thresh) continue;
      need = a.thresh / (bmax * Qi);
      if (as_const(a.kscr + j0)->Q < need) continue;
    }
    if (a.cut32 > 0.0) {
      if (!a.fp32 && Qi * as_const(a.kscr + j0)->Q < a.cut32) continue;
      if (a.fp32 && !(Qi * as_const(a.kscr + (j1 - 1))->Q < a.cut32)) continue;
    }
    __syncthreads();  // the previous item's rows, queue and sums have been read
    if (tid < kRowBuckets) s_hist[tid] = 0;
    if (tid == 0) s_next = 0;
    __syncthreads();
    const PairScr P = a.bscr[i];
    const ScreenArgs sa{a.Bg, a.Bm, a.mol_boff, a.mol_ns, a.nmat, a.thresh, a.screen};
    int ncand = 0;
    double psum = 0.0;
    constexpr int kPer = kRowChunk / 256;
    unsigned mine[kPer];  // ket, contractions
    int place[kPer];      // bucket and rank in it (< 0: none)
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int t = tid + u * nthread, j = j0 + t;
      bool pass = false, cand = false;
      unsigned mask = 0;
      int kk = 0, npp = 0;
      if (t < kRowChunk && j < j1) {
        const PairScr Q = a.kscr[j];
        npp = a.ket[j].npp;
        const double qq = P.Q * Q.Q;
        kk = Q.kk;
        const bool lo32 = a.cut32 > 0.0 && qq < a.cut32;
        if (lo32 == (a.fp32 != 0) && (!a.screen || Q.Q >= need)) {
          cand = true;
          pass = screen_candidate(sa, P, Q, a.bra_pn + (size_t)i * (a.nmat + 1), a.ket_pn + (size_t)j * (a.nmat + 1),
                                  qq, mask);
        }
      }
      ncand += __popcll(__ballot(cand));
      mine[u] = (unsigned)t | (mask << 16);
      place[u] = -1;
      if (pass) {
        psum += (double)P.kk * (double)kk;
        const int b = row_bucket(npp);
        place[u] = b | (atomicAdd(&s_hist[b], 1) << 8);
      }
    }
    psum = wave_sum(psum);
    if (lane == 0) {
      if (ncand) atomicAdd(&s_tot[1], (unsigned long long)ncand);
      if (psum != 0.0) unsafeAtomicAdd(&s_psum, psum);
    }
    __syncthreads();
    // every wave for itself: kets in the buckets from lane's own up (the
    // queue is in descending order), and the primitive pairs of all
    const int cnt = s_hist[lane], most = bucket_most(lane);
    int upto = cnt, work = cnt * most;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_down(upto, o);
      if (lane + o < 64) upto += v;
      work += __shfl_xor(work, o);
    }
    const int n = __builtin_amdgcn_readfirstlane(upto);
    if (n == 0) continue;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int first = __shfl(upto - cnt, place[u] & (kRowBuckets - 1));
      if (place[u] >= 0) s_queue[first + (place[u] >> 8)] = mine[u];
    }
    if (tid == 0) s_tot[0] += (unsigned long long)n;
    // Lanes per ket: a lane takes at most `turns` primitive pairs, so that no
    // ket outlasts an even share of the block's work (one lane each in a full
    // chunk, whose digestion then uses every lane; up to 64 where a bra has a
    // handful of kets); kets [end[l + 1], end[l]) of the queue get 2^l lanes.
    work = __builtin_amdgcn_readfirstlane(work);
    const int turns = max(1, work / nthread);
    int end[8], nunit = 0;
    end[0] = n;
    end[7] = 0;
#pragma unroll
    for (int l = 1; l < 7; ++l) {
      const unsigned long long more = __ballot(most > (turns << (l - 1)));
      end[l] = more ? __builtin_amdgcn_readlane(upto, (int)__builtin_ctzll(more)) : 0;
    }
#pragma unroll
    for (int l = 0; l < 7; ++l) nunit += (((end[l] - end[l + 1]) << l) + 63) >> 6;
    // with fewer units than waves, each unit's bra primitives are dealt over
    // several waves (the digestion is linear in the integrals), two or more
    // each: a chain of 64 bra primitives is 8 long in a small molecule
    const int nb = bp->npp;
    int nsplit = 1;
    while (2 * nsplit * nunit <= nthread / 64 && nb >= 4 * nsplit) nsplit *= 2;
    // the molecule's planes; density rows in, exchange rows cleared
    const bool one = a.nmol == 1;
    const ConstPtr<MolPlanes> mp = as_const(a.mols + (one ? 0 : mol));
    const int N = one ? a.m0.nbc : mp->nbc;
    const int bfa = bp->bfa, bfb = bp->bfb;
    const int *colmap = a.colmap + (size_t)mol * w;
    for (int p = 0; p < a.nk; ++p) {
      const RowPlane &rp = a.k[p];
      const GlobalDouble *x = (const GlobalDouble *)(one ? a.m0.kx[rp.kind] : mp->kx[rp.kind]) + rp.idx;
      const int S = a.kps[rp.kind];
      double *xs = s_x + p * NROW * w, *ks = s_k + p * NROW * w;
      for (int c = tid; c < w; c += nthread) {
        const int f = colmap[c];
        if (f < 0) continue;
#pragma unroll
        for (int r = 0; r < NROW; ++r) {
          const int fr = r < K::NCA ? bfa + r : bfb + (r - K::NCA);
          if constexpr (XL)
            xs[r * w + c] = rp.sign * x[(size_t)(rp.colwise ? f + (size_t)fr * N : fr + (size_t)f * N) * S];
          ks[r * w + c] = 0.0;
        }
      }
    }
    for (int e = tid; e < a.nj * NAB; e += nthread) s_jab[e] = 0.0;
    __syncthreads();
    const int pa = bp->a, pb = bp->b;
    const double bra_scale = 0.5 * (pa == pb ? 1.0 : 2.0);
    for (;;) {
      int grp = 0;
      if (lane == 0) grp = atomicAdd(&s_next, 1);
      grp = __builtin_amdgcn_readfirstlane(grp);
      if (grp >= nunit * nsplit) break;
      const int part = grp / nunit;
      int unit = grp - part * nunit, lg = 0, from = 0, to = 0;
#pragma unroll
      for (int l = 6; l >= 0; --l) {
        const int m = (((end[l] - end[l + 1]) << l) + 63) >> 6;
        if (unit >= 0 && unit < m) {
          lg = l;
          from = end[l + 1] + (unit << (6 - l));
          to = end[l];
        }
        unit -= m;
      }
      const int G = 1 << lg, slot = from + (lane >> lg), g = lane & (G - 1);
      const bool valid = slot < to;
      const unsigned q = valid ? s_queue[slot] : 0u;
      const int j = j0 + (int)(q & 0xFFFFu);
      const unsigned mask = q >> 16;
      int koff = 0, nkp = 0, c = 0, d = 0, fc = 0, fd = 0;
      double Cc[3] = {}, CD[3] = {};
      if (valid) {
        const RowKet &kt = a.ket[j];
        koff = kt.pp_off;
        nkp = kt.npp;
        c = kt.colc;
        d = kt.cold;
        fc = kt.bfc;
        fd = kt.bfd;
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          Cc[e] = kt.C[e];
          CD[e] = kt.CD[e];
        }
      }
      R I[K::NC];
#pragma unroll
      for (int o = 0; o < K::NC; ++o) I[o] = 0;
      eval_bra<LA, LB, LC, LD, R, XL>(a.prims, a.primc32, s_tab, bp, nb * part / nsplit, nb * (part + 1) / nsplit, Cc, CD,
                                  koff, nkp, g, G, I);
      for (int off = G >> 1; off > 0; off >>= 1) {
#pragma unroll
        for (int o = 0; o < K::NC; ++o) I[o] += __shfl_xor(I[o], off);
      }
      const bool take = valid && g == 0;
      // degeneracy in the 8-fold loop (direct.hpp:1664-1667, 1793-1802) and the 1/2 of :1849-1850
      const double scale =
          take ? bra_scale * (LC == LD && c == d ? 1.0 : 2.0) * (a.same_class && i == j ? 1.0 : 2.0) : 0.0;
      double Id[K::NC];
#pragma unroll
      for (int o = 0; o < K::NC; ++o) Id[o] = (double)I[o] * scale;
      if (take)
        for (int p = 0; p < a.nk; ++p) {
          const RowPlane &rp = a.k[p];
          if (!((mask >> rp.mat) & 1u)) continue;
          if constexpr (XL) {
            const double *xs = s_x + p * NROW * w;
            digest_rows<K>(Id, [&](int r, int e, bool second) { return xs[r * w + (second ? d : c) + e]; },
                           s_k + p * NROW * w, w, c, d);
          } else {
            const GlobalDouble *x = (const GlobalDouble *)(one ? a.m0.kx[rp.kind] : mp->kx[rp.kind]) + rp.idx;
            const int S = a.kps[rp.kind];
            digest_rows<K>(
                Id,
                [&](int r, int e, bool second) {
                  const unsigned f = (second ? fd : fc) + e, fr = r < K::NCA ? bfa + r : bfb + (r - K::NCA);
                  return rp.sign * x[(size_t)(rp.colwise ? f + fr * N : fr + f * N) * S];
                },
                s_k + p * NROW * w, w, c, d);
          }
        }
      for (int p = 0; p < a.nj; ++p) {
        // J(a, b) += I X(d, c) over the wave, J(d, c) += I X(a, b) (direct.hpp:1863-1883, 1925-1960)
        const bool on = take && ((mask >> a.jmat[p]) & 1u);
        double x[NCD];
#pragma unroll
        for (int e = 0; e < NCD; ++e) x[e] = on ? a.jx_ket[(size_t)(p * NCD + e) * a.nket + j] : 0.0;
        double t[NCD];
#pragma unroll
        for (int e = 0; e < NCD; ++e) t[e] = 0.0;
        // J(a, b) sums formed together (a divisor of NAB)
        constexpr int NS = NAB <= 10 ? NAB : NAB % 9 == 0 ? 9 : NAB % 10 == 0 ? 10 : 5;
#pragma unroll
        for (int ab0 = 0; ab0 < NAB; ab0 += NS) {
          double s[NS];
#pragma unroll
          for (int k = 0; k < NS; ++k) {
            const int ab = ab0 + k;
            const double xab = as_const(a.jx_bra)[(size_t)(p * NAB + ab) * a.nbra + i];
            s[k] = 0.0;
#pragma unroll
            for (int e = 0; e < NCD; ++e) {
              s[k] = fma(Id[ab * NCD + e], x[e], s[k]);
              t[e] = fma(Id[ab * NCD + e], xab, t[e]);
            }
          }
          wave_sums_add<NS, 32>(s, 0, NS, s_jab + p * NAB + ab0, lane);
        }
        if (on)
#pragma unroll
          for (int e = 0; e < NCD; ++e)
            unsafeAtomicAdd(a.ja_ket + (size_t)(p * NCD + e) * a.nket + j, a.jcoef[p] * t[e]);
      }
    }
    __syncthreads();
    // rows and J(a, b) out
    for (int p = 0; p < a.nk; ++p) {
      const RowPlane &rp = a.k[p];
      GlobalDouble *acc = (GlobalDouble *)(one ? a.m0.ka[rp.kind] : mp->ka[rp.kind]) + rp.idx;
      const int S = a.kps[rp.kind];
      const double *ks = s_k + p * NROW * w;
      const double coef = 0.5 * rp.sign;
      for (int c = tid; c < w; c += nthread) {
        const int f = colmap[c];
        if (f < 0) continue;
#pragma unroll
        for (int r = 0; r < NROW; ++r) {
          const int fr = r < K::NCA ? bfa + r : bfb + (r - K::NCA);
          const double v = ks[r * w + c];
          if (v != 0.0)
            __builtin_amdgcn_global_atomic_fadd_f64(
                acc + (size_t)(rp.colwise ? f + (size_t)fr * N : fr + (size_t)f * N) * S, coef * v);
        }
      }
    }
    for (int e = tid; e < a.nj * NAB; e += nthread) {
      const double v = s_jab[e];
      if (v != 0.0) unsafeAtomicAdd(a.ja_bra + (size_t)e * a.nbra + i, a.jcoef[e / NAB] * v);
    }
  }
  __syncthreads();
  if (tid == 0) {
    if (s_tot[0]) atomicAdd(a.count, s_tot[0]);
    if (s_tot[1]) atomicAdd(a.count + 1, s_tot[1]);
    if (s_psum != 0.0) unsafeAtomicAdd(a.prim_sum, s_psum);
  }
}

// LDS of a block in bytes: the static arrays (with padding), the exchange rows
// and, with XL, the density rows
template <class K, class R, bool XL>
size_t row_lds(int nk, int width) {
  const size_t fixed = sizeof(R) * RysRow<K::NR, R, K::NC == 1, XL>::kLen + 4 * (kRowChunk + kRowBuckets) + 8 * kRowJ * K::NCA * K::NCB + 256;
  return fixed + (size_t)(XL ? 2 : 1) * nk * (K::NCA + K::NCB) * width * sizeof(double);
}

constexpr long long kRowGrid = 8192;

// Threads of a block of the launch: the size that keeps more wavefronts on a
// CU, as its registers (of the kernel) and LDS allow; the smaller of two that
// keep as many, since its blocks screen while others evaluate.  C40H82 / 6-31G(d), ms a
// launch, 256 and 512 threads: (ss|ss), equal wavefronts, 2.18 and 2.27;
// (pp|ps), with rows that leave room for two blocks, 1.07 and 1.23; with rows
// that leave room for one (dp|ps) 1.67 and 1.38, (dd|ss) 0.61 and 0.45; 32
// water clusters, mixed, 26.7 -> 22.3 ms a build.  A launch of few items
// leaves CUs idle whatever the size and takes the larger one ((H2O)4 /
// cc-pVDZ, up to 406 items a launch, 0.69 -> 0.61 ms a build; with the line
// at 1024 the launches of (H2O)6 / cc-pVTZ lose, 9.39 -> 9.60).
constexpr long long kRowFew = 512;
inline int row_block(int most, int vgprs, size_t lds, long long items) {
  if (most <= 256 || items <= kRowFew) return most;
  const int per_cu = 4 * std::min(8, 512 / ((std::max(vgprs, 1) + 7) / 8 * 8));  // wavefronts
  auto waves = [&](int n) { return std::min<int>((int)(kRowLdsMax / lds), per_cu / (n / 64)) * (n / 64); };
  return waves(512) > waves(256) ? 512 : 256;
}

template <int LA, int LB, int LC, int LD, class R, bool XL>
hipError_t launch_row_x(const RowLaunch &a, hipStream_t s) {
  using K = Cls<LA, LB, LC, LD>;
  auto kern = eri_row_kernel<LA, LB, LC, LD, R, XL>;
  static std::once_flag once;  // allow dynamic LDS beyond the default limit, once per instantiation
  static hipError_t attr = hipSuccess;
  static int vgprs = 0;
  std::call_once(once, [&] {
    hipFuncAttributes fa{};
    attr = hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(kern));
    if (attr != hipSuccess) return;
    vgprs = fa.numRegs;
    attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(kRowLdsMax - row_lds<K, R, XL>(0, 0)));
  });
  if (attr != hipSuccess) return attr;
  const long long items = (long long)a.nbra * a.nchunk;
  const size_t dyn = (size_t)(XL ? 2 : 1) * a.nk * (K::NCA + K::NCB) * a.width * sizeof(double);
  hipLaunchKernelGGL(kern, dim3((unsigned)(items < kRowGrid ? items : kRowGrid)), dim3(row_block(row_threads<K>(), vgprs, row_lds<K, R, XL>(a.nk, a.width), items)), dyn, s, a);
  return hipGetLastError();
}

template <int LA, int LB, int LC, int LD, class R>
hipError_t launch_row_cls(const RowLaunch &a, hipStream_t s) {
  using K = Cls<LA, LB, LC, LD>;
  if ((long long)a.nbra * a.nchunk <= 0) return hipSuccess;
  // density rows in LDS where both sets fit: GHF (H2O)16 (eight planes)
  // takes the second form for (ps|ps) and up, 11.5 -> 9.4 ms a build with it
  if (row_lds<K, R, true>(a.nk, a.width) <= kRowLdsMax) return launch_row_x<LA, LB, LC, LD, R, true>(a, s);
  if (row_lds<K, R, false>(a.nk, a.width) <= kRowLdsMax) return launch_row_x<LA, LB, LC, LD, R, false>(a, s);
  return hipErrorInvalidValue;
}

template <int LA, int LB, int LC, int LD>
hipError_t launch_row_prec(const RowLaunch &a, hipStream_t s) {
  if (!a.fp32) return launch_row_cls<LA, LB, LC, LD, double>(a, s);
  if constexpr (LA <= 2) return launch_row_cls<LA, LB, LC, LD, float>(a, s);
  return hipErrorInvalidValue;
}

}  // namespace

// classes with a row kernel, in groups that compile apart
#define CQX_ROW_CLASSES_A(X) X(0, 0, 0, 0) X(1, 0, 0, 0) X(1, 0, 1, 0) X(1, 1, 0, 0) X(2, 0, 0, 0) X(1, 1, 1, 0)
#define CQX_ROW_CLASSES_B(X) X(2, 0, 1, 0) X(2, 1, 0, 0) X(2, 0, 2, 0) X(2, 2, 0, 0) X(2, 1, 1, 0)
#define CQX_ROW_CLASSES_C(X) X(2, 0, 1, 1) X(1, 1, 1, 1) X(2, 1, 2, 0) X(2, 2, 1, 0)
// with an f or g shell, up to 45 components (FP64 only, as their quartet
// lists): (fs|ss) of (H2O)6 / cc-pVTZ 0.61 ms on the wave kernel, 0.21 here,
// but (fs|ds) 0.25 and 0.60: beyond, a block holds one wave per SIMD
#define CQX_ROW_CLASSES_D(X) \
  X(3, 0, 0, 0) X(3, 0, 1, 0) X(3, 1, 0, 0) X(4, 0, 0, 0) X(4, 0, 1, 0) X(4, 1, 0, 0)

template <int GROUP>
hipError_t launch_row_group(const RowLaunch &a, hipStream_t s);
template <int GROUP>
bool row_group_lds(int la, int lb, int lc, int ld, int fp32, int nk, int width, size_t &bytes);

#define CQX_ROW_GROUP(GROUP, LIST)                                                                         \
  template <>                                                                                              \
  hipError_t launch_row_group<GROUP>(const RowLaunch &a, hipStream_t s) {                                  \
    LIST(CQX_ROW_LAUNCH) return hipErrorNotSupported;                                                      \
  }                                                                                                        \
  template <>                                                                                              \
  bool row_group_lds<GROUP>(int la, int lb, int lc, int ld, int fp32, int nk, int width, size_t &bytes) {  \
    LIST(CQX_ROW_LDS) return false;                                                                        \
  }
#define CQX_ROW_LAUNCH(A, B, C, D)                          \
  if (a.la == A && a.lb == B && a.lc == C && a.ld == D)     \
    return launch_row_prec<A, B, C, D>(a, s);
#define CQX_ROW_LDS(A, B, C, D)                                             \
  if (la == A && lb == B && lc == C && ld == D) {                           \
    bytes = fp32 ? row_lds<Cls<A, B, C, D>, float, false>(nk, width)               \
                 : row_lds<Cls<A, B, C, D>, double, false>(nk, width);             \
    return true;                                                            \
  }

}  // namespace cqx
