// Gradient kernels of the s/p/d classes, templated on the class.
//
// The generic kernel (grad.hip) builds one primitive quartet at a time with
// 3 n_r of 64 lanes busy and run-time sizes (private arrays in scratch):
// (ss|ss) of (H2O)3 / cc-pVDZ took 24.1 ms for 23005 quartets, whose longest
// have 4096 primitive quartets one after the other, and adds each integral
// to HBM once per update.  Two forms replace it:
// - up to 9 Cartesian components, G lanes split the primitive quartets, each
//   with its 2D integrals and the derivative sums of one centre at a time in
//   registers ((ss|ss) 24.1 -> 0.19 ms, (ps|ss) 16.3 -> 0.43 ms);
// - beyond, one wave (four above 200 components) per quartet builds the 2D
//   tables of several primitive quartets in LDS and each thread keeps its
//   components ((dp|ps) 2.5 -> 0.16 ms, (dp|pp) 2.1 -> 0.16, (dd|dd) 0.83 ->
//   0.04; the register form took 2.2 ms for (dp|ps), in nine passes).
// Both then form every J / K target of the twelve derivative quartets from
// LDS and add it once.  getGDGrad of (H2O)3 / cc-pVDZ: 94 -> 4.1 ms.
#pragma once

#include <hip/hip_runtime.h>

#include "digest.hpp"
#include "eri_class.hpp"
#include "kernels.hpp"

namespace cqx {

namespace {

template <int LA, int LB, int LC, int LD>
struct GradCls {
  using K = Cls<LA, LB, LC, LD>;
  static constexpr int NR = (LA + LB + LC + LD + 1) / 2 + 1;  // one more unit of angular momentum
  // lanes per quartet: all of them for the classes with the longest
  // contractions (64 primitive pairs a side in cc-pVDZ's oxygen s shells)
  static constexpr int G = K::NC <= 3 ? 64 : 16;
};

// 2D integrals of one root and direction with centre C of (A, B, C) raised
// by one; f(...) of the plain and derivative factors reads them by constants
template <int LA, int LB, int LC, int LD, int CEN>
struct Raised {
  static constexpr int A = LA + (CEN == 0), B = LB + (CEN == 1), C = LC + (CEN == 2), D = LD;
  static constexpr int NH = (A + 1) * (B + 1) * (C + 1) * (D + 1);
  static constexpr int at(int a, int b, int c, int d) { return ((a * (B + 1) + b) * (C + 1) + c) * (D + 1) + d; }
};

// Sums over the lane's primitive quartets (flattened index k = g, g + G, ...)
// of the derivatives of centre CEN along the three directions.
template <int LA, int LB, int LC, int LD, int CEN>
__device__ __forceinline__ void grad_pass(const GradLaunch &a, const double *__restrict__ tab, const PairRec &bp,
                                          const PairRec &kp, int g, int G,
                                          double (&acc)[3][Cls<LA, LB, LC, LD>::NC]) {
  using K = Cls<LA, LB, LC, LD>;
  using H = Raised<LA, LB, LC, LD, CEN>;
  constexpr int NR = GradCls<LA, LB, LC, LD>::NR;
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int o = 0; o < K::NC; ++o) acc[t][o] = 0.0;
  const int nk = kp.npp, ntot = bp.npp * nk;
  for (int k = g; k < ntot; k += G) {
    const int i = k / nk, j = k - i * nk;
    const PrimPair P = a.prims[bp.pp_off + i], Q = a.prims[kp.pp_off + j];
    const double ala = a.prim_alpha[bp.pp_off + i];
    const double two = 2.0 * (CEN == 0 ? ala : CEN == 1 ? P.p - ala : a.prim_alpha[kp.pp_off + j]);
    const double r = eval_rsqrt<double>(P.p + Q.p), rpq = r * r;
    const double aq = P.p * rpq, bq = Q.p * rpq;
    const double PQ[3] = {P.P[0] - Q.P[0], P.P[1] - Q.P[1], P.P[2] - Q.P[2]};
    const double T = P.p * bq * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
    const double pref = P.K * Q.K * kTwoPi52 * P.rp * Q.rp * r;
    // one root at a time: unrolled, the 2D integrals of all roots are live together
#pragma unroll 1
    for (int n = 0; n < NR; ++n) {
      double t2, wt;
      rys_root_sec<NR, double>(T, tab, n, t2, wt);
      const double B00 = 0.5 * t2 * rpq, B10 = 0.5 * P.rp * (1.0 - bq * t2), B01 = 0.5 * Q.rp * (1.0 - aq * t2);
      double h[3][H::NH];
#pragma unroll
      for (int d = 0; d < 3; ++d)
        rys_2d_full<H::A, H::B, H::C, H::D, double>(P.P[d] - bp.A[d] - bq * t2 * PQ[d],
                                                    Q.P[d] - kp.A[d] + aq * t2 * PQ[d], B10, B01, B00, bp.AB[d],
                                                    kp.AB[d], d == 2 ? pref * wt : 1.0, h[d]);
#pragma unroll
      for (int ia = 0; ia < K::NCA; ++ia)
#pragma unroll
        for (int ib = 0; ib < K::NCB; ++ib)
#pragma unroll
          for (int ic = 0; ic < K::NCC; ++ic)
#pragma unroll
            for (int id = 0; id < K::NCD; ++id) {
              double f[3], df[3];
#pragma unroll
              for (int d = 0; d < 3; ++d) {
                const int e0 = cexp(LA, ia, d), e1 = cexp(LB, ib, d), e2 = cexp(LC, ic, d), e3 = cexp(LD, id, d);
                const int ec = CEN == 0 ? e0 : CEN == 1 ? e1 : e2;
                f[d] = h[d][H::at(e0, e1, e2, e3)];
                df[d] = two * h[d][H::at(e0 + (CEN == 0), e1 + (CEN == 1), e2 + (CEN == 2), e3)];
                if (ec) df[d] -= ec * h[d][H::at(e0 - (CEN == 0), e1 - (CEN == 1), e2 - (CEN == 2), e3)];
              }
              const int o = K::oidx(ia, ib, ic, id);
              acc[0][o] = fma(df[0], f[1] * f[2], acc[0][o]);
              acc[1][o] = fma(df[1], f[0] * f[2], acc[1][o]);
              acc[2][o] = fma(df[2], f[0] * f[1], acc[2][o]);
            }
    }
  }
}

// One centre, summed over the group and written (scaled) to the
// quartet's derivative arrays sd[centre 3 + direction][component].
template <int LA, int LB, int LC, int LD, int CEN>
__device__ __forceinline__ void grad_centre(const GradLaunch &a, const double *__restrict__ tab, const PairRec &bp,
                                            const PairRec &kp, int g, double scale, double *sd) {
  using K = Cls<LA, LB, LC, LD>;
  using GC = GradCls<LA, LB, LC, LD>;
  double acc[3][K::NC];
  grad_pass<LA, LB, LC, LD, CEN>(a, tab, bp, kp, g, GC::G, acc);
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int o = 0; o < K::NC; ++o) {
      double v = acc[t][o];
#pragma unroll
      for (int off = GC::G / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
      if (o % GC::G == g) sd[(CEN * 3 + t) * K::NC + o] = scale * v;
    }
}

// Targets A(ar, ac) += coef sum D(t) X(xr, xc) of one update term for the
// twelve derivative quartets, over the G lanes of the group.
template <class K, int G, int AR, int AC, int XR, int XC>
__device__ __forceinline__ void grad_term(const double *sd, const int (&bf)[4], const int (&coord)[4],
                                          const GradLaunch &a, int m, double coef, int g) {
  constexpr int NT = K::n(AR) * K::n(AC);
  constexpr int ST[4] = {K::NCB * K::NCC * K::NCD, K::NCC * K::NCD, K::NCD, 1};
  const int N = a.nbc;
  const size_t n2 = (size_t)N * N;
  const double *__restrict__ X = a.X + (size_t)m * n2 + bf[XR] + (size_t)bf[XC] * N;
  for (int it = g; it < 12 * NT; it += G) {
    const int t = it / NT, tgt = it - t * NT;
    const int t1 = tgt / K::n(AR), t0 = tgt - t1 * K::n(AR);
    const double *I = sd + t * K::NC + t0 * ST[AR] + t1 * ST[AC];
    double v = 0.0;
#pragma unroll
    for (int u1 = 0; u1 < K::n(XC); ++u1)
#pragma unroll
      for (int u0 = 0; u0 < K::n(XR); ++u0) v = fma(I[u0 * ST[XR] + u1 * ST[XC]], X[u0 + (size_t)u1 * N], v);
    if (v == 0.0) continue;
    const int cen = t / 3, dir = t - cen * 3;
    const int c3 = cen == 0 ? coord[0] : cen == 1 ? coord[1] : cen == 2 ? coord[2] : coord[3];
    unsafeAtomicAdd(a.acc + ((size_t)(c3 + dir) * a.nmat + m) * n2 + bf[AR] + t0 + (size_t)(bf[AC] + t1) * N,
                    coef * v);
  }
}

// Every update of the twelve derivative quartets sd by G threads.
template <class K, int G>
__device__ __forceinline__ void grad_digest(const double *sd, const PairRec &bp, const PairRec &kp,
                                            const GradLaunch &a, int g) {
  const int bf[4] = {bp.bfa, bp.bfb, kp.bfa, kp.bfb};
  const int coord[4] = {3 * a.shell_atom[bp.a], 3 * a.shell_atom[bp.b], 3 * a.shell_atom[kp.a],
                        3 * a.shell_atom[kp.b]};
  for (int m = 0; m < a.nmat; ++m) {
    if (!((a.kmask >> m) & 1u)) {  // direct.hpp:2450-2470
      grad_term<K, G, 0, 1, 3, 2>(sd, bf, coord, a, m, 1.0, g);
      grad_term<K, G, 3, 2, 0, 1>(sd, bf, coord, a, m, 1.0, g);
    } else {  // :2471-2497
      grad_term<K, G, 0, 2, 3, 1>(sd, bf, coord, a, m, 0.5, g);
      grad_term<K, G, 3, 1, 0, 2>(sd, bf, coord, a, m, 0.5, g);
      grad_term<K, G, 3, 0, 1, 2>(sd, bf, coord, a, m, 0.5, g);
      grad_term<K, G, 1, 2, 3, 0>(sd, bf, coord, a, m, 0.5, g);
    }
  }
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void grad_lane_kernel(GradLaunch a) {
  using K = Cls<LA, LB, LC, LD>;
  using GC = GradCls<LA, LB, LC, LD>;
  constexpr int G = GC::G, QPW = 64 / G;
  __shared__ double s_d[4 * QPW][12 * K::NC];
  __shared__ double s_tab[rys_tab_len(GC::NR)];
  for (int e = threadIdx.x; e < rys_tab_len(GC::NR); e += 256) s_tab[e] = a.rys[rys_tab_off(GC::NR) + e];
  __syncthreads();
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane & (G - 1);
  const int slot = wv * QPW + lane / G;
  double *sd = s_d[slot];
  const long long per = 4 * QPW, nround = (a.nq + per - 1) / per;
  for (long long round = blockIdx.x; round < nround; round += gridDim.x) {
    const long long q = round * per + slot;
    const bool valid = q < a.nq;
    int i = 0, j = 0;
    if (valid) {
      if (a.same_class) {  // j <= i, row-major lower triangle
        long long r = (long long)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
        while (r * (r + 1) / 2 > q) --r;
        while ((r + 1) * (r + 2) / 2 <= q) ++r;
        i = (int)r;
        j = (int)(q - r * (r + 1) / 2);
      } else {
        i = (int)(q / a.nket);
        j = (int)(q - (long long)i * a.nket);
      }
    }
    PairRec bp = a.bra[i], kp = a.ket[j];
    if (!valid) bp.npp = 0;
    // degeneracy of the quartet in the 8-fold loop and the 1/2 (direct.hpp:2382-2388)
    const bool same_pair = bp.a == kp.a && bp.b == kp.b;
    const double scale = 0.5 * (bp.a == bp.b ? 1.0 : 2.0) * (kp.a == kp.b ? 1.0 : 2.0) * (same_pair ? 1.0 : 2.0);
    grad_centre<LA, LB, LC, LD, 0>(a, s_tab, bp, kp, g, scale, sd);
    grad_centre<LA, LB, LC, LD, 1>(a, s_tab, bp, kp, g, scale, sd);
    grad_centre<LA, LB, LC, LD, 2>(a, s_tab, bp, kp, g, scale, sd);
    wave_sync();
    // centre D from translational invariance
    for (int e = g; e < 3 * K::NC; e += G) sd[9 * K::NC + e] = -(sd[e] + sd[3 * K::NC + e] + sd[6 * K::NC + e]);
    wave_sync();
    if (valid) grad_digest<K, G>(sd, bp, kp, a, g);
    wave_sync();  // the next round rewrites the derivative arrays
  }
}

template <int LA, int LB, int LC, int LD>
hipError_t launch_grad_cls(const GradLaunch &a, hipStream_t s) {
  constexpr long long per = 4 * (64 / GradCls<LA, LB, LC, LD>::G);
  const long long rounds = (a.nq + per - 1) / per;
  hipLaunchKernelGGL((grad_lane_kernel<LA, LB, LC, LD>), dim3((unsigned)(rounds < 65536 ? rounds : 65536)), dim3(256),
                     0, s, a);
  return hipGetLastError();
}

// The larger s/p/d classes: NT threads take one quartet.  Lanes (primitive
// quartet of the round, root, direction) build the 2D integrals raised by
// one on A, B and C into LDS from registers; every thread then adds the
// round to the nine derivative sums of its components, kept in LDS.
template <int LA, int LB, int LC, int LD>
struct GradWave {
  using K = Cls<LA, LB, LC, LD>;
  static constexpr int NR = (LA + LB + LC + LD + 1) / 2 + 1;
  static constexpr int SC = LD + 1, SB = (LC + 2) * SC, SA = (LB + 2) * SB, NH = (LA + 2) * SA;
  static constexpr int NT = K::NC > 200 ? 256 : 64;
  static constexpr int by_lanes = NT / (3 * NR), by_lds = 24576 / (3 * NR * NH * 8);
  static constexpr int PP = by_lanes < by_lds ? by_lanes : (by_lds > 0 ? by_lds : 1);
};

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__((GradWave<LA, LB, LC, LD>::NT)) void grad_wave_kernel(GradLaunch a) {
  using K = Cls<LA, LB, LC, LD>;
  using W = GradWave<LA, LB, LC, LD>;
  __shared__ double s_h[W::PP][3 * W::NR][W::NH];
  __shared__ double s_two[W::PP][3];
  __shared__ double s_d[12 * K::NC];
  const int tid = threadIdx.x;
  const double *tab = a.rys + rys_tab_off(W::NR);
  for (long long q = blockIdx.x; q < a.nq; q += gridDim.x) {
    int i, j;
    if (a.same_class) {  // j <= i, row-major lower triangle
      long long r = (long long)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
      while (r * (r + 1) / 2 > q) --r;
      while ((r + 1) * (r + 2) / 2 <= q) ++r;
      i = (int)r;
      j = (int)(q - r * (r + 1) / 2);
    } else {
      i = (int)(q / a.nket);
      j = (int)(q - (long long)i * a.nket);
    }
    const PairRec bp = a.bra[i], kp = a.ket[j];
    const int nk = kp.npp, ntot = bp.npp * nk;
    if (ntot == 0) continue;  // (the barriers between clearing and reading the sums are those of the loop below)
    for (int e = tid; e < 9 * K::NC; e += W::NT) s_d[e] = 0.0;
    const int grp = tid / (3 * W::NR), sub = tid - grp * (3 * W::NR), root = sub / 3, d = sub - root * 3;
    for (int k0 = 0; k0 < ntot; k0 += W::PP) {
      const int cnt = min(W::PP, ntot - k0);
      if (grp < cnt) {
        const int pi = (k0 + grp) / nk, pj = k0 + grp - pi * nk;
        const PrimPair P = a.prims[bp.pp_off + pi], Q = a.prims[kp.pp_off + pj];
        const double ala = a.prim_alpha[bp.pp_off + pi];
        const double r = eval_rsqrt<double>(P.p + Q.p), rpq = r * r;
        const double aq = P.p * rpq, bq = Q.p * rpq;
        const double PQ[3] = {P.P[0] - Q.P[0], P.P[1] - Q.P[1], P.P[2] - Q.P[2]};
        const double T = P.p * bq * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
        const double pref = P.K * Q.K * kTwoPi52 * P.rp * Q.rp * r;
        double t2, w;
        rys_root_sec<W::NR, double>(T, tab, root, t2, w);
        const double PQd = d == 0 ? PQ[0] : d == 1 ? PQ[1] : PQ[2];
        const double Pd = d == 0 ? P.P[0] - bp.A[0] : d == 1 ? P.P[1] - bp.A[1] : P.P[2] - bp.A[2];
        const double Qd = d == 0 ? Q.P[0] - kp.A[0] : d == 1 ? Q.P[1] - kp.A[1] : Q.P[2] - kp.A[2];
        const double AB = d == 0 ? bp.AB[0] : d == 1 ? bp.AB[1] : bp.AB[2];
        const double CD = d == 0 ? kp.AB[0] : d == 1 ? kp.AB[1] : kp.AB[2];
        double h[W::NH];
        rys_2d_full<LA + 1, LB + 1, LC + 1, LD, double>(Pd - bq * t2 * PQd, Qd + aq * t2 * PQd,
                                                        0.5 * P.rp * (1.0 - bq * t2), 0.5 * Q.rp * (1.0 - aq * t2),
                                                        0.5 * t2 * rpq, AB, CD, d == 2 ? pref * w : 1.0, h);
#pragma unroll
        for (int e = 0; e < W::NH; ++e)
          if (!(e / W::SA == LA + 1 && e / W::SB % (LB + 2) == LB + 1)) s_h[grp][sub][e] = h[e];  // not both raised
        if (sub == 0) {
          s_two[grp][0] = 2.0 * ala;
          s_two[grp][1] = 2.0 * (P.p - ala);
          s_two[grp][2] = 2.0 * a.prim_alpha[kp.pp_off + pj];
        }
      }
      __syncthreads();
      for (int o = tid; o < K::NC; o += W::NT) {
        int rem = o;
        const int id = rem % K::NCD; rem /= K::NCD;
        const int ic = rem % K::NCC; rem /= K::NCC;
        const int ib = rem % K::NCB;
        const int ia = rem / K::NCB;
        int at[3], e0[3], e1[3], e2[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) {
          e0[u] = cexp(LA, ia, u);
          e1[u] = cexp(LB, ib, u);
          e2[u] = cexp(LC, ic, u);
          at[u] = e0[u] * W::SA + e1[u] * W::SB + e2[u] * W::SC + cexp(LD, id, u);
        }
        double acc[9] = {};
        for (int g = 0; g < cnt; ++g) {
          const double twa = s_two[g][0], twb = s_two[g][1], twc = s_two[g][2];
#pragma unroll 1
          for (int r = 0; r < W::NR; ++r) {
            double f[3], df[3][3];
#pragma unroll
            for (int u = 0; u < 3; ++u) {
              const double *h = s_h[g][3 * r + u] + at[u];
              f[u] = h[0];
              df[0][u] = fma(twa, h[W::SA], -e0[u] * h[e0[u] ? -W::SA : 0]);
              df[1][u] = fma(twb, h[W::SB], -e1[u] * h[e1[u] ? -W::SB : 0]);
              df[2][u] = fma(twc, h[W::SC], -e2[u] * h[e2[u] ? -W::SC : 0]);
            }
            const double yz = f[1] * f[2], xz = f[0] * f[2], xy = f[0] * f[1];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              acc[3 * c] = fma(df[c][0], yz, acc[3 * c]);
              acc[3 * c + 1] = fma(df[c][1], xz, acc[3 * c + 1]);
              acc[3 * c + 2] = fma(df[c][2], xy, acc[3 * c + 2]);
            }
          }
        }
#pragma unroll
        for (int t = 0; t < 9; ++t) s_d[t * K::NC + o] += acc[t];
      }
      __syncthreads();
    }
    const bool same_pair = bp.a == kp.a && bp.b == kp.b;
    const double scale = 0.5 * (bp.a == bp.b ? 1.0 : 2.0) * (kp.a == kp.b ? 1.0 : 2.0) * (same_pair ? 1.0 : 2.0);
    for (int e = tid; e < 3 * K::NC; e += W::NT) {  // scaled; centre D from translational invariance
      const double x = scale * s_d[e], y = scale * s_d[3 * K::NC + e], z = scale * s_d[6 * K::NC + e];
      s_d[e] = x;
      s_d[3 * K::NC + e] = y;
      s_d[6 * K::NC + e] = z;
      s_d[9 * K::NC + e] = -(x + y + z);
    }
    __syncthreads();
    grad_digest<K, W::NT>(s_d, bp, kp, a, tid);
    __syncthreads();
  }
}

template <int LA, int LB, int LC, int LD>
hipError_t launch_grad_wave(const GradLaunch &a, hipStream_t s) {
  hipLaunchKernelGGL((grad_wave_kernel<LA, LB, LC, LD>), dim3((unsigned)(a.nq < 65536 ? a.nq : 65536)),
                     dim3(GradWave<LA, LB, LC, LD>::NT), 0, s, a);
  return hipGetLastError();
}

}  // namespace

// classes of these kernels, in groups that compile apart
#define CQX_GRAD_CLASSES_0(X, Y) \
  X(0, 0, 0, 0) X(1, 0, 0, 0) X(1, 0, 1, 0) X(1, 1, 0, 0) X(2, 0, 0, 0) Y(1, 1, 1, 0) Y(2, 0, 1, 0)
#define CQX_GRAD_CLASSES_1(X, Y) Y(2, 1, 0, 0) Y(2, 0, 2, 0) Y(2, 2, 0, 0) Y(2, 1, 1, 0) Y(2, 0, 1, 1) Y(1, 1, 1, 1)
#define CQX_GRAD_CLASSES_2(X, Y) Y(2, 1, 2, 0) Y(2, 2, 1, 0) Y(2, 1, 1, 1) Y(2, 2, 2, 0)
#define CQX_GRAD_CLASSES_3(X, Y) Y(2, 1, 2, 1) Y(2, 2, 1, 1) Y(2, 2, 2, 1) Y(2, 2, 2, 2)

template <int GROUP>
hipError_t launch_grad_group(const GradLaunch &a, hipStream_t s);

#define CQX_GRAD_CASE(A, B, C, D) \
  if (a.la == A && a.lb == B && a.lc == C && a.ld == D) return launch_grad_cls<A, B, C, D>(a, s);
#define CQX_GRAD_WCASE(A, B, C, D) \
  if (a.la == A && a.lb == B && a.lc == C && a.ld == D) return launch_grad_wave<A, B, C, D>(a, s);
#define CQX_GRAD_GROUP(GROUP)                                               \
  template <>                                                               \
  hipError_t launch_grad_group<GROUP>(const GradLaunch &a, hipStream_t s) { \
    CQX_GRAD_CLASSES_##GROUP(CQX_GRAD_CASE, CQX_GRAD_WCASE)                \
    return hipErrorNotSupported;                                           \
  }

}  // namespace cqx
