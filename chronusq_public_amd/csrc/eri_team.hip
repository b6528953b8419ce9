// Generic Rys ERI + J/K digestion kernel: one block per shell quartet (or
// part of one), any class through (gg|gg), sizes at run time except the
// second shell's angular momentum.
//
// An earlier form gave each quartet one 64-lane wave that built one
// primitive quartet at a time, with run-time indexed private arrays and
// three LDS reads per component and root: the three (gg|gg) quartets of
// (H2O)2 / cc-pVQZ took 11.4 ms, and (ss|ss) Schwarz diagonals with 4096
// primitive quartets 2 ms.  Here
// - lanes (primitive quartet, root, direction) run the vertical recursion
//   for as many primitive quartets at once as there are lanes and LDS; two
//   columns of it stay in registers;
// - the horizontal transfers are one sum per table entry,
//   (a b|c d) = sum_uv C(b,u) AB^(b-u) C(d,v) CD^(d-v) (a+u 0|c+v 0),
//   spread over all threads;
// - a thread takes (a component, ket component) and all components of b:
//   3 (lb + 1) LDS reads per root for (lb + 1)(lb + 2) / 2 components;
// - the quartet is digested by the block from LDS with each term's density
//   block staged there first.
// Measured, (H2O)2 / cc-pVQZ RHF J/K: (gg|gg) 11.4 -> 0.17 ms, (gg|gf) 6.1 ->
// 0.16, the build 43 -> 15.9 ms.  The wave kernels, built up to 1080
// components, win below ((H2O)6 / cc-pVTZ: (fd|dp) 0.27 against 0.52 ms,
// (dd|dp) 0.39 against 0.44).
//
// A quartet too large for LDS is split over ranges of its first shell's
// components, each a work item of its own (a is the slowest index of the
// layout and every J/K update is linear in the integrals), with the tables
// of a few roots at a time.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "digest.hpp"
#include "eri_class.hpp"
#include "kernels.hpp"
#include "rys.hpp"

namespace cqx {

namespace {

constexpr int kTeamI = 2 * kMaxLDev + 1;  // la + lb + 1 at most

struct TeamDims {
  int la, lb, lc, ld, nca, ncb, ncc, ncd, nket, ni, nk, nr, nh;
};
__host__ __device__ inline TeamDims team_dims(int la, int lb, int lc, int ld) {
  TeamDims d;
  d.la = la; d.lb = lb; d.lc = lc; d.ld = ld;
  d.nca = (la + 1) * (la + 2) / 2; d.ncb = (lb + 1) * (lb + 2) / 2;
  d.ncc = (lc + 1) * (lc + 2) / 2; d.ncd = (ld + 1) * (ld + 2) / 2;
  d.nket = d.ncc * d.ncd;
  d.ni = la + lb + 1;
  d.nk = lc + ld + 1;
  d.nr = (la + lb + lc + ld) / 2 + 1;
  d.nh = (la + 1) * (lb + 1) * (lc + 1) * (ld + 1);
  return d;
}

// Launch shape: components of the first shell per work item, roots per
// table group, primitive quartets per round, threads, and the doubles of the
// regions of dynamic LDS: vertical tables, full tables (both hold the
// density blocks afterwards), quartet.
struct TeamShape {
  int ca, rpp, pp, nt;
  int tab, quart;
};

// the fixed part of the LDS: HRR coefficients, component and entry tables
constexpr int kTeamCoef = 2 * 3 * 25;
constexpr int kTeamFixed = kTeamCoef * 8 + 15 * 4 + 225 * 4 + 640 * 2 + 64;

bool team_plan(const TeamDims &d, int lds_bytes, TeamShape &s) {
  const int nbcd = d.ncb * d.nket;
  s.nt = d.nca * d.nket <= 64 ? 64 : 256;
  // the staged density of one plane needs this much of the table region
  const int most = std::max(std::max(d.nca, d.ncb), std::max(d.ncc, d.ncd)), xneed = most * most;
  const int total = (lds_bytes - kTeamFixed) / 8;
  auto table = [&](int pp, int rpp) {
    return std::max(pp * (3 * d.nr * d.ni * d.nk + 3 * rpp * d.nh), xneed);
  };
  // half of the LDS at most for the quartet, a quarter when that still holds
  // a component of a, so that two blocks share a CU
  for (int share : {4, 2, 1}) {
    const int cap = total / share;
    s.ca = std::min(d.nca, (cap / 2) / nbcd);
    if (s.ca < 1) continue;
    // equal passes
    const int passes = (d.nca + s.ca - 1) / s.ca;
    s.ca = (d.nca + passes - 1) / passes;
    s.quart = s.ca * nbcd;
    s.rpp = d.nr;
    while (s.rpp > 1 && s.quart + table(1, s.rpp) > cap) --s.rpp;
    if (s.quart + table(1, s.rpp) > cap) continue;
    s.pp = std::max(1, s.nt / (3 * d.nr));
    while (s.pp > 1 && s.quart + table(s.pp, s.rpp) > cap) --s.pp;
    s.tab = table(s.pp, s.rpp);
    return true;
  }
  return false;
}

// One update term of the sub-quartet in sI (roles' sizes n, first functions
// bf): its density block for planes [p0, p0 + np) is staged, then every
// thread forms targets (plane fastest) and adds each once.
__device__ __forceinline__ void team_term(const double *sI, double *sX, const int (&n)[4], const int (&bf)[4],
                                          const int (&st)[4], const PlaneSet &ps, const MolPlanes &mp, int kind,
                                          int p0, int np, int ar, int ac, int xr, int xc, double base,
                                          unsigned mask, int tid, int NT) {
  const int N = mp.nbc, S = ps.kps[kind], first = ps.kstart[kind];
  const double *xk = mp.kx[kind];
  double *ak = mp.ka[kind];
  const int nxr = n[xr], nxc = n[xc], nx = nxr * nxc;
  __syncthreads();  // the previous term's block has been read
  for (int e = tid; e < nx * np; e += NT) {
    const int p = e % np, k = e / np, r = k % nxr, c = k / nxr;
    sX[e] = xk[(p0 + p) + ((size_t)(bf[xr] + r) + (size_t)(bf[xc] + c) * N) * S];
  }
  __syncthreads();
  const int nar = n[ar], nt = nar * n[ac];
  for (int t = tid; t < nt * np; t += NT) {
    const int p = t % np, tgt = t / np, t0 = tgt % nar, t1 = tgt / nar;
    const Plane &P = ps.p[first + p0 + p];
    if (!((mask >> P.mat) & 1u)) continue;
    const double *Ib = sI + t0 * st[ar] + t1 * st[ac];
    const double *Xb = sX + p;
    double s0 = 0.0, s1 = 0.0;
    for (int c = 0; c < nxc; ++c) {
      const double *Iu = Ib + c * st[xc];
      const double *Xu = Xb + c * nxr * np;
      int r = 0;
      for (; r + 1 < nxr; r += 2) {
        s0 = fma(Iu[r * st[xr]], Xu[r * np], s0);
        s1 = fma(Iu[(r + 1) * st[xr]], Xu[(r + 1) * np], s1);
      }
      if (r < nxr) s0 = fma(Iu[r * st[xr]], Xu[r * np], s0);
    }
    const double coef = kind == kKHer ? base * P.sign : base;
    unsafeAtomicAdd(ak + (p0 + p) + ((size_t)(bf[ar] + t0) + (size_t)(bf[ac] + t1) * N) * S, coef * (s0 + s1));
  }
}

template <int LB, int NT>
__global__ __launch_bounds__(NT) void eri_team_kernel(EriLaunch a, TeamShape sh) {
  constexpr int NCB = ncart_c(LB);
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const TeamDims D = team_dims(a.la, LB, a.lc, a.ld);
  double *s_ab = lds, *s_cd = lds + 75;  // C(b, u) AB^(b - u) per direction, and of the ket
  double *s_tab = lds + kTeamCoef;
  double *s_I = s_tab + sh.tab;
  unsigned *s_pa = reinterpret_cast<unsigned *>(s_I + sh.quart);  // table offsets of a's components
  unsigned *s_pk = s_pa + 15;                                      // of the ket components
  unsigned short *s_dec = reinterpret_cast<unsigned short *>(s_pk + 225);  // exponents of a table entry
  const int sc = D.ld + 1, sb = (D.lc + 1) * sc, sa = (LB + 1) * sb;
  const int GN = D.ni * D.nk;
  for (int e = tid; e < D.nca; e += NT)
    s_pa[e] = (unsigned)(cexp(D.la, e, 0) * sa) | ((unsigned)(cexp(D.la, e, 1) * sa) << 10) |
              ((unsigned)(cexp(D.la, e, 2) * sa) << 20);
  for (int e = tid; e < D.nket; e += NT) {
    const int ic = e / D.ncd, id = e - ic * D.ncd;
    unsigned v = 0;
    for (int d = 0; d < 3; ++d) v |= (unsigned)(cexp(D.lc, ic, d) * sc + cexp(D.ld, id, d)) << (10 * d);
    s_pk[e] = v;
  }
  for (int e = tid; e < D.nh; e += NT) {
    const int xd = e % sc, xc = e / sc % (D.lc + 1), xb = e / sb % (LB + 1), xa = e / sa;
    s_dec[e] = (unsigned short)(xa | (xb << 4) | (xc << 8) | (xd << 12));
  }
  // quartet count: the list's device counter for a launch sized to the
  // list's capacity before the list was built
  const long long nq = a.nq_dev ? min((long long)*a.nq_dev - a.nq_base, a.nq) : a.nq;
  const int npass = (D.nca + sh.ca - 1) / sh.ca;
  const int grp = tid / (3 * D.nr), sub = tid - grp * (3 * D.nr), root = sub / 3, dir = sub - root * 3;
  for (long long w = blockIdx.x; w < nq * npass; w += gridDim.x) {
    const long long q = w / npass;
    const int ia0 = (int)(w - q * npass) * sh.ca, na = min(sh.ca, D.nca - ia0);
    const Quartet qt = a.quartets[q];
    const PairRec &bp = a.bra[qt.bra];
    const PairRec &kp = a.ket[qt.ket_mask & 0xFFFFFFu];
    const int nkp = kp.npp, ntot = bp.npp * nkp;
    const int nbcd = NCB * D.nket, nsub = na * nbcd;
    __syncthreads();  // the previous item's quartet has been read
    for (int o = tid; o < nsub; o += NT) s_I[o] = 0.0;
    if (tid < 6) {
      const int d = tid % 3, l = tid < 3 ? LB : D.ld;
      const double x = tid < 3 ? bp.AB[d] : kp.AB[d];
      double *t = (tid < 3 ? s_ab : s_cd) + d * 25;  // t[l 5 + u] = C(l, u) x^(l - u)
      for (int k = 0; k <= l; ++k)
        for (int u = 0; u <= k; ++u)
          t[k * 5 + u] = k == 0 ? 1.0 : (u < k ? x * t[(k - 1) * 5 + u] : 0.0) + (u > 0 ? t[(k - 1) * 5 + u - 1] : 0.0);
    }
    for (int k0 = 0; k0 < ntot; k0 += sh.pp) {
      const int cnt = min(sh.pp, ntot - k0);
      double *s_H = s_tab + sh.pp * 3 * D.nr * GN;
      if (grp < cnt) {
        const int pi = (k0 + grp) / nkp, pj = k0 + grp - pi * nkp;
        const PrimPair P = a.prims[bp.pp_off + pi], Q = a.prims[kp.pp_off + pj];
        const double r = eval_rsqrt<double>(P.p + Q.p), rpq = r * r;
        const double aq = P.p * rpq, bq = Q.p * rpq;
        const double PQ[3] = {P.P[0] - Q.P[0], P.P[1] - Q.P[1], P.P[2] - Q.P[2]};
        const double T = P.p * bq * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
        double t2, wt;
        rys_root_rt(D.nr, root, T, a.rys, t2, wt);
        const double pref = P.K * Q.K * kTwoPi52 * P.rp * Q.rp * r;
        const double PQd = dir == 0 ? PQ[0] : dir == 1 ? PQ[1] : PQ[2];
        const double C00 = (dir == 0 ? P.P[0] : dir == 1 ? P.P[1] : P.P[2]) - bp.A[dir] - bq * t2 * PQd;
        const double D00 = (dir == 0 ? Q.P[0] : dir == 1 ? Q.P[1] : Q.P[2]) - kp.A[dir] + aq * t2 * PQd;
        const double B00 = 0.5 * t2 * rpq, B10 = 0.5 * P.rp * (1.0 - bq * t2), B01 = 0.5 * Q.rp * (1.0 - aq * t2);
        double *G = s_tab + (grp * 3 * D.nr + sub) * GN;  // [k][i]
        double cur[kTeamI], prev[kTeamI];
#pragma unroll
        for (int i = 0; i < kTeamI; ++i) {
          prev[i] = 0.0;
          if (i < D.ni) {
            const double below = i > 0 ? cur[i > 0 ? i - 1 : 0] : 0.0;
            const double below2 = i > 1 ? cur[i > 1 ? i - 2 : 0] : 0.0;
            cur[i] = i == 0 ? (dir == 2 ? pref * wt : 1.0) : C00 * below + (i - 1) * B10 * below2;
            G[i] = cur[i];
          }
        }
        for (int k = 1; k < D.nk; ++k) {
          double *Gk = G + k * D.ni;
          double below = 0.0;  // cur[i - 1] before this column
#pragma unroll
          for (int i = 0; i < kTeamI; ++i)
            if (i < D.ni) {
              const double c = cur[i];
              const double v = D00 * c + (k - 1) * B01 * prev[i] + i * B00 * below;
              below = c;
              prev[i] = c;
              cur[i] = v;
              Gk[i] = v;
            }
        }
      }
      for (int r0 = 0; r0 < D.nr; r0 += sh.rpp) {
        const int nrp = min(sh.rpp, D.nr - r0);
        __syncthreads();
        // horizontal transfers: entry e of (primitive quartet, root, direction) t
        const int per = 3 * nrp, nent = cnt * per * D.nh;
        for (int x = tid; x < nent; x += NT) {
          const int t = x / D.nh, e = x - t * D.nh, p = t / per, rd = t - p * per, d = rd % 3;
          const int dc = s_dec[e], xa = dc & 15, xb = (dc >> 4) & 15, xc = (dc >> 8) & 15, xd = dc >> 12;
          const double *G = s_tab + (p * 3 * D.nr + 3 * r0 + rd) * GN + xa;
          const double *ab = s_ab + d * 25 + xb * 5, *cd = s_cd + d * 25 + xd * 5;
          double s = 0.0;
          for (int v = 0; v <= xd; ++v) {
            const double *Gv = G + (xc + v) * D.ni;
            double u0 = 0.0;
            for (int u = 0; u <= xb; ++u) u0 = fma(ab[u], Gv[u], u0);
            s = fma(cd[v], u0, s);
          }
          s_H[(p * 3 * sh.rpp + rd) * D.nh + e] = s;
        }
        __syncthreads();
        // (a component, ket component) items, split over the primitive
        // quartets when there are fewer of them than threads
        const int nitem = na * D.nket;
        const int S = nitem * 2 <= NT ? min(NT / nitem, cnt) : 1;
        for (int x = tid; x < nitem * S; x += NT) {
          const int sl = x / nitem, it = x - sl * nitem, ia = it / D.nket, cd = it - ia * D.nket;
          const unsigned off = s_pa[ia0 + ia] + s_pk[cd];
          const int ox = off & 1023, oy = (off >> 10) & 1023, oz = off >> 20;
          double acc[NCB];
#pragma unroll
          for (int b = 0; b < NCB; ++b) acc[b] = 0.0;
          for (int p = sl; p < cnt; p += S)
            for (int r = 0; r < nrp; ++r) {
              const double *H = s_H + (size_t)((p * sh.rpp + r) * 3) * D.nh;
              double hx[LB + 1], hy[LB + 1], hz[LB + 1];
#pragma unroll
              for (int b = 0; b <= LB; ++b) {
                hx[b] = H[ox + b * sb];
                hy[b] = H[D.nh + oy + b * sb];
                hz[b] = H[2 * D.nh + oz + b * sb];
              }
#pragma unroll
              for (int b = 0; b < NCB; ++b)
                acc[b] = fma(hx[cexp(LB, b, 0)] * hy[cexp(LB, b, 1)], hz[cexp(LB, b, 2)], acc[b]);
            }
          double *o = s_I + ia * nbcd + cd;
#pragma unroll
          for (int b = 0; b < NCB; ++b) {
            if (S == 1) o[b * D.nket] += acc[b];
            else unsafeAtomicAdd(o + b * D.nket, acc[b]);
          }
        }
      }
      __syncthreads();
    }
    if (a.store_mode) {
      double *out = a.store + a.store_off[q] + (size_t)ia0 * nbcd;
      for (int o = tid; o < nsub; o += NT) out[o] = s_I[o];
      continue;
    }
    // degeneracy of the quartet in the 8-fold loop (direct.hpp:1664-1667,
    // 1793-1802), times the 1/2 of direct.hpp:1849-1850
    const bool same_pair = (bp.a == kp.a && bp.b == kp.b);
    const double deg =
        0.5 * (bp.a == bp.b ? 1.0 : 2.0) * (kp.a == kp.b ? 1.0 : 2.0) * (same_pair ? 1.0 : 2.0);
    for (int o = tid; o < nsub; o += NT) s_I[o] *= deg;
    const int n[4] = {na, NCB, D.ncc, D.ncd};
    const int bf[4] = {bp.bfa + ia0, bp.bfb, kp.bfa, kp.bfb};
    const int st[4] = {nbcd, D.nket, D.ncd, 1};
    const PlaneSet &ps = a.planes;
    const MolPlanes &mp = ps.nmol == 1 ? ps.m0 : ps.mols[bp.mol];
    const unsigned mask = qt.ket_mask >> 24;
    for (int kind = 0; kind < 4; ++kind) {
      const int np = ps.kcount[kind];
      if (np == 0) continue;
      const double base = kind == kJHer ? 1.0 : 0.5;
      for (int term = 0; term < kDigestTerms.n[kind]; ++term) {
        const int ar = kDigestTerms.t[kind][term][0], ac = kDigestTerms.t[kind][term][1];
        const int xr = kDigestTerms.t[kind][term][2], xc = kDigestTerms.t[kind][term][3];
        const int fit = max(1, min(np, sh.tab / (n[xr] * n[xc])));
        for (int p0 = 0; p0 < np; p0 += fit)
          team_term(s_I, s_tab, n, bf, st, ps, mp, kind, p0, min(fit, np - p0), ar, ac, xr, xc, base, mask, tid, NT);
      }
    }
  }
}

template <int LB, int NT>
hipError_t launch_team(const EriLaunch &a, const TeamShape &sh, long long items, hipStream_t s) {
  static std::once_flag once;  // once per process (contexts on several host threads launch concurrently)
  static hipError_t attr = hipSuccess;
  std::call_once(once, [] {
    attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&eri_team_kernel<LB, NT>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  });
  if (attr != hipSuccess) return attr;
  const size_t lds = (size_t)(sh.tab + sh.quart) * 8 + kTeamFixed;
  const long long grid = items < 65536 ? items : 65536;
  hipLaunchKernelGGL((eri_team_kernel<LB, NT>), dim3((unsigned)grid), dim3(NT), lds, s, a, sh);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_eri_team(const EriLaunch &a, hipStream_t s) {
  if (a.nq <= 0) return hipSuccess;
  if (a.la > kMaxLDev || a.lb > kMaxLDev || a.lc > kMaxLDev || a.ld > kMaxLDev) return hipErrorInvalidValue;
  const TeamDims D = team_dims(a.la, a.lb, a.lc, a.ld);
  TeamShape sh{};
  if (!team_plan(D, 160 * 1024, sh)) return hipErrorInvalidValue;
  const long long items = a.nq * ((D.nca + sh.ca - 1) / sh.ca);
#define CQX_TEAM(L) \
  case L: return sh.nt == 64 ? launch_team<L, 64>(a, sh, items, s) : launch_team<L, 256>(a, sh, items, s);
  switch (a.lb) {
    CQX_TEAM(0) CQX_TEAM(1) CQX_TEAM(2) CQX_TEAM(3)
    default: return sh.nt == 64 ? launch_team<4, 64>(a, sh, items, s) : launch_team<4, 256>(a, sh, items, s);
  }
#undef CQX_TEAM
}

}  // namespace cqx
