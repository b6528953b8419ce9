// J/K digestion of a tile of contracted Cartesian shell quartets with the
// density blocks staged in LDS.
//
// The updates are those of digest_tile.hpp.  There every work item reads its
// density elements from global memory: an element is loaded once per target
// it contributes to (222 vector loads per (fd|dp) quartet of a J/K pair),
// and each term's loads queue behind the previous term's atomics on the
// wave's in-order memory counter.  Here the wave first loads every density
// element of the tile's quartets once (64 per instruction, all loads in
// flight together), then forms every target from LDS, and only then are
// atomics issued.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_types.hpp"
#include "digest.hpp"
#include "digest_tile.hpp"
#include "eri_bra.hpp"

namespace cqx {

// Density blocks (row role, column role) that the updates of one quartet
// read.  Hermitian K: blocks 2-5; non-Hermitian K: 2-9.  A J update reads
// (d, c) and (a, b); for a non-Hermitian J the staged value is X(r, c) +
// X(c, r), since both orders contribute to the same targets.
constexpr int kXRoles[10][2] = {{3, 2}, {0, 1}, {3, 1}, {0, 2}, {1, 2}, {3, 0}, {1, 3}, {2, 0}, {2, 1}, {0, 3}};

template <class K>
struct XLayout {
  static constexpr int size(int b) { return K::n(kXRoles[b][0]) * K::n(kXRoles[b][1]); }
  // first element of block b within its kind's elements of one quartet
  static constexpr int off(int b) {
    int o = 0;
    for (int k = b < 2 ? 0 : 2; k < b; ++k) o += size(k);
    return o;
  }
  static constexpr int EJ = size(0) + size(1);
  static constexpr int EK = size(2) + size(3) + size(4) + size(5);
  static constexpr int EKN = EK + size(6) + size(7) + size(8) + size(9);
  static __host__ __device__ constexpr int per_kind(int kind) {
    return kind == kJHer || kind == kJNonHer ? EJ : kind == kKHer ? EK : EKN;
  }
};

__host__ __device__ inline int plane_shift(int np) {
  return np <= 1 ? 0 : np <= 2 ? 1 : np <= 4 ? 2 : np <= 8 ? 3 : 4;
}

struct DigestPlanes {  // one molecule's arrays of one kind
  const GlobalDouble *x;
  GlobalDouble *a;
  int n, stride, p0, np, lgp;
};

// Stage block B of the quartets of molecule mol (whose planes P are) among
// [0, nq) (first functions sbf, E elements each): the value of (quartet q,
// element e, plane p) goes to sX[((q E + off(B) + e) << lgp) + p].  Another
// molecule's functions may lie beyond the end of these planes: its quartets
// are left for their own turn.
template <class K, int B, int E>
__device__ __forceinline__ void stage_block(const int (*__restrict__ sbf)[4], const int *__restrict__ smol, int mol,
                                            int nq, bool both, const DigestPlanes &P, double *__restrict__ sX,
                                            int lane) {
  using L = XLayout<K>;
  constexpr int R = kXRoles[B][0], C = kXRoles[B][1], NR = K::n(R), SZ = L::size(B);
  const int items = (nq * SZ) << P.lgp;
  for (int it = lane; it < items; it += 64) {
    const int p = it & ((1 << P.lgp) - 1), r = it >> P.lgp, q = r / SZ, e = r - q * SZ;
    if (smol[q] != mol) continue;
    const int row = sbf[q][R] + e % NR, col = sbf[q][C] + e / NR;
    double v = 0.0;
    if (p < P.np) {
      v = P.x[((size_t)row + (size_t)col * P.n) * P.stride + p];
      if (both) v += P.x[((size_t)col + (size_t)row * P.n) * P.stride + p];
    }
    sX[((q * E + L::off(B) + e) << P.lgp) + p] = v;
  }
}

// The targets of one update term: A(ar, ac) += coef sum I X(block XB), for
// the quartets [0, nq) of the molecule.  HER as in digest_tile.hpp; BOTH (a
// non-Hermitian J): added to A(ac, ar) too.
template <class K, int AR, int AC, int XB, int E, bool HER, bool BOTH>
__device__ __forceinline__ void staged_term(const double *__restrict__ sI, const int (*__restrict__ sbf)[4],
                                            const unsigned *__restrict__ smask, const int *__restrict__ smol, int mol,
                                            int nq, const PlaneSet &ps, const DigestPlanes &P,
                                            const double *__restrict__ sX, double base_coef, bool neg_ok, int lane) {
  using L = XLayout<K>;
  constexpr int XR = kXRoles[XB][0], XC = kXRoles[XB][1], XO = L::off(XB);
  constexpr int NAR = K::n(AR), NT = NAR * K::n(AC);
  constexpr int ST[4] = {K::NCB * K::NCC * K::NCD, K::NCC * K::NCD, K::NCD, 1};
  constexpr bool TR = HER && K::n(AC) > K::n(AR);  // store A(ac, ar) instead
  constexpr int NFAST = TR ? K::n(AC) : NAR;
  const int items = (nq * NT) << P.lgp;
  for (int it = lane; it < items; it += 64) {
    const int p = it & ((1 << P.lgp) - 1);
    if (p >= P.np) continue;
    const int r = it >> P.lgp, qi = r / NT, tgt = r - qi * NT;
    const int tslow = tgt / NFAST, tfast = tgt - tslow * NFAST;
    const int t0 = TR ? tslow : tfast, t1 = TR ? tfast : tslow;
    const int mat = (int)((ps.mats >> (4 * (P.p0 + p))) & 15ull);
    if (!((smask[qi] >> mat) & 1u) || smol[qi] != mol) continue;
    const double *__restrict__ Iq = sI + qi * K::NC + t0 * ST[AR] + t1 * ST[AC];
    const double *__restrict__ X = sX + ((qi * E + XO) << P.lgp) + p;
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int u1 = 0; u1 < K::n(XC); ++u1)
#pragma unroll
      for (int u0 = 0; u0 < K::n(XR); ++u0) {
        const double v = Iq[u0 * ST[XR] + u1 * ST[XC]] * X[(u0 + u1 * K::n(XR)) << P.lgp];
        if ((u0 + u1 * K::n(XR)) & 1) s1 += v; else s0 += v;
      }
    const int *bf = sbf[qi];
    const int row = bf[AR] + t0, col = bf[AC] + t1;
    const bool neg = (ps.negs >> (P.p0 + p)) & 1u;
    // conj of Im X for Hermitian K; a transposed update of an imaginary plane flips sign again
    const double v = ((neg_ok && neg) != (TR && neg)) ? -base_coef * (s0 + s1) : base_coef * (s0 + s1);
    const size_t rc = (size_t)row + (size_t)col * P.n, cr = (size_t)col + (size_t)row * P.n;
    __builtin_amdgcn_global_atomic_fadd_f64(P.a + (TR ? cr : rc) * P.stride + p, v);
    if constexpr (BOTH) __builtin_amdgcn_global_atomic_fadd_f64(P.a + cr * P.stride + p, v);
  }
}

// digest_tile with staged density blocks; sX: XCAP doubles of the wave.  A
// plane set too wide for even one quartet's elements takes digest_tile,
// whose lanes then share 64-byte segments of the interleaved planes.
template <class K, int XCAP>
__device__ __forceinline__ void digest_staged(const double *sI, const int (*sbf)[4], const unsigned *smask,
                                              const int *smol, int nq, const PlaneSet &ps, double *sX, int lane) {
  using L = XLayout<K>;
  int per_q = 0;
  for (int kind = 0; kind < 4; ++kind)
    if (ps.kcount[kind]) per_q += L::per_kind(kind) << plane_shift(ps.kcount[kind]);
  if (per_q > XCAP) {
    digest_tile<K>(sI, sbf, smask, smol, nq, ps, lane);
    return;
  }
  const int step = min(nq, XCAP / per_q);
  for (int q0 = 0; q0 < nq; q0 += step) {
    const int n = min(step, nq - q0);
    const double *tI = sI + q0 * K::NC;
    const int(*tbf)[4] = sbf + q0;
    const unsigned *tmask = smask + q0;
    const int *tmol = smol + q0;
    // molecules of the sub-tile, nearly always one
    unsigned todo = (1u << n) - 1u;
    while (todo) {
      const int mol = __builtin_amdgcn_readfirstlane(tmol[__builtin_ctz(todo)]);
      todo &= ~(unsigned)__ballot(lane < n && tmol[lane] == mol);
      const ConstPtr<MolPlanes> mp = as_const(ps.mols + (ps.nmol == 1 ? 0 : mol));
      auto planes_of = [&](int kind) {
        DigestPlanes P;
        P.x = (const GlobalDouble *)(ps.nmol == 1 ? ps.m0.kx[kind] : mp->kx[kind]);
        P.a = (GlobalDouble *)(ps.nmol == 1 ? ps.m0.ka[kind] : mp->ka[kind]);
        P.n = ps.nmol == 1 ? ps.m0.nbc : mp->nbc;
        P.stride = ps.kps[kind];
        P.p0 = ps.kstart[kind];
        P.np = ps.kcount[kind];
        P.lgp = plane_shift(P.np);
        return P;
      };
      int xoff = 0;
      for (int kind = 0; kind < 4; ++kind) {
        if (ps.kcount[kind] == 0) continue;
        const DigestPlanes P = planes_of(kind);
        double *X = sX + xoff;
        xoff += (n * L::per_kind(kind)) << P.lgp;
#define CQX_STAGE(B, E) stage_block<K, B, E>(tbf, tmol, mol, n, kind == kJNonHer, P, X, lane)
        if (kind == kJHer || kind == kJNonHer) {
          CQX_STAGE(0, L::EJ);
          CQX_STAGE(1, L::EJ);
        } else if (kind == kKHer) {
          CQX_STAGE(2, L::EK);
          CQX_STAGE(3, L::EK);
          CQX_STAGE(4, L::EK);
          CQX_STAGE(5, L::EK);
        } else {
          CQX_STAGE(2, L::EKN);
          CQX_STAGE(3, L::EKN);
          CQX_STAGE(4, L::EKN);
          CQX_STAGE(5, L::EKN);
          CQX_STAGE(6, L::EKN);
          CQX_STAGE(7, L::EKN);
          CQX_STAGE(8, L::EKN);
          CQX_STAGE(9, L::EKN);
        }
#undef CQX_STAGE
      }
      wave_sync();
      xoff = 0;
      for (int kind = 0; kind < 4; ++kind) {
        if (ps.kcount[kind] == 0) continue;
        const DigestPlanes P = planes_of(kind);
        const double *X = sX + xoff;
        xoff += (n * L::per_kind(kind)) << P.lgp;
#define CQX_TERM(AR, AC, XB, E, HER, BOTH, COEF, NEG) \
  staged_term<K, AR, AC, XB, E, HER, BOTH>(tI, tbf, tmask, tmol, mol, n, ps, P, X, COEF, NEG, lane)
        switch (kind) {
          case kJHer:
            CQX_TERM(0, 1, 0, L::EJ, true, false, 1.0, false);
            CQX_TERM(3, 2, 1, L::EJ, true, false, 1.0, false);
            break;
          case kKHer:
            CQX_TERM(0, 2, 2, L::EK, true, false, 0.5, true);
            CQX_TERM(3, 1, 3, L::EK, true, false, 0.5, true);
            CQX_TERM(3, 0, 4, L::EK, true, false, 0.5, true);
            CQX_TERM(1, 2, 5, L::EK, true, false, 0.5, true);
            break;
          case kJNonHer:
            CQX_TERM(0, 1, 0, L::EJ, false, true, 0.5, false);
            CQX_TERM(3, 2, 1, L::EJ, false, true, 0.5, false);
            break;
          default:
            CQX_TERM(2, 0, 2, L::EKN, false, false, 0.5, false);  // X(d, b)
            CQX_TERM(1, 3, 3, L::EKN, false, false, 0.5, false);  // X(a, c)
            CQX_TERM(0, 3, 4, L::EKN, false, false, 0.5, false);  // X(b, c)
            CQX_TERM(2, 1, 5, L::EKN, false, false, 0.5, false);  // X(d, a)
            CQX_TERM(0, 2, 6, L::EKN, false, false, 0.5, false);  // X(b, d)
            CQX_TERM(3, 1, 7, L::EKN, false, false, 0.5, false);  // X(c, a)
            CQX_TERM(3, 0, 8, L::EKN, false, false, 0.5, false);  // X(c, b)
            CQX_TERM(1, 2, 9, L::EKN, false, false, 0.5, false);  // X(a, d)
            break;
        }
#undef CQX_TERM
      }
      wave_sync();  // the staged blocks are rewritten
    }
  }
}

}  // namespace cqx
