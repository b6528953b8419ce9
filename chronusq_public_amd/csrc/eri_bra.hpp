// Primitive loops of a contracted Cartesian shell quartet whose bra pair is
// the same for the whole wave: the bra's records come through the scalar
// cache and the ket's primitive pairs are loaded once, so the loop over
// primitive quartets holds no vector memory access (the earlier form loaded
// both primitive pairs per primitive quartet, eight vector loads for about
// 80 FP64 operations of an (ss|ss), and kept the vector address unit busier
// than the ALUs).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "eri_class.hpp"

namespace cqx {

// A wave-uniform read of memory that no kernel writes goes through the
// scalar cache when its address is in the constant address space.
template <class T>
using ConstPtr = const __attribute__((address_space(4))) T *;
template <class T>
__device__ __forceinline__ ConstPtr<T> as_const(const T *p) {
  return (ConstPtr<T>)p;
}
// Pointers read from a table are generic to the compiler; the planes are
// known to be global memory (a generic access would also wait on LDS).
using GlobalDouble = __attribute__((address_space(1))) double;

namespace {

// Add to I the primitive quartets of primitives [i0, i1) of a bra pair that
// is the same for the whole wave (bp; its records come through the scalar cache) with the ket's
// primitive pairs g, g + G, ... below nk, each held in registers while the
// bra's primitives pass by.
template <int LA, int LB, int LC, int LD, class R, bool ROOM>
__device__ __forceinline__ void eval_bra(const PrimPair *prims, const PrimC32 *pc32, const R *__restrict__ rysn,
                                         ConstPtr<PairRec> bp, int i0, int i1, const double (&Cc)[3], const double (&CDc)[3],
                                         int koff, int nk, int g, int G, R (&I)[Cls<LA, LB, LC, LD>::NC]) {
  using K = Cls<LA, LB, LC, LD>;
  constexpr bool F32 = std::is_same<R, float>::value;
  const int boff = bp->pp_off;
  R AB[3], CD[3], AC[3];
  double Ac[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    Ac[d] = bp->A[d];
    AB[d] = (R)bp->AB[d];
    CD[d] = (R)CDc[d];
    AC[d] = (R)(Ac[d] - Cc[d]);  // A - C in FP64 before the rounding
  }
  for (int j = g; j < nk; j += G) {
    R bq, rq, Q[3], QC[3];
    double Kq;
    if constexpr (F32) {
      const PrimC32 B = pc32[koff + j];
      bq = B.p;
      Kq = B.K * kTwoPi52;
      rq = eval_rcp<R>(bq);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        QC[d] = -B.bp * CD[d];
        Q[d] = AC[d] - QC[d];  // A - Q
      }
    } else {
      const PrimPair B = prims[koff + j];
      bq = B.p;
      rq = B.rp;
      Kq = B.K * kTwoPi52 * B.rp;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        Q[d] = B.P[d];
        QC[d] = B.P[d] - Cc[d];
      }
    }
    for (int i = i0; i < i1; ++i) {
      R ap, rp, PA[3], PQ[3], pref;
      R r, rpq;
      if constexpr (F32) {
        const auto A = as_const(pc32 + boff + i);
        ap = A->p;
        rp = eval_rcp<R>(ap);
        r = eval_rsqrt<R>(ap + bq);
        rpq = r * r;
        pref = (R)(A->K * Kq) * (rp * rq) * r;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          PA[d] = -A->bp * AB[d];
          PQ[d] = Q[d] + PA[d];
        }
      } else {
        const auto A = as_const(prims + boff + i);
        ap = A->p;
        rp = A->rp;
        r = eval_rsqrt<R>(ap + bq);
        rpq = r * r;
        pref = A->K * rp * (Kq * r);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          PQ[d] = A->P[d] - Q[d];
          PA[d] = A->P[d] - Ac[d];
        }
      }
      const R aq = ap * rpq, bqr = bq * rpq;  // p / (p + q), q / (p + q)
      const R rho = ap * bqr;
      const R T = rho * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
      R x[K::NR], w[K::NR];
      rys_roots_row<K::NR, R, K::NC == 1, ROOM>(T, rysn, x, w);
      if constexpr (K::NC == 1) {
        I[0] = fma(pref, w[0], I[0]);
      } else {
#pragma unroll
        for (int t = 0; t < K::NR; ++t) {
          const R t2 = x[t];
          const R B00 = (R)0.5 * t2 * rpq;
          const R B10 = (R)0.5 * rp * ((R)1 - bqr * t2);
          const R B01 = (R)0.5 * rq * ((R)1 - aq * t2);
          R H[3][K::NH];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const R C00 = PA[d] - bqr * t2 * PQ[d];
            const R D00 = QC[d] + aq * t2 * PQ[d];
            rys_2d_full<LA, LB, LC, LD, R>(C00, D00, B10, B01, B00, AB[d], CD[d],
                                           d == 2 ? pref * w[t] : (R)1, H[d]);
          }
          constexpr HTab<LA, LB, LC, LD> HT = make_htab<LA, LB, LC, LD>();
#pragma unroll
          for (int o = 0; o < K::NC; ++o) I[o] = fma(H[0][HT.x[o]] * H[1][HT.y[o]], H[2][HT.z[o]], I[o]);
        }
      }
    }
  }
}

}  // namespace

}  // namespace cqx
