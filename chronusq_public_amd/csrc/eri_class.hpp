// What the templated ERI kernels share: class sizes and Cartesian tables,
// the 2D Rys recursions and the factors of a primitive quartet.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_types.hpp"
#include "rys.hpp"

namespace cqx {

namespace {

constexpr double kTwoPi52 = 34.98683665524972;  // 2 pi^(5/2)

constexpr int ncart_c(int l) { return (l + 1) * (l + 2) / 2; }

// Cartesian exponents of component c of an l shell (lx descending, then ly)
constexpr int cexp(int l, int c, int dir) {
  int k = c, lx = l;
  while (k >= l - lx + 1) {
    k -= l - lx + 1;
    --lx;
  }
  const int lz = k, ly = l - lx - lz;
  return dir == 0 ? lx : (dir == 1 ? ly : lz);
}

__device__ __forceinline__ void atomic_add(double *p, double v) { unsafeAtomicAdd(p, v); }

template <int LA, int LB, int LC, int LD>
struct Cls {
  static constexpr int NCA = ncart_c(LA), NCB = ncart_c(LB), NCC = ncart_c(LC), NCD = ncart_c(LD);
  static constexpr int NC = NCA * NCB * NCC * NCD;
  static constexpr int NI = LA + LB + 1, NK = LC + LD + 1;
  static constexpr int NR = (LA + LB + LC + LD) / 2 + 1;
  static constexpr int NH = (LA + 1) * (LB + 1) * (LC + 1) * (LD + 1);
  static constexpr int n(int role) { return role == 0 ? NCA : role == 1 ? NCB : role == 2 ? NCC : NCD; }
  static constexpr int oidx(int ia, int ib, int ic, int id) { return ((ia * NCB + ib) * NCC + ic) * NCD + id; }
  static constexpr int hidx(int a, int b, int c, int d) {
    return ((a * (LB + 1) + b) * (LC + 1) + c) * (LD + 1) + d;
  }
};

// For each Cartesian component o of the quartet, the offsets of its x, y
// and z factors in the 2D-integral tables; built at compile time so that an
// unrolled loop over o indexes the tables with constants.
template <int LA, int LB, int LC, int LD>
struct HTab {
  int x[Cls<LA, LB, LC, LD>::NC], y[Cls<LA, LB, LC, LD>::NC], z[Cls<LA, LB, LC, LD>::NC];
};

template <int LA, int LB, int LC, int LD>
constexpr HTab<LA, LB, LC, LD> make_htab() {
  using K = Cls<LA, LB, LC, LD>;
  HTab<LA, LB, LC, LD> t{};
  for (int ia = 0; ia < K::NCA; ++ia)
    for (int ib = 0; ib < K::NCB; ++ib)
      for (int ic = 0; ic < K::NCC; ++ic)
        for (int id = 0; id < K::NCD; ++id) {
          const int o = K::oidx(ia, ib, ic, id);
          t.x[o] = K::hidx(cexp(LA, ia, 0), cexp(LB, ib, 0), cexp(LC, ic, 0), cexp(LD, id, 0));
          t.y[o] = K::hidx(cexp(LA, ia, 1), cexp(LB, ib, 1), cexp(LC, ic, 1), cexp(LD, id, 1));
          t.z[o] = K::hidx(cexp(LA, ia, 2), cexp(LB, ib, 2), cexp(LC, ic, 2), cexp(LD, id, 2));
        }
  return t;
}

// 2D integrals of one root along one direction: VRR on (i, k), then HRR to
// (ia, ib, ic, id); H has Cls::NH entries.
template <int LA, int LB, int LC, int LD, class R>
__device__ __forceinline__ void rys_2d_full(R C00, R D00, R B10, R B01, R B00, R ABd, R CDd, R scale,
                                            R (&H)[Cls<LA, LB, LC, LD>::NH]) {
  using K = Cls<LA, LB, LC, LD>;
  R G[K::NI][K::NK];
  G[0][0] = scale;
  if constexpr (K::NI > 1) G[1][0] = C00 * scale;
#pragma unroll
  for (int i = 1; i + 1 < K::NI; ++i) G[i + 1][0] = C00 * G[i][0] + i * B10 * G[i - 1][0];
  if constexpr (K::NK > 1) {
#pragma unroll
    for (int k = 0; k + 1 < K::NK; ++k) {
      if (k == 0) {
        G[0][1] = D00 * G[0][0];
#pragma unroll
        for (int i = 1; i < K::NI; ++i) G[i][1] = D00 * G[i][0] + i * B00 * G[i - 1][0];
      } else {
        G[0][k + 1] = D00 * G[0][k] + k * B01 * G[0][k - 1];
#pragma unroll
        for (int i = 1; i < K::NI; ++i)
          G[i][k + 1] = D00 * G[i][k] + k * B01 * G[i][k - 1] + i * B00 * G[i - 1][k];
      }
    }
  }
  // bra transfer: E[i][j][k], (i, j+1) = (i+1, j) + AB (i, j)
  R E[K::NI][LB + 1][K::NK];
#pragma unroll
  for (int i = 0; i < K::NI; ++i)
#pragma unroll
    for (int k = 0; k < K::NK; ++k) E[i][0][k] = G[i][k];
#pragma unroll
  for (int j = 1; j <= LB; ++j)
#pragma unroll
    for (int i = 0; i + j < K::NI; ++i)
#pragma unroll
      for (int k = 0; k < K::NK; ++k) E[i][j][k] = E[i + 1][j - 1][k] + ABd * E[i][j - 1][k];
  // ket transfer for each (ia, ib)
#pragma unroll
  for (int ia = 0; ia <= LA; ++ia)
#pragma unroll
    for (int ib = 0; ib <= LB; ++ib) {
      R F[K::NK][LD + 1];
#pragma unroll
      for (int k = 0; k < K::NK; ++k) F[k][0] = E[ia][ib][k];
#pragma unroll
      for (int l = 1; l <= LD; ++l)
#pragma unroll
        for (int k = 0; k + l < K::NK; ++k) F[k][l] = F[k + 1][l - 1] + CDd * F[k][l - 1];
#pragma unroll
      for (int ic = 0; ic <= LC; ++ic)
#pragma unroll
        for (int id = 0; id <= LD; ++id) H[K::hidx(ia, ib, ic, id)] = F[ic][id];
    }
}

// The factors of a primitive quartet (bra exponent sum p, ket q) that need
// a division, from one reciprocal d = 1 / (p q (p + q)):
// 1 / (p + q), 1 / (p q), and the prefactor K_ab K_cd 2 pi^(5/2) / (p q sqrt(p + q)).
template <class R>
struct PrimRecip {
  R rpq, rab, pref;
};
template <class R>
__device__ __forceinline__ PrimRecip<R> prim_recip(R ap, R bq, double kk) {
  const R pq = ap + bq, ab = ap * bq;
  const R d = eval_rcp<R>(ab * pq);
  PrimRecip<R> r;
  r.rpq = ab * d;
  r.rab = pq * d;
  r.pref = (R)(kk * kTwoPi52) * r.rab * eval_sqrt<R>(r.rpq);
  return r;
}

// Rys table of the evaluation precision
template <class R> __device__ __forceinline__ const R *rys_table(const double *r64, const float *r32);
template <> __device__ __forceinline__ const double *rys_table<double>(const double *r64, const float *) { return r64; }
template <> __device__ __forceinline__ const float *rys_table<float>(const double *, const float *r32) { return r32; }

}  // namespace

}  // namespace cqx
