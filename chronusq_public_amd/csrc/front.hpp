// Launchers of a build's front and back kernels (front.hip): everything
// before and after the ERI launches, each step one launch over every
// molecule, contraction and class.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "device_types.hpp"
#include "kernels.hpp"

namespace cqx {

constexpr int kMaxClass = (kMaxLDev + 1) * (kMaxLDev + 2) / 2;

// One molecule of a context: sizes, first functions / shells, and where its
// blocks start in the flattened ranges (block norms, functions squared).
struct MolInfo {
  int nb, nbc, ns, bf0, bfc0, sh0;
  long long boff, nb2, nbc2;
};

struct FrontArgs {
  const MolInfo *mol;      // nmol + 1 entries (the last: the totals)
  int nmol, nmat, cplx;
  unsigned her;            // bit j: contraction j is Hermitian
  CartMap map;             // of the whole context (bf0 = bfc0 = 0)
  const int *sh_nf;
  // X and AX of contraction j of molecule m: xs[j], axs[j] of a one-molecule
  // context, else x[m nmat + j], ax[m nmat + j]
  const double *xs[kMaxMat];
  double *axs[kMaxMat];
  const double *const *x;
  double *const *ax;
  MolPlanes m0;            // planes of a one-molecule context
  const MolPlanes *mols;
  int kps[4];
  int kind[kMaxMat], re[kMaxMat], im[kMaxMat];  // planes of contraction j (im < 0: none)
  double *Bm, *Bg, *molmax;
  // pairs of every class: screening records, own norms, and the row
  // kernels' Coulomb planes in pair order (jx, ja: class k from joff[k] on)
  const PairScr *scr[kMaxClass];
  const PairRec *pairs[kMaxClass];
  double *pn[kMaxClass];
  int npair[kMaxClass];
  long long cstart[kMaxClass + 1];  // class k's (component, pair) range
  size_t joff[kMaxClass];
  int nj, jkind[4], jidx[4];
  double *jx;
  double *ja;
};

// ranges of doubles cleared by one launch
struct ZeroRanges {
  static constexpr int kMax = 8;
  double *p[kMax];
  size_t n[kMax];
  int count = 0;
  void add(double *q, size_t m) {
    if (!m) return;
    p[count] = q;
    n[count++] = m;
  }
};

hipError_t launch_zero_ranges(const ZeroRanges &z, hipStream_t s);
// shell-block norms (per matrix and global) and each molecule's largest;
// molmax cleared before
hipError_t launch_norms(const FrontArgs &a, long long nblock, hipStream_t s);
// Cartesian planes of every contraction
hipError_t launch_planes(const FrontArgs &a, long long nbc2, hipStream_t s);
// the pairs' own norms and Coulomb planes in pair order
hipError_t launch_pairs(const FrontArgs &a, hipStream_t s);
// candidate counts of every class pair and their prefix sums, one block per
// class pair; tot[k]: the total
hipError_t launch_candidates_all(const CandLaunch *table, int n, long long *tot, hipStream_t s);
// pair-order Coulomb sums onto the accumulators
hipError_t launch_pairs_back(const FrontArgs &a, hipStream_t s);
// accumulators to pure functions, Hermitian finalisation, added to AX:
// functions squared [first, last) of the flattened range, contractions
// [j0, j0 + nj)
hipError_t launch_back(const FrontArgs &a, long long first, long long last, int j0, int nj, hipStream_t s);

}  // namespace cqx
