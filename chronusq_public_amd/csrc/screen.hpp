// The reference's screen of one candidate shell quartet on the device
// (direct.hpp:1689-1789), shared by the list kernels and the kernels that
// screen their own kets.
#pragma once

#include <hip/hip_runtime.h>

#include "device_types.hpp"

namespace cqx {

// Bra pair P with its own block norms pb, ket pair Q with pk: the Schwarz
// product against the max of the six shell-block norms in reference labels
// (the pair the reference loop visits later is the bra), globally and per
// matrix (separated screen).  Returns whether any contraction survives and
// their mask.
struct ScreenArgs {
  const double *Bg, *Bm;
  const long long *mol_boff;
  const int *mol_ns;
  int nmat;
  double thresh;
  int screen;
};
__device__ __forceinline__ bool screen_candidate(const ScreenArgs &a, const PairScr &P, const PairScr &Q,
                                                 const double *pb, const double *pk, double qq, unsigned &mask) {
  mask = 0;
  const int ps1 = (int)(P.s12 & 0xFFFFu), ps2 = (int)(P.s12 >> 16);
  const int qs1 = (int)(Q.s12 & 0xFFFFu), qs2 = (int)(Q.s12 >> 16);
  const bool p_first = (ps1 > qs1) || (ps1 == qs1 && ps2 >= qs2);
  const int s1 = p_first ? ps1 : qs1, s2 = p_first ? ps2 : qs2;
  const int s3 = p_first ? qs1 : ps1, s4 = p_first ? qs2 : ps2;
  // lower bounds from the pairs' own block norms: enough to accept
  if (!a.screen) {
    mask = (1u << a.nmat) - 1u;
    return true;
  }
  if (!(fmax(pb[0], pk[0]) * qq < a.thresh)) {
    if (a.nmat == 1) {
      mask = 1u;
      return true;
    }
    unsigned lm = 0;
    for (int m = 0; m < a.nmat; ++m)
      if (!(fmax(pb[1 + m], pk[1 + m]) * qq < a.thresh)) lm |= 1u << m;
    if (lm == (1u << a.nmat) - 1u) {
      mask = lm;
      return true;
    }
  }
  const long long boff = a.mol_boff[P.mol];
  const int ns = a.mol_ns[P.mol];
  auto bmax = [&](const double *B, int ld, int m) {
    auto at = [&](int x, int y) { return B[(boff + x + (size_t)y * ns) * ld + m]; };
    double v = fmax(at(s1, s2), fmax(at(s1, s3), at(s2, s3)));
    v = fmax(v, at(s3, s4));
    v = fmax(v, fmax(at(s1, s4), at(s2, s4)));
    return v;
  };
  if (bmax(a.Bg, 1, 0) * qq < a.thresh) return false;
  if (a.nmat == 1) {
    mask = 1u;
  } else {
    // per-matrix norms interleaved: the nmat values of one block share a line
    for (int m = 0; m < a.nmat; ++m)
      if (!(bmax(a.Bm, a.nmat, m) * qq < a.thresh)) mask |= 1u << m;
  }
  return mask != 0u;
}

}  // namespace cqx
