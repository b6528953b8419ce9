// The J/K updates of a contracted Cartesian shell quartet, as the generic
// kernel walks through them: those of the reference (direct.hpp:1858-2002)
// in the kernel's canonical labels a, b, c, d (roles 0..3).  Each update
//   A(ar, ac) += coef * sum_{xr, xc} I(a,b,c,d) X(xr, xc)
#pragma once

#include <hip/hip_runtime.h>

#include "device_types.hpp"

namespace cqx {

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// (ar, ac, xr, xc) of every update, per plane kind; coefficient per kind
// in the digestion (1 for Hermitian J, sign/2 for Hermitian K, 1/2 otherwise)
struct DigestTerms {
  int n[4];
  signed char t[4][8][4];
};

__device__ __constant__ const DigestTerms kDigestTerms = {
    {2, 4, 8, 8},
    {{{0, 1, 3, 2}, {3, 2, 0, 1}},
     {{0, 2, 3, 1}, {3, 1, 0, 2}, {3, 0, 1, 2}, {1, 2, 3, 0}},
     {{0, 1, 3, 2}, {0, 1, 2, 3}, {1, 0, 3, 2}, {1, 0, 2, 3},
      {2, 3, 1, 0}, {2, 3, 0, 1}, {3, 2, 1, 0}, {3, 2, 0, 1}},
     {{2, 0, 3, 1}, {3, 1, 2, 0}, {3, 0, 2, 1}, {2, 1, 3, 0},
      {0, 2, 1, 3}, {1, 3, 0, 2}, {0, 3, 1, 2}, {1, 2, 0, 3}}}};

}  // namespace cqx
