// Coefficients of the Cartesian <-> pure transforms on the device.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace cqx {

namespace {

__device__ __forceinline__ int ncart_f(int l) { return (l + 1) * (l + 2) / 2; }

__device__ __forceinline__ int sph_off(int l) {
  // sum_{k<l} (2k+1) ncart(k): 0, 1, 10, 40, 110
  return l == 0 ? 0 : l == 1 ? 1 : l == 2 ? 10 : l == 3 ? 40 : 110;
}
// coefficient T(cart comp c, pure function m) of a shell
__device__ __forceinline__ double tcoef(const CartMap &M, int s, int c, int m) {
  if (!M.sh_pure[s]) return c == m ? 1.0 : 0.0;
  const int l = M.sh_l[s];
  return M.sph[sph_off(l) + m * ncart_f(l) + c];
}
__device__ __forceinline__ int nfunc(const CartMap &M, int s) {
  return M.sh_pure[s] ? 2 * M.sh_l[s] + 1 : ncart_f(M.sh_l[s]);
}

}  // namespace

}  // namespace cqx
