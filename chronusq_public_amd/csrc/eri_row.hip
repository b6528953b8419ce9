// Dispatch of the row kernels (eri_row_impl.hpp) and the transforms of the
// Coulomb planes between matrix and pair order.
#include <hip/hip_runtime.h>

#include "eri_row.hpp"

namespace cqx {

template <int GROUP>
hipError_t launch_row_group(const RowLaunch &a, hipStream_t s);
template <int GROUP>
bool row_group_lds(int la, int lb, int lc, int ld, int fp32, int nk, int width, size_t &bytes);

namespace {

bool row_lds_of(int la, int lb, int lc, int ld, int fp32, int nk, int width, size_t &bytes) {
  return row_group_lds<0>(la, lb, lc, ld, fp32, nk, width, bytes) ||
         row_group_lds<1>(la, lb, lc, ld, fp32, nk, width, bytes) ||
         row_group_lds<2>(la, lb, lc, ld, fp32, nk, width, bytes) ||
         row_group_lds<3>(la, lb, lc, ld, fp32, nk, width, bytes);
}

__device__ __forceinline__ const MolPlanes &planes_of(const PairOrder &a, int mol) {
  return a.nmol == 1 ? a.m0 : a.mols[mol];
}

__global__ void pair_pack_kernel(PairOrder a) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nc = a.na * a.nb;
  if (t >= (long long)a.npair * nc * a.nj) return;
  const int i = (int)(t % a.npair), rest = (int)(t / a.npair);
  const int e = rest % nc, j = rest / nc;
  const PairRec &P = a.pairs[i];
  const MolPlanes &mp = planes_of(a, P.mol);
  const int r = P.bfa + e / a.nb, c = P.bfb + e % a.nb, k = a.kind[j];
  const double *x = mp.kx[k] + a.idx[j];
  double v = x[((size_t)c + (size_t)r * mp.nbc) * a.stride[j]];
  if (k == kJNonHer) v += x[((size_t)r + (size_t)c * mp.nbc) * a.stride[j]];
  a.jx[t] = v;
}

__global__ void pair_unpack_kernel(PairOrder a) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nc = a.na * a.nb;
  if (t >= (long long)a.npair * nc * a.nj) return;
  const double v = a.ja[t];
  if (v == 0.0) return;
  const int i = (int)(t % a.npair), rest = (int)(t / a.npair);
  const int e = rest % nc, j = rest / nc;
  const PairRec &P = a.pairs[i];
  const MolPlanes &mp = planes_of(a, P.mol);
  const int r = P.bfa + e / a.nb, c = P.bfb + e % a.nb, k = a.kind[j];
  double *o = mp.ka[k] + a.idx[j];
  unsafeAtomicAdd(o + ((size_t)r + (size_t)c * mp.nbc) * a.stride[j], v);
  if (k == kJNonHer) unsafeAtomicAdd(o + ((size_t)c + (size_t)r * mp.nbc) * a.stride[j], v);
}

}  // namespace

bool eri_row_built(int la, int lb, int lc, int ld) {
  size_t b = 0;
  return row_lds_of(la, lb, lc, ld, 0, 0, 0, b);
}

size_t eri_row_lds(int la, int lb, int lc, int ld, int fp32, int nk, int width) {
  size_t b = 0;
  if (!row_lds_of(la, lb, lc, ld, fp32, nk, width, b)) return 0;
  return b <= 160 * 1024 ? b : 0;
}

hipError_t launch_eri_row(const RowLaunch &a, hipStream_t s) {
  hipError_t e = launch_row_group<0>(a, s);
  if (e == hipErrorNotSupported) e = launch_row_group<1>(a, s);
  if (e == hipErrorNotSupported) e = launch_row_group<2>(a, s);
  if (e == hipErrorNotSupported) e = launch_row_group<3>(a, s);
  return e;
}

hipError_t launch_pair_pack(const PairOrder &a, hipStream_t s) {
  const long long n = (long long)a.npair * a.na * a.nb * a.nj;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(pair_pack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_pair_unpack(const PairOrder &a, hipStream_t s) {
  const long long n = (long long)a.npair * a.na * a.nb * a.nj;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(pair_unpack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace cqx
