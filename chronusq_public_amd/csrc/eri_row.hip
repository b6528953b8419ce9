// Dispatch of the row kernels (eri_row_impl.hpp).
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

}  // namespace

size_t eri_row_lds(int la, int lb, int lc, int ld, int fp32, int nk, int width) {
  size_t b = 0;
  if (!row_lds_of(la, lb, lc, ld, fp32, nk, width, b)) return 0;
  return b <= kRowLdsMax ? b : 0;
}

hipError_t launch_eri_row(const RowLaunch &a, hipStream_t s) {
  hipError_t e = launch_row_group<0>(a, s);
  if (e == hipErrorNotSupported) e = launch_row_group<1>(a, s);
  if (e == hipErrorNotSupported) e = launch_row_group<2>(a, s);
  if (e == hipErrorNotSupported) e = launch_row_group<3>(a, s);
  return e;
}

}  // namespace cqx
