// Rys quadrature nodes and weights on the device.
//
// For n roots: nodes x_r = t_r^2 in (0, 1) and weights w_r with
// sum_r w_r x_r^k = F_k(T) for k < 2n (F_k: Boys function).  Below the
// per-n cut-off T_n the values come from Chebyshev fits on unit intervals
// of T (gen_rys_table.py), which the build rewrites in powers of
// t = T - (i + 1/2): 13 fused multiply-adds a value, where the Chebyshev
// recurrence takes 27 operations.  On |t| <= 1/2 the powers fall faster
// than their rounding matters (the k-th coefficient is the k-th derivative
// over k!).  Above the cut-off: the Gauss-Hermite asymptotic form
// x = r^2 / T, w = W / sqrt(T), from one reciprocal square root.
#pragma once

#include <hip/hip_runtime.h>

#include "rys_table.h"

namespace cqx {

// Reciprocal and square root in the evaluation precision: correctly
// rounded in FP64; the hardware's one-instruction forms (1 ulp) in FP32,
// whose rounding is below the FP32 quartets' own.
template <class R> __device__ __forceinline__ R eval_rcp(R x);
template <> __device__ __forceinline__ double eval_rcp<double>(double x) { return 1.0 / x; }
template <> __device__ __forceinline__ float eval_rcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }
template <class R> __device__ __forceinline__ R eval_sqrt(R x);
template <> __device__ __forceinline__ double eval_sqrt<double>(double x) { return sqrt(x); }
template <> __device__ __forceinline__ float eval_sqrt<float>(float x) { return __builtin_amdgcn_sqrtf(x); }

// 1 / sqrt(x): in FP64 the hardware estimate refined by one third-order
// step (error about one ulp), in FP32 the hardware form.
template <class R> __device__ __forceinline__ R eval_rsqrt(R x);
template <> __device__ __forceinline__ double eval_rsqrt<double>(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x, y * y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}
template <> __device__ __forceinline__ float eval_rsqrt<float>(float x) { return __builtin_amdgcn_rsqf(x); }

// A table entry at t = T - (i + 1/2); R = double, or float for the
// reduced-precision quartets (table in FP32)
template <class R>
__device__ __forceinline__ R rys_poly(const R *__restrict__ c, R t) {
  R v = c[CQX_RYS_NCOEF - 1];
#pragma unroll
  for (int k = CQX_RYS_NCOEF - 2; k >= 0; --k) v = fma(t, v, c[k]);
  return v;
}

// The n-root section of the table: its offset and length (entries)
__host__ __device__ constexpr int rys_tab_off(int n) {
  int off = 0;
  for (int k = 1; k < n; ++k) off += (34 + 6 * k) * 2 * k * CQX_RYS_NCOEF;
  return off;
}
__host__ __device__ constexpr int rys_tab_len(int n) { return (34 + 6 * n) * 2 * n * CQX_RYS_NCOEF; }

// All n roots and weights, n known at compile time; tabn points at the
// table's n-root section (global memory or an LDS copy of it).
template <int N, class R>
__device__ __forceinline__ void rys_roots_sec(R T, const R *__restrict__ tabn, R *__restrict__ x,
                                              R *__restrict__ w) {
  constexpr int kTcut = 34 + 6 * N;
  if (T >= (R)kTcut) {
    const R rs = eval_rsqrt<R>(T), rt = rs * rs;
#pragma unroll
    for (int r = 0; r < N; ++r) {
      x[r] = (R)cqx_rys_asym_x[N][r] * rt;
      w[r] = (R)cqx_rys_asym_w[N][r] * rs;
    }
  } else {
    const int i = (int)T;
    const R t = T - ((R)i + (R)0.5);
    const R *c = tabn + (size_t)i * (2 * N * CQX_RYS_NCOEF);
#pragma unroll
    for (int r = 0; r < N; ++r) {
      x[r] = rys_poly<R>(c + r * CQX_RYS_NCOEF, t);
      w[r] = rys_poly<R>(c + (N + r) * CQX_RYS_NCOEF, t);
    }
  }
}

// The row kernels' own form of the table: LDS copies, read by every lane for
// itself, 14 coefficients a value, keep the LDS (128 bytes a cycle and CU) as
// busy as the ALUs where there is little else to do per quadrature point.  On
// half intervals of T 11 terms leave the FP64 series' error at their rounding
// (one root, largest relative error over the table 2.1e-16, mean 5.3e-17, as
// with 14 on unit intervals), and 6 terms the FP32 one's (1.2e-7 both ways).
// Layout [half interval][power][value]: nodes and weights of one power lie
// side by side; an (ss|ss) class keeps the weights alone (WONLY).  The FP64
// section of two roots grows from 20.6 to 32.4 KB, so a block that has no
// room to spare (ROOM false) keeps unit intervals: 32 water clusters 27.0 ->
// 25.5 ms a build, but GHF (H2O)16 / cc-pVDZ 8.6 -> 9.1, its (ds|ps) rows then
// not fitting any more.  FP64 sections of three roots and more stay as they
// are (35 -> 55 KB).
template <int N, class R, bool WONLY, bool ROOM>
struct RysRow {
  static constexpr bool kF32 = sizeof(R) == 4;
  static constexpr bool kHalf = kF32 || N == 1 || (N == 2 && ROOM);
  static constexpr int kCoef = kF32 ? 6 : 11;
  static constexpr int kVal = 2 * N, kFirst = WONLY ? N : 0, kKeep = kVal - kFirst;
  static constexpr int kLen = kHalf ? (34 + 6 * N) * 2 * kCoef * kKeep : rys_tab_len(N);
  // entry e of the LDS copy in the table
  static __device__ __forceinline__ int src(int e) {
    if (!kHalf) return rys_tab_off(N) + e;
    int o = 0;
    for (int k = 1; k < N; ++k) o += (34 + 6 * k) * 2 * kCoef * 2 * k;
    return o + e / kKeep * kVal + kFirst + e % kKeep;
  }
};
template <int N, class R, bool WONLY, bool ROOM>
__device__ __forceinline__ void rys_roots_row(R T, const R *__restrict__ tabn, R *__restrict__ x, R *__restrict__ w) {
  using S = RysRow<N, R, WONLY, ROOM>;
  if constexpr (!S::kHalf) {
    rys_roots_sec<N, R>(T, tabn, x, w);
  } else if (T >= (R)(34 + 6 * N)) {
    const R rs = eval_rsqrt<R>(T), rt = rs * rs;
#pragma unroll
    for (int r = 0; r < N; ++r) {
      x[r] = (R)cqx_rys_asym_x[N][r] * rt;
      w[r] = (R)cqx_rys_asym_w[N][r] * rs;
    }
  } else {
    const int i = (int)(T + T);
    const R t = T - ((R)0.5 * (R)i + (R)0.25);
    const R *c = tabn + i * (S::kCoef * S::kKeep);
    R v[S::kKeep];
#pragma unroll
    for (int r = 0; r < S::kKeep; ++r) v[r] = c[(S::kCoef - 1) * S::kKeep + r];
#pragma unroll
    for (int k = S::kCoef - 2; k >= 0; --k)
#pragma unroll
      for (int r = 0; r < S::kKeep; ++r) v[r] = fma(t, v[r], c[k * S::kKeep + r]);
#pragma unroll
    for (int r = 0; r < N; ++r) {
      if (!WONLY) x[r] = v[r];
      w[r] = v[N - S::kFirst + r];
    }
  }
}

// All n roots and weights, n known at compile time.
template <int N, class R>
__device__ __forceinline__ void rys_roots(R T, const R *__restrict__ tab, R *__restrict__ x,
                                          R *__restrict__ w) {
  constexpr int kTcut = 34 + 6 * N, kOff = rys_tab_off(N);
  if (T >= (R)kTcut) {
    const R rs = eval_rsqrt<R>(T), rt = rs * rs;
#pragma unroll
    for (int r = 0; r < N; ++r) {
      x[r] = (R)cqx_rys_asym_x[N][r] * rt;
      w[r] = (R)cqx_rys_asym_w[N][r] * rs;
    }
  } else {
    const int i = (int)T;
    const R t = T - ((R)i + (R)0.5);
    const R *c = tab + kOff + (size_t)i * (2 * N * CQX_RYS_NCOEF);
#pragma unroll
    for (int r = 0; r < N; ++r) {
      x[r] = rys_poly<R>(c + r * CQX_RYS_NCOEF, t);
      w[r] = rys_poly<R>(c + (N + r) * CQX_RYS_NCOEF, t);
    }
  }
}

// Root r (and its weight) of an N-point rule, N known at compile time; tabn
// points at the table's N-root section.
template <int N, class R>
__device__ __forceinline__ void rys_root_sec(R T, const R *__restrict__ tabn, int r, R &x, R &w) {
  constexpr int kTcut = 34 + 6 * N;
  if (T >= (R)kTcut) {
    const R rs = eval_rsqrt<R>(T);
    x = (R)cqx_rys_asym_x[N][r] * (rs * rs);
    w = (R)cqx_rys_asym_w[N][r] * rs;
  } else {
    const int i = (int)T;
    const R t = T - ((R)i + (R)0.5);
    const R *c = tabn + (size_t)i * (2 * N * CQX_RYS_NCOEF);
    x = rys_poly<R>(c + r * CQX_RYS_NCOEF, t);
    w = rys_poly<R>(c + (N + r) * CQX_RYS_NCOEF, t);
  }
}
// the same from the whole table
template <int N, class R>
__device__ __forceinline__ void rys_root(R T, const R *__restrict__ tab, int r, R &x, R &w) {
  rys_root_sec<N, R>(T, tab + rys_tab_off(N), r, x, w);
}

// Root r (and its weight) of an n-point rule, n (<= CQX_RYS_NMAX) known at
// run time.
__device__ __forceinline__ void rys_root_rt(int n, int r, double T,
                                            const double *__restrict__ tab,
                                            double &x, double &w) {
  const int tcut = 34 + 6 * n;  // 40, 46, ..., 88
  if (T >= (double)tcut) {
    const double rs = eval_rsqrt<double>(T);
    x = cqx_rys_asym_x_dev(n, r) * (rs * rs);
    w = cqx_rys_asym_w_dev(n, r) * rs;
  } else {
    int off = 0;
    for (int k = 1; k < n; ++k) off += (34 + 6 * k) * 2 * k * CQX_RYS_NCOEF;
    const int i = (int)T;
    const double t = T - ((double)i + 0.5);
    const double *c = tab + off + (size_t)i * (2 * n * CQX_RYS_NCOEF);
    x = rys_poly<double>(c + r * CQX_RYS_NCOEF, t);
    w = rys_poly<double>(c + (n + r) * CQX_RYS_NCOEF, t);
  }
}

}  // namespace cqx
