// A block of GPU threads on the CPU, for tests that run the device functions
// and kernels of the headers: every thread runs up to the next barrier in
// turn, thread 0 first, so that a missing barrier shows the same way each
// time.  Only what those headers use; every thread (of the one wave, for the
// wave-wide calls) must reach each call that exchanges values or waits.
#pragma once

#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <functional>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __constant__
#define __shared__ static
#define __launch_bounds__(...)
#define __forceinline__ inline

using std::fma;
using std::max;
using std::min;

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
inline dim3 threadIdx(0), blockIdx(0), blockDim, gridDim;
enum hipError_t { hipSuccess, hipErrorNotSupported, hipErrorInvalidValue };
using hipStream_t = void *;
inline hipError_t hipGetLastError() { return hipSuccess; }
#define hipLaunchKernelGGL(...) ((void)0)

namespace host_wave {

inline std::vector<ucontext_t> thread;
inline ucontext_t scheduler;
inline std::function<void(int)> body;
inline std::vector<char> ended;
inline double slot[64];

inline void enter(int t) {
  body(t);
  ended[t] = 1;
}
// f(thread) for the threads of one block
inline void run(int n, const std::function<void(int)> &f) {
  constexpr size_t kStack = 256 << 10;
  static std::vector<char> stacks;
  stacks.resize(n * kStack);
  thread.assign(n, ucontext_t{});
  ended.assign(n, 0);
  body = f;
  blockDim.x = (unsigned)n;
  for (int t = 0; t < n; ++t) {
    getcontext(&thread[t]);
    thread[t].uc_stack.ss_sp = stacks.data() + t * kStack;
    thread[t].uc_stack.ss_size = kStack;
    thread[t].uc_link = &scheduler;
    makecontext(&thread[t], (void (*)())enter, 1, t);
  }
  for (bool more = true; more;) {
    more = false;
    for (int t = 0; t < n; ++t) {
      if (ended[t]) continue;
      threadIdx.x = (unsigned)t;
      swapcontext(&scheduler, &thread[t]);
      more = more || !ended[t];
    }
  }
}
inline void meet() { swapcontext(&thread[threadIdx.x], &scheduler); }
template <class T>
T from_lane(T v, int l) {
  slot[threadIdx.x & 63] = (double)v;
  meet();
  const T r = (T)slot[l];
  meet();
  return r;
}

}  // namespace host_wave

inline void __syncthreads() { host_wave::meet(); }
inline unsigned long long __ballot(bool p) {
  host_wave::slot[threadIdx.x & 63] = p;
  host_wave::meet();
  unsigned long long m = 0;
  for (int l = 0; l < 64; ++l) m |= (unsigned long long)(host_wave::slot[l] != 0.0) << l;
  host_wave::meet();
  return m;
}
inline double __shfl_xor(double v, int o) { return host_wave::from_lane(v, (threadIdx.x & 63) ^ o); }
inline void unsafeAtomicAdd(double *p, double v) { *p += v; }

#define __builtin_amdgcn_readfirstlane(x) host_wave::from_lane((int)(x), 0)
#define __builtin_amdgcn_wave_barrier() host_wave::meet()
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_global_atomic_fadd_f64(p, v) unsafeAtomicAdd(p, v)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
#define __builtin_amdgcn_rsq(x) (1.0 / std::sqrt(x))
