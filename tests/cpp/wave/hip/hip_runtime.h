// A 64-lane wave on the CPU, for tests that run the wave-wide device
// functions of the kernel headers: one thread per lane, meeting at a barrier
// where the lanes exchange values or wait for each other's LDS writes.  Only
// what those functions use; every lane must reach each of these calls.
#pragma once

#include <algorithm>
#include <atomic>
#include <barrier>
#include <cmath>
#include <thread>
#include <vector>

#define __device__
#define __host__
#define __constant__
#define __forceinline__ inline

using std::fma;
using std::max;
using std::min;

namespace host_wave {

inline std::barrier<> meet(64);
inline long long slot[64];
inline thread_local int lane;

template <class F>
void run(const F &f) {
  std::vector<std::thread> t;
  for (int l = 0; l < 64; ++l)
    t.emplace_back([&f, l] {
      lane = l;
      f(l);
    });
  for (auto &x : t) x.join();
}
inline long long from_first(long long v) {
  slot[lane] = v;
  meet.arrive_and_wait();
  const long long r = slot[0];
  meet.arrive_and_wait();
  return r;
}

}  // namespace host_wave

inline unsigned long long __ballot(bool p) {
  host_wave::slot[host_wave::lane] = p;
  host_wave::meet.arrive_and_wait();
  unsigned long long m = 0;
  for (int l = 0; l < 64; ++l) m |= (unsigned long long)host_wave::slot[l] << l;
  host_wave::meet.arrive_and_wait();
  return m;
}
inline void unsafeAtomicAdd(double *p, double v) { std::atomic_ref<double>(*p).fetch_add(v); }

#define __builtin_amdgcn_readfirstlane(x) ((int)host_wave::from_first(x))
#define __builtin_amdgcn_wave_barrier() host_wave::meet.arrive_and_wait()
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_global_atomic_fadd_f64(p, v) unsafeAtomicAdd(p, v)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
#define __builtin_amdgcn_rsq(x) (1.0 / std::sqrt(x))
