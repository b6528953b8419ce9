// A HIP runtime without a device, for tests of the host side of a build:
// device memory is host memory, kernels do nothing, and streams and events are
// followed so that a test can ask what is still in flight.  Loaded before
// libcqx.so with its symbols global.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

using Clock = std::map<void *, long long>;  // per stream: its launches known to precede
struct Alloc { size_t n; bool written; };

std::map<char *, Alloc> allocs;
std::map<const void *, std::string> names;
std::map<void *, Clock> streams, events;
Clock issued, done;
long long fail_in = 0, word = 0, unwritten = 0;
float elapsed = 1.0f;
dim3 cfg_grid, cfg_block;
size_t cfg_lds;
hipStream_t cfg_stream;
char handles[1 << 16], *next_handle = handles;
alignas(256) char symbol[64 << 20];

Alloc *find(const void *p) {
  auto it = allocs.upper_bound((char *)p);
  if (it == allocs.begin()) return nullptr;
  --it;
  return (char *)p < it->first + it->second.n ? &it->second : nullptr;
}
void merge(Clock &a, const Clock &b) {
  for (const auto &x : b)
    if (a[x.first] < x.second) a[x.first] = x.second;
}
hipError_t copy(void *dst, const void *src, size_t n, hipMemcpyKind kind) {
  if (kind == hipMemcpyDeviceToHost && word && n % 8 == 0)
    for (size_t k = 0; k < n; k += 8) std::memcpy((char *)dst + k, &word, 8);
  else
    std::memmove(dst, src, n);
  if (Alloc *a = find(dst)) a->written = true;
  return hipSuccess;
}

}  // namespace

extern "C" {

// the k-th allocation from now fails (0: none)
void fake_fail_malloc(long long k) { fail_in = k; }
// every 8 bytes read back from the device become w (0: memory as it is)
void fake_read_back(long long w) { word = w; }
// launches not known to have ended
long long fake_in_flight() {
  long long n = 0;
  for (const auto &x : issued) n += x.second - done[x.first];
  return n;
}
// launches of list and candidate kernels whose table was never uploaded
long long fake_unwritten_tables() { return unwritten; }

void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *) {
  names[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  cfg_grid = g;
  cfg_block = b;
  cfg_lds = lds;
  cfg_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = cfg_grid;
  *b = cfg_block;
  *lds = cfg_lds;
  *s = cfg_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s) {
  streams[s][s] = ++issued[s];
  const std::string &n = names[f];
  if (n.find("quartet_lists_kernel") != std::string::npos || n.find("candidates_kernel") != std::string::npos) {
    const Alloc *a = find(*(void **)args[0]);
    if (!a || !a->written) ++unwritten;
  }
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (fail_in && --fail_in == 0) return hipErrorOutOfMemory;
  *p = std::calloc(n ? n : 1, 1);
  allocs[(char *)*p] = {n ? n : 1, false};
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  allocs.erase((char *)p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return copy(d, s, n, k); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)next_handle++;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  merge(done, streams[s]);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  merge(streams[s], events[e]);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t)next_handle++;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  events[e] = streams[s];
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  merge(done, events[e]);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = elapsed;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 65536;
  return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) {
  *a = hipFuncAttributes{};
  a->numRegs = 128;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = symbol;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  if (!find(p)) return hipErrorInvalidValue;
  *a = hipPointerAttribute_t{};
  a->type = hipMemoryTypeDevice;
  return hipSuccess;
}

}  // extern "C"
