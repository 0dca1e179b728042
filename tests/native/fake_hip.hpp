// The HIP runtime functions that the library calls, on host memory, so that its
// host side runs without a GPU: allocations are calloc'd blocks, copies are
// memcpy, kernels are named and passed to a hook, streams and events are
// counted handles.  Defined in an executable that exports its symbols, they
// take the place of the runtime's.
#pragma once
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

struct Dim3 {
  uint32_t x, y, z;
};

namespace fake {
struct Launch {
  std::string name;  // mangled
  Dim3 grid, block;
  void **args;
};
inline std::mutex mu;
inline std::map<uintptr_t, size_t> blocks;  // device allocations alive
// (filled by the libraries' constructors, before this program's)
inline std::map<const void *, std::string> &kernels() {
  static std::map<const void *, std::string> k;
  return k;
}
inline int events = 0, streams = 0;
inline int device = 0, cus = 256;
inline int fail_malloc = 0;      // the n-th hipMalloc from now fails, and those after it
inline int last_error = 0;
inline std::function<void(const Launch &)> on_launch;
inline std::function<void(void *)> on_record;
inline std::function<float(void *, void *)> elapsed;

inline bool is_device(const void *p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.upper_bound((uintptr_t)p);
  if (it == blocks.begin()) return false;
  --it;
  return (uintptr_t)p < it->first + it->second;
}
inline size_t held() {
  std::lock_guard<std::mutex> lk(mu);
  return blocks.size();
}
}  // namespace fake

extern "C" {
struct Config {
  Dim3 g, b;
  size_t shm;
  void *stream;
};
inline thread_local std::vector<Config> config;

void **__hipRegisterFatBinary(const void *) {
  static void *h[4];
  return h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  fake::kernels()[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t shm, void *s) {
  config.push_back({g, b, shm, s});
  return 0;
}
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *shm, void **s) {
  *g = config.back().g;
  *b = config.back().b;
  *shm = config.back().shm;
  *s = config.back().stream;
  config.pop_back();
  return 0;
}
int hipLaunchKernel(const void *fn, Dim3 g, Dim3 b, void **args, size_t, void *) {
  if (fake::on_launch) fake::on_launch({fake::kernels()[fn], g, b, args});
  return 0;
}
int hipMalloc(void **p, size_t n) {
  if (fake::fail_malloc > 0 && --fake::fail_malloc == 0) {
    fake::fail_malloc = 1;
    return fake::last_error = 2;  // hipErrorOutOfMemory
  }
  *p = std::calloc(1, n);
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::blocks[(uintptr_t)*p] = n;
  return 0;
}
int hipFree(void *p) {
  std::lock_guard<std::mutex> lk(fake::mu);
  if (p && !fake::blocks.erase((uintptr_t)p)) std::abort();  // (not ours, or freed twice)
  std::free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(1, n);
  return 0;
}
int hipHostFree(void *p) {
  std::free(p);
  return 0;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
  if (!d || !s) return 1;
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int,
                     void *) {
  for (size_t r = 0; r < h; r++) std::memcpy((char *)d + r * dp, (const char *)s + r * sp, w);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) {
  if (!d) return 1;
  std::memset(d, v, n);
  return 0;
}
int hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = size_t(1) << 36;
  return 0;
}
int hipPointerGetAttributes(void *attr, const void *p) {
  if (!fake::is_device(p)) return 1;
  *(int *)attr = 2;  // the first member: hipMemoryTypeDevice
  return 0;
}
int hipGetSymbolAddress(void **d, const void *s) {
  *d = const_cast<void *>(s);
  return 0;
}
int hipGetDevice(int *d) {
  *d = fake::device;
  return 0;
}
int hipDeviceGetAttribute(int *v, int, int) {
  *v = fake::cus;
  return 0;
}
int hipFuncGetAttributes(void *, const void *) { return 1; }
const char *hipGetErrorString(int) { return "failed"; }
int hipGetLastError() {
  const int e = fake::last_error;
  fake::last_error = 0;
  return e;
}
int hipStreamCreateWithFlags(void **s, unsigned) {
  fake::streams++;
  *s = std::malloc(1);
  return 0;
}
int hipStreamDestroy(void *s) {
  fake::streams--;
  std::free(s);
  return 0;
}
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipEventCreateWithFlags(void **e, unsigned) {
  fake::events++;
  *e = std::malloc(1);
  return 0;
}
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) {
  fake::events--;
  std::free(e);
  return 0;
}
int hipEventRecord(void *e, void *) {
  if (fake::on_record) fake::on_record(e);
  return 0;
}
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) {
  *ms = fake::elapsed ? fake::elapsed(a, b) : 1.0f;
  return 0;
}
}
