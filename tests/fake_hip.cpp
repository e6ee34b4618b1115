// A HIP runtime of bookkeeping alone, preloaded over the real one, so that the host
// code's choices (which kernels, which grids, what memory) can be seen without a
// GPU.  Device memory is addresses counted against FAKE_HIP_BYTES; launches and
// copies do nothing.  A line a call goes to FAKE_HIP_LOG:
//   malloc BYTES | free BYTES | launch KERNEL GX GY GZ BX BY BZ LDS
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <map>
#include <mutex>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
constexpr int kOk = 0, kOutOfMemory = 2;
std::mutex mu;
std::map<uintptr_t, size_t> held;
size_t in_use = 0;
uintptr_t next_addr = (uintptr_t)1 << 44;
int last_error = kOk;

size_t total() {
  const char* e = getenv("FAKE_HIP_BYTES");
  return e ? strtoull(e, nullptr, 10) : (size_t)288 << 30;
}
FILE* out() {
  static FILE* f = fopen(getenv("FAKE_HIP_LOG"), "a");
  return f;
}
}  // namespace

extern "C" {
int hipGetDeviceCount(int* n) { return *n = 1, kOk; }
int hipGetDevice(int* d) { return *d = 0, kOk; }
int hipSetDevice(int) { return kOk; }
int hipGetLastError() {
  const int e = last_error;
  last_error = kOk;
  return e;
}
int hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(mu);
  if (in_use + n > total()) return last_error = kOutOfMemory;
  held[next_addr] = n;
  *p = (void*)next_addr;
  next_addr += (n + 4095) / 4096 * 4096;
  in_use += n;
  fprintf(out(), "malloc %zu\n", n);
  return fflush(out()), kOk;
}
int hipFree(void* p) {
  std::lock_guard<std::mutex> l(mu);
  const auto it = held.find((uintptr_t)p);
  if (it == held.end()) return p ? 1 : kOk;
  fprintf(out(), "free %zu\n", it->second);
  in_use -= it->second;
  held.erase(it);
  return fflush(out()), kOk;
}
int hipMemGetInfo(size_t* f, size_t* t) {
  std::lock_guard<std::mutex> l(mu);
  *t = total();
  *f = *t - in_use;
  return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return *p = malloc(n), kOk; }
int hipHostFree(void* p) { return free(p), kOk; }
int hipMemcpyAsync(void*, const void*, size_t, int, void*) { return kOk; }
int hipMemcpy(void*, const void*, size_t, int) { return kOk; }
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = (void*)16, kOk; }
int hipStreamDestroy(void*) { return kOk; }
int hipStreamSynchronize(void*) { return kOk; }
int hipStreamIsCapturing(void*, int* s) { return *s = 0, kOk; }
int hipDeviceSynchronize() { return kOk; }
int hipEventCreate(void** e) { return *e = (void*)32, kOk; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = (void*)32, kOk; }
int hipEventDestroy(void*) { return kOk; }
int hipEventRecord(void*, void*) { return kOk; }
int hipEventSynchronize(void*) { return kOk; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 1.f, kOk; }
int hipStreamWaitEvent(void*, void*, unsigned) { return kOk; }
int hipGetSymbolAddress(void** p, const void*) { return *p = (void*)((uintptr_t)1 << 43), kOk; }
thread_local struct Config {
  Dim3 g, b;
  size_t lds;
  void* st;
} config;
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void* st) {
  config = {g, b, lds, st};
  return kOk;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** st) {
  *g = config.g;
  *b = config.b;
  *lds = config.lds;
  *st = config.st;
  return kOk;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3 b, void**, size_t lds, void*) {
  std::lock_guard<std::mutex> l(mu);
  Dl_info i{};
  const char* name = dladdr(f, &i) && i.dli_sname ? i.dli_sname : "?";
  fprintf(out(), "launch %s %u %u %u %u %u %u %zu\n", name, g.x, g.y, g.z, b.x, b.y, b.z, lds);
  return fflush(out()), kOk;
}
}
