// A host-only stand-in for the HIP runtime entry points libgsq.so calls, for tests of its host side
// without a GPU: every launch, allocation and function attribute is recorded instead of done.
// Device pointers are made-up addresses. Loaded with RTLD_GLOBAL before libgsq.so, whose references
// then resolve here (the registration of its code object still goes to the real runtime).
#include <stdint.h>
#include <string.h>
#include <unistd.h>

#include <mutex>
#include <vector>

struct dim3_t { uint32_t x, y, z; };

namespace {
std::mutex mu;
struct Launch { int thread; const void* kernel; };
std::vector<Launch> launches;
std::vector<size_t> mallocs;
struct Attr { int device; const void* kernel; };
std::vector<Attr> attrs;
uintptr_t next_address = uintptr_t(1) << 40;
thread_local int thread_id = 0;
thread_local struct { dim3_t grid, block; size_t shared; void* stream; } config;
}  // namespace

extern "C" {
// set by the tests
int stub_device = 0, stub_capturing = 0, stub_attr_fails = 0, stub_launch_us = 0;
size_t stub_malloc_limit = SIZE_MAX;  // larger requests fail

void stub_thread(int id) { thread_id = id; }
int stub_launches(void) { return (int)launches.size(); }
int stub_launch_thread(int i) { return launches[i].thread; }
const void* stub_launch_kernel(int i) { return launches[i].kernel; }
int stub_mallocs(void) { return (int)mallocs.size(); }
size_t stub_malloc_bytes(int i) { return mallocs[i]; }
int stub_attrs(void) { return (int)attrs.size(); }
int stub_attr_device(int i) { return attrs[i].device; }
void stub_clear(void) { launches.clear(); mallocs.clear(); attrs.clear(); }

int hipGetDevice(int* d) { *d = stub_device; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  if (n > stub_malloc_limit) { *p = nullptr; return 2; }
  mallocs.push_back(n);
  *p = (void*)next_address;
  next_address += (n + 4095) / 4096 * 4096;
  return 0;
}
int hipFree(void*) { return 0; }
int hipMemcpy(void*, const void*, size_t, int) { return 0; }
int hipMemset(void*, int, size_t) { return 0; }
int hipStreamIsCapturing(void*, int* st) { *st = stub_capturing; return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = (void*)(uintptr_t(1) << 39); return 0; }
int hipFuncGetAttributes(void* a, const void*) { memset(a, 0, 56); return 0; }
int hipFuncSetAttribute(const void* k, int, int) {
  std::lock_guard<std::mutex> lk(mu);
  if (stub_attr_fails) return 1;
  attrs.push_back({stub_device, k});
  return 0;
}
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int) { return "stub"; }
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t shared, void* stream) {
  config = {grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* shared, void** stream) {
  *grid = config.grid; *block = config.block; *shared = config.shared; *stream = config.stream;
  return 0;
}
int hipLaunchKernel(const void* k, dim3_t, dim3_t, void**, size_t, void*) {
  {
    std::lock_guard<std::mutex> lk(mu);
    launches.push_back({thread_id, k});
  }
  if (stub_launch_us) usleep(stub_launch_us);  // lets another thread's launch in between
  return 0;
}
}
