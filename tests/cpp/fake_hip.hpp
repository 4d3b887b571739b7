// A HIP runtime without a device, for drivers of libitnbp.so that test its host code:
// defined in the executable, these functions take the place of the runtime's.  Kernels
// do nothing (device memory reads as zeros), and copies and fills run when the host
// waits, as an asynchronous copy may: a copy whose host memory is freed or changed
// before that reads something else (under the address sanitizer: ends the program).
#pragma once
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstring>
#include <functional>
#include <map>
#include <vector>

namespace fake {
struct Launch {
  dim3 grid, block;
  size_t lds;
  const char* kernel;  // mangled name
};
inline std::map<const void*, const char*>& kernels() {  // the library registers them before main
  static std::map<const void*, const char*> k;
  return k;
}
inline std::vector<Launch> config, launches;
inline std::vector<std::function<void()>> pending;
inline std::map<void*, size_t> allocated;
inline size_t free_bytes = 64ull << 30, largest_alloc = 0;
inline int changed_copies = 0;  // host-to-device copies whose source changed before they ran

inline hipError_t wait() {
  std::vector<std::function<void()>> p;
  p.swap(pending);
  for (auto& f : p) f();
  return hipSuccess;
}
inline bool on_device(const void* p) {
  auto it = allocated.upper_bound(const_cast<void*>(p));
  return it != allocated.begin() && (--it, (const char*)p < (char*)it->first + it->second);
}
}  // namespace fake

extern "C" {
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }
hipError_t hipStreamCreate(hipStream_t* s) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return fake::wait(); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return fake::wait(); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  n = std::max<size_t>(n, 1);
  void* q = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (q == MAP_FAILED) return hipErrorOutOfMemory;
  fake::allocated[q] = n;
  fake::largest_alloc = std::max(fake::largest_alloc, n);
  *p = q;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  (void)fake::wait();
  auto it = fake::allocated.find(p);
  if (it != fake::allocated.end()) {
    munmap(p, it->second);
    fake::allocated.erase(it);
  }
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = fake::free_bytes;
  *t = 288ull << 30;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  if (!fake::on_device(src)) {
    std::vector<char> then((const char*)src, (const char*)src + n);
    fake::pending.push_back([=, then = std::move(then)] {
      if (n && std::memcmp(src, then.data(), n) != 0) ++fake::changed_copies;
      std::memcpy(dst, then.data(), n);
    });
  } else
    fake::pending.push_back([=] { std::memcpy(dst, src, n); });
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* dst, int v, size_t n, hipStream_t) {
  fake::pending.push_back([=] {
    char* a = (char*)(((size_t)dst + 4095) & ~(size_t)4095);  // zeroed pages go back to the system
    char* e = (char*)(((size_t)dst + n) & ~(size_t)4095);
    if (v != 0 || a >= e) {
      std::memset(dst, v, n);
      return;
    }
    std::memset(dst, 0, a - (char*)dst);
    madvise(a, e - a, MADV_DONTNEED);
    std::memset(e, 0, (char*)dst + n - e);
  });
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t) {
  fake::config.push_back({grid, block, lds, ""});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = fake::config.back().grid;
  *block = fake::config.back().block;
  *lds = fake::config.back().lds;
  *s = nullptr;
  fake::config.pop_back();
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
  fake::kernels()[f] = name;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t) {
  fake::launches.push_back({grid, block, lds, fake::kernels()[f]});
  return hipSuccess;
}
}
