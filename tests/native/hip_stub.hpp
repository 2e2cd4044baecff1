// The HIP runtime calls that the library's host code makes, on the CPU: device
// memory is host memory, copies happen at once, and the rules a program can
// break are checked (an event belongs to the device that was current when it
// was made and is recorded on a stream of that device; errors stay pending
// until they are asked for).  For programs that test host code without a GPU.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace stub {

inline thread_local int device = 0;
inline thread_local hipError_t pending = hipSuccess;
inline std::mutex mu;
inline std::map<const char*, size_t> pinned, on_device;  // allocations: address, size
inline std::map<hipEvent_t, int> events;                 // device of each
// what was asked of the streams, in order: kinds of copies, kWait
constexpr int kWait = -1;
inline int asked[1024], n_asked = 0;
inline void ask(int what) {
  if (n_asked < 1024) asked[n_asked++] = what;
}
inline std::atomic<int> copies{0}, direct{0};  // all copies; those from or to the array `watch`
inline const char* watch = nullptr;
inline size_t watch_bytes = 0;
inline int fail_event = -1;  // event creations until one fails (once)
inline size_t device_limit = SIZE_MAX, device_used = 0;
inline void (*on_copy)() = nullptr;  // runs once, after the first copy

inline hipError_t ret(hipError_t e) {
  if (e != hipSuccess) pending = e;
  return e;
}
inline bool holds(const std::map<const char*, size_t>& m, const void* p) {
  auto it = m.upper_bound(static_cast<const char*>(p));
  if (it == m.begin()) return false;
  --it;
  return static_cast<const char*>(p) < it->first + it->second;
}
// a stream handle is its device's number plus 1 (the default stream: 0)
inline hipStream_t stream_of(int dev) { return reinterpret_cast<hipStream_t>(static_cast<uintptr_t>(dev + 1)); }
inline int device_of(hipStream_t s) { return s ? static_cast<int>(reinterpret_cast<uintptr_t>(s)) - 1 : device; }

}  // namespace stub

extern "C" {
inline __attribute__((used)) hipError_t hipGetDevice(int* d) { *d = stub::device; return hipSuccess; }
inline __attribute__((used)) hipError_t hipSetDevice(int d) { stub::device = d; return hipSuccess; }
inline __attribute__((used)) hipError_t hipGetLastError() {
  const hipError_t e = stub::pending;
  stub::pending = hipSuccess;
  return e;
}
inline __attribute__((used)) hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> l(stub::mu);
  *p = std::malloc(n);
  stub::pinned[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(stub::mu);
  if (!stub::pinned.erase(static_cast<char*>(p))) return stub::ret(hipErrorInvalidValue);
  std::free(p);
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(stub::mu);
  if (n > stub::device_limit - stub::device_used) return stub::ret(hipErrorOutOfMemory);
  *p = std::malloc(n ? n : 1);
  stub::device_used += n;
  stub::on_device[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> l(stub::mu);
  auto it = stub::on_device.find(static_cast<char*>(p));
  if (it == stub::on_device.end()) return p ? stub::ret(hipErrorInvalidValue) : hipSuccess;
  stub::device_used -= it->second;
  stub::on_device.erase(it);
  std::free(p);
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> l(stub::mu);
  if (stub::fail_event >= 0 && stub::fail_event-- == 0) return stub::ret(hipErrorOutOfMemory);
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  stub::events[*e] = stub::device;
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> l(stub::mu);
  if (!stub::events.erase(e)) return stub::ret(hipErrorInvalidHandle);
  std::free(reinterpret_cast<void*>(e));
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> l(stub::mu);
  auto it = stub::events.find(e);
  if (it == stub::events.end() || it->second != stub::device_of(s)) return stub::ret(hipErrorInvalidHandle);
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline __attribute__((used)) hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> l(stub::mu);
  stub::ask(stub::kWait);
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
  std::memcpy(d, s, n);
  ++stub::copies;
  const auto in = [](const void* p) {
    const char* c = static_cast<const char*>(p);
    return stub::watch && c >= stub::watch && c < stub::watch + stub::watch_bytes;
  };
  if (in(d) || in(s)) ++stub::direct;
  void (*f)() = nullptr;
  {
    std::lock_guard<std::mutex> l(stub::mu);
    stub::ask(kind);
    std::swap(f, stub::on_copy);
  }
  if (f) f();
  return hipSuccess;
}
inline __attribute__((used)) hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::lock_guard<std::mutex> l(stub::mu);
  std::memset(a, 0, sizeof(*a));
  a->type = stub::holds(stub::pinned, p)      ? hipMemoryTypeHost
            : stub::holds(stub::on_device, p) ? hipMemoryTypeDevice
                                              : hipMemoryTypeUnregistered;
  return hipSuccess;
}
}
