// Large copies between pageable host memory and the device.
//
// An array that the runtime knows (pinned, managed, a device's) is copied by it
// alone: staged, 35 MB of pinned memory took 1.0 ms instead of 0.63, 1 GB 21.5
// instead of 17.5.  A caller's array is mostly pageable and often fresh: the
// runtime's own copy of 830 MB into new arrays runs at 9 GB/s, one thread
// faulting their pages in.
// Here a few threads each take a contiguous part of the array through two
// pinned pieces of their own: while one piece is on the link, the other is
// copied to or from the array.  Measured on 830 MB of ensemble states: into
// new arrays 90 -> 27 ms, from arrays 29 -> 19 ms (eight threads 25 and 20).
#include "solar_internal.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace solar {

namespace {

constexpr int kThreads = 4;
constexpr size_t kPiece = size_t(4) << 20;
constexpr size_t kSettle = size_t(64) << 10;
constexpr size_t kLeast = size_t(32) << 20;  // below, starting the threads costs more than it gives
// A new staging costs about 3.4 ms, for the page faults of its first use (less
// where the runtime has such memory left over from another handle), and saves
// 0.012 ms a MB to the device and 0.07 from it.  So the first copy of an object
// makes it only where that copy pays for it; a second one shows a program that
// goes on copying.  First copies of a process, made at once and now: 35 MB to
// the device 4.5 -> 1.8 ms, 126 MB 6.6 -> 5.0, 35 MB from it 11.7 -> 4.3, as the
// runtime's own.
constexpr size_t kPaysUp = size_t(320) << 20, kPaysDown = size_t(56) << 20;

// Makes `device` current for the calling thread while it lives: events belong
// to the device that is current when they are made, and the caller's comes back.
class OnDevice {
 public:
  explicit OnDevice(int device) {
    int cur = -1;
    status_ = hipGetDevice(&cur);
    if (status_ == hipSuccess && cur != device) {
      status_ = hipSetDevice(device);
      if (status_ == hipSuccess) back_ = cur;
    }
  }
  ~OnDevice() {
    if (back_ >= 0) (void)hipSetDevice(back_);
  }
  OnDevice(const OnDevice&) = delete;
  OnDevice& operator=(const OnDevice&) = delete;
  hipError_t status() const { return status_; }

 private:
  hipError_t status_;
  int back_ = -1;
};

// Whether the runtime can put the memory at p on the link as it is.
bool runtime_knows(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // an ordinary array
  return false;
}

}  // namespace

struct HostCopy::Staging {
  char* buf = nullptr;  // pinned, kThreads x 2 pieces
  void* dev = nullptr;  // kSettle bytes on the device
  hipEvent_t ev[kThreads][2] = {};
  int made = 0;

  hipError_t make() {
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&buf), kThreads * 2 * kPiece, hipHostMallocDefault);
    if (e == hipSuccess) e = hipMalloc(&dev, kSettle);
    while (made < 2 * kThreads && e == hipSuccess) {
      e = hipEventCreateWithFlags(&ev[made / 2][made % 2], hipEventDisableTiming);
      if (e == hipSuccess) ++made;
    }
    return e;
  }
  ~Staging() {
    for (int x = 0; x < made; ++x) (void)hipEventDestroy(ev[x / 2][x % 2]);
    if (dev) (void)hipFree(dev);
    if (buf) (void)hipHostFree(buf);
  }

  // Readies the stream for the pieces.  A copy queued behind other work, or a
  // download that is the first copy after kernels, leaves a stream in a state
  // in which every copy that follows takes 0.12 ms more (4 MiB pieces at 20
  // GB/s instead of 47) until an upload of 64 KiB or more finds it idle; two of
  // them in a row ended it nearly always, one in most cases.  Measured over new
  // handles, without and with: 425 MB to the device 9.3 to 21.7 ms -> 9.4, from
  // it after steps 12 to 22 -> 10 to 13; 126 MB to the device 3.2 to 7.2 -> 3.1.
  hipError_t settle(hipStream_t st) {
    hipError_t e = hipStreamSynchronize(st);
    for (int x = 0; x < 2 && e == hipSuccess; ++x) {
      e = hipMemcpyAsync(dev, buf, kSettle, hipMemcpyHostToDevice, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
    }
    return e;
  }
};

HostCopy::~HostCopy() { delete s_; }

// One thread's part: pieces in order, alternating between the two buffers.
hipError_t HostCopy::part(int t, char* host, char* dev, size_t bytes, bool down, int device, hipStream_t st) {
  const OnDevice on(device);
  hipError_t e = on.status();
  const size_t np = (bytes + kPiece - 1) / kPiece;
  char* buf[2] = {s_->buf + (2 * t) * kPiece, s_->buf + (2 * t + 1) * kPiece};
  auto size = [&](size_t p) { return std::min(kPiece, bytes - p * kPiece); };
  // down: piece p is on the link while piece p - 1 is copied out; up: piece p
  // is copied in while piece p - 1 is on the link
  for (size_t p = 0; p < np + (down ? 1 : 2) && e == hipSuccess; ++p) {
    if (down) {
      if (p < np) {
        e = hipMemcpyAsync(buf[p & 1], dev + p * kPiece, size(p), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(s_->ev[t][p & 1], st);
      }
      if (p > 0 && e == hipSuccess) {
        e = hipEventSynchronize(s_->ev[t][(p - 1) & 1]);
        if (e == hipSuccess) std::memcpy(host + (p - 1) * kPiece, buf[(p - 1) & 1], size(p - 1));
      }
    } else {
      if (p >= 2) e = hipEventSynchronize(s_->ev[t][p & 1]);  // piece p - 2 has left its buffer
      if (p < np && e == hipSuccess) {
        std::memcpy(buf[p & 1], host + p * kPiece, size(p));
        e = hipMemcpyAsync(dev + p * kPiece, buf[p & 1], size(p), hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipEventRecord(s_->ev[t][p & 1], st);
      }
    }
  }
  return e;
}

hipError_t HostCopy::run(void* host, void* dev, size_t bytes, bool down, int device, hipStream_t st) {
  auto plain = [&]() {
    const hipError_t e = down ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st)
                              : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  };
  if (bytes < kLeast || runtime_knows(host)) return plain();
  const std::unique_lock<std::mutex> lock(mu_, std::try_to_lock);
  if (!lock) return plain();  // another thread's copy has the staging
  const OnDevice on(device);
  if (on.status() != hipSuccess) {
    (void)hipGetLastError();
    return plain();
  }
  if (!s_) {
    const bool first = !copied_;
    copied_ = true;
    if (first && bytes < (down ? kPaysDown : kPaysUp)) return plain();
    Staging* s = new (std::nothrow) Staging();
    if (!s || s->make() != hipSuccess) {
      delete s;
      (void)hipGetLastError();  // no failure of the staging for a later launch to report
      return plain();
    }
    s_ = s;
  }
  if (const hipError_t e = s_->settle(st)) return e;
  const size_t each = (bytes / kThreads + kPiece - 1) / kPiece * kPiece;
  hipError_t err[kThreads] = {};
  auto work = [&](int t) {
    const size_t a = std::min(bytes, each * t), b = t == kThreads - 1 ? bytes : std::min(bytes, each * (t + 1));
    err[t] = part(t, static_cast<char*>(host) + a, static_cast<char*>(dev) + a, b - a, down, device, st);
  };
  std::thread th[kThreads];
  for (int t = 1; t < kThreads; ++t) {
    try {
      th[t] = std::thread(work, t);
    } catch (...) {  // no thread to be had, or no memory for it: this one does the part
      work(t);
    }
  }
  work(0);
  for (int t = 1; t < kThreads; ++t)
    if (th[t].joinable()) th[t].join();
  for (hipError_t e : err)
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(st);  // nothing of the copy is in flight on return
      return e;
    }
  return hipSuccess;
}

}  // namespace solar
