// Checks of solar_hostcopy.cpp on the CPU (hip_stub.hpp); the argument names
// one, the exit status is 0 if it holds.
#include "hip_stub.hpp"
#include "solar_internal.hpp"

#include <algorithm>
#include <cstdio>
#include <functional>
#include <new>
#include <string>
#include <thread>
#include <vector>

// Allocations of this thread until one fails (once).
static thread_local int fail_new = -1;
void* operator new(size_t n) {
  if (fail_new >= 0 && fail_new-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

constexpr size_t kBytes = (size_t(41) << 20) + 24;  // above the staging's least size, no whole pieces

int failures = 0;
void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  ++failures;
}

struct Arrays {
  std::vector<char> src, dst;
  void* dev = nullptr;
  explicit Arrays(char seed, size_t bytes = kBytes) : src(bytes), dst(bytes) {
    for (size_t x = 0; x < bytes; ++x) src[x] = static_cast<char>(x * 7 + x / 4096 + seed);
    (void)hipMalloc(&dev, bytes);
  }
  ~Arrays() { (void)hipFree(dev); }
  // the second has the staging
  bool round_trips(solar::HostCopy& h, int device = 0) { return round_trip(h, device) && round_trip(h, device); }
  bool round_trip(solar::HostCopy& h, int device = 0) {
    const hipStream_t st = stub::stream_of(device);
    if (h.to_device(dev, src.data(), src.size(), device, st) != hipSuccess) return false;
    if (h.to_host(dst.data(), dev, dst.size(), device, st) != hipSuccess) return false;
    return src == dst;
  }
};

// A handle of another device than the caller's current one.
void other_device() {
  solar::HostCopy h;
  Arrays a(1);
  stub::device = 0;
  check(a.round_trips(h, 1) && a.round_trip(h, 1), "copies for device 1 while device 0 is current");
  check(stub::device == 0, "the caller's current device stays");
  check(hipGetLastError() == hipSuccess, "no error left behind");
}

// Host arrays that are pinned, or memory of a device: the runtime copies those
// by itself, in one piece.
void known_memory() {
  solar::HostCopy h;
  Arrays a(2);
  void* mem[2] = {nullptr, nullptr};
  (void)hipHostMalloc(&mem[0], kBytes, 0);
  (void)hipMalloc(&mem[1], kBytes);
  for (void* p : mem) {
    const size_t from = 4096;  // the middle of the allocation
    stub::watch = static_cast<char*>(p) + from;
    stub::watch_bytes = kBytes - from;
    std::memcpy(static_cast<char*>(p) + from, a.src.data(), kBytes - from);
    stub::copies = stub::direct = 0;
    check(h.to_device(a.dev, stub::watch, kBytes - from, 0, stub::stream_of(0)) == hipSuccess, "to the device");
    check(stub::copies == 1 && stub::direct == 1, "one copy from the array itself");
    std::memset(static_cast<char*>(p) + from, 0, kBytes - from);
    check(h.to_host(static_cast<char*>(p) + from, a.dev, kBytes - from, 0, stub::stream_of(0)) == hipSuccess, "back");
    check(stub::copies == 2 && stub::direct == 2, "one copy into the array itself");
    check(std::memcmp(stub::watch, a.src.data(), kBytes - from) == 0, "the same bytes");
  }
  stub::watch = nullptr;
  (void)hipHostFree(mem[0]);
  (void)hipFree(mem[1]);
}

// The staging cannot be made: the copy goes on without it, and nothing of the
// failure stays behind.
void events_fail() {
  for (int k : {0, 3, 7}) {
    solar::HostCopy h;
    Arrays a(3);
    stub::fail_event = k;
    check(a.round_trips(h), "copies while an event creation fails");
    check(hipGetLastError() == hipSuccess, "no error left for the next launch to report");
    stub::fail_event = -1;
    check(a.round_trips(h), "copies afterwards");
  }
  check(stub::events.empty() && stub::pinned.empty(), "everything is given back");
}

// No memory for a thread's record: the calling thread does that part itself.
void no_thread() {
  solar::HostCopy h;
  Arrays a(4);
  check(a.round_trips(h), "with threads");
  for (int k = 0; k < 3; ++k) {
    fail_new = k;
    check(h.to_device(a.dev, a.src.data(), kBytes, 0, stub::stream_of(0)) == hipSuccess, "to the device");
    fail_new = k;
    check(h.to_host(a.dst.data(), a.dev, kBytes, 0, stub::stream_of(0)) == hipSuccess, "back");
    fail_new = -1;
    check(a.src == a.dst, "the same bytes");
    std::fill(a.dst.begin(), a.dst.end(), 0);
  }
}

// A second thread's copy in the middle of the first one's, on the same object.
solar::HostCopy* shared_copy;
Arrays* shared_array;
bool shared_ok;
void copy_meanwhile() {
  std::thread([] { shared_ok = shared_array->round_trip(*shared_copy); }).join();
}
void two_threads() {
  solar::HostCopy h;
  Arrays a(5), b(6);
  check(a.round_trips(h), "alone");
  shared_copy = &h;
  shared_array = &b;
  for (int down = 0; down < 2; ++down) {
    shared_ok = false;
    stub::on_copy = copy_meanwhile;
    std::memset(down ? static_cast<void*>(a.dst.data()) : a.dev, 0, kBytes);
    check((down ? h.to_host(a.dst.data(), a.dev, kBytes, 0, stub::stream_of(0))
                : h.to_device(a.dev, a.src.data(), kBytes, 0, stub::stream_of(0))) == hipSuccess, "the first copy");
    check(std::memcmp(down ? static_cast<void*>(a.dst.data()) : a.dev, a.src.data(), kBytes) == 0, "the first array is whole");
    check(shared_ok, "the second array is whole");
  }
}

// Before its pieces, a staged copy waits for the stream and sends two small
// uploads, each waited for.
void settled_stream() {
  solar::HostCopy h;
  Arrays a(7);
  check(a.round_trips(h), "round trips");
  for (bool down : {true, false}) {
    stub::n_asked = 0;
    check((down ? h.to_host(a.dst.data(), a.dev, kBytes, 0, stub::stream_of(0))
                : h.to_device(a.dev, a.src.data(), kBytes, 0, stub::stream_of(0))) == hipSuccess, "a copy");
    const int want[] = {stub::kWait, hipMemcpyHostToDevice, stub::kWait, hipMemcpyHostToDevice, stub::kWait};
    check(stub::n_asked > 5 && std::equal(want, want + 5, stub::asked),
          "wait, upload, wait, upload, wait");
  }
}

// The first copy makes the staging only where it pays for it, a second one does.
void first_copy() {
  for (bool down : {false, true}) {
    solar::HostCopy h;
    Arrays a(8);
    char* host = down ? a.dst.data() : a.src.data();
    stub::watch = host;
    stub::watch_bytes = kBytes;
    int plain = 0;
    for (; plain < 100; ++plain) {
      stub::direct = 0;
      check((down ? h.to_host(host, a.dev, kBytes, 0, stub::stream_of(0))
                  : h.to_device(a.dev, host, kBytes, 0, stub::stream_of(0))) == hipSuccess, "a copy");
      if (stub::direct == 0) break;
    }
    check(plain == 1, "the first copy of a new object goes without the staging, the second with it");
    stub::watch = nullptr;
  }
  solar::HostCopy h;
  Arrays a(9, size_t(90) << 20);
  stub::watch = a.dst.data();
  stub::watch_bytes = a.dst.size();
  stub::direct = 0;
  check(h.to_host(a.dst.data(), a.dev, a.dst.size(), 0, stub::stream_of(0)) == hipSuccess, "a large download");
  check(stub::direct == 0, "a download that pays for the staging by itself makes it");
}

}  // namespace

int main(int argc, char** argv) {
  const std::vector<std::pair<std::string, std::function<void()>>> all = {
      {"other_device", other_device},
      {"known_memory", known_memory},
      {"events_fail", events_fail},
      {"no_thread", no_thread},
      {"two_threads", two_threads},
      {"settled_stream", settled_stream},
      {"first_copy", first_copy},
  };
  for (const auto& c : all)
    if (argc == 2 && c.first == argv[1]) {
      c.second();
      return failures != 0;
    }
  return 2;
}
