// Helpers shared by the C-ABI translation units (not part of the ABI).
#pragma once
#include <hip/hip_runtime_api.h>

#include <mutex>
#include <string>
#include <vector>

#include "solar_kernels.hpp"
#include "solar_tables.hpp"

namespace solar {

// Records msg as this thread's last error (solar_last_error) and returns code.
int set_error(int code, const std::string& msg);
void clear_error();

// Device copies of the time-invariant tables; every allocation is appended to
// *allocs and its size added to *bytes.
int upload_tables(const Tables& t, DevTables* d, std::vector<void*>* allocs, size_t* bytes);

// The static device scratch of solar_compute_rhs_noalloc (solar_noalloc.hip):
// its size, and its address on `device` (the current device), looked up once
// per device.
size_t scratch_bytes();
hipError_t scratch_address(int device, void** addr);

// Copies between a caller's host array and the device, synchronous, ordered
// after the work on `st` (solar_hostcopy.cpp).  Large ones go through pinned
// staging (32 MiB) that the object makes when they are worth it and keeps; a copy
// that comes while another thread's has the staging goes without it.
class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy();
  hipError_t to_device(void* dev, const void* host, size_t bytes, int device, hipStream_t st) {
    return run(const_cast<void*>(host), dev, bytes, false, device, st);
  }
  hipError_t to_host(void* host, const void* dev, size_t bytes, int device, hipStream_t st) {
    return run(host, const_cast<void*>(dev), bytes, true, device, st);
  }

 private:
  struct Staging;
  Staging* s_ = nullptr;
  bool copied_ = false;  // there was a large copy
  std::mutex mu_;  // held by the copy that uses them
  hipError_t run(void* host, void* dev, size_t bytes, bool down, int device, hipStream_t st);
  hipError_t part(int t, char* host, char* dev, size_t bytes, bool down, int device, hipStream_t st);
};

}  // namespace solar
