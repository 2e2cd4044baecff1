// solar_ensemble.cpp on the CPU (hip_stub.hpp): what an ensemble allocates and
// which schedule it steps with, by the device memory there is.  The launchers
// are stand-ins that write down the stages they are asked for.
#include "hip_stub.hpp"
#include "../../include/solar_amd.h"
#include "solar_internal.hpp"

#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

static size_t reported = 0;  // free memory the runtime names, if not what there is
static std::string steps;  // per stage launch: stage, q buffer, qw buffer, stored-q or all

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { *s = stub::stream_of(0); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *t = stub::device_limit;
  *f = reported ? reported : stub::device_limit - stub::device_used;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = nullptr; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace solar {
int set_error(int code, const std::string& msg) { std::printf("%s\n", msg.c_str()); return code; }
void clear_error() {}
int upload_tables(const Tables&, DevTables*, std::vector<void*>*, size_t*) { return SOLAR_OK; }
hipError_t launch_stage_ens(const EnsMember* M, const int*, int, int, int, int, int stage, int cur, int wcur,
                            bool stored_q, hipStream_t) {
  if (stored_q && !M[0].qw[1]) return hipErrorInvalidValue;
  steps += std::to_string(stage) + std::to_string(cur) + std::to_string(wcur) + (stored_q ? "q " : "a ");
  return hipSuccess;
}
hipError_t launch_filter_ens(const EnsMember*, const int*, int, int, int, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_gather_ens(const EnsMember*, const int*, int, int, int, bool, int, bool, int, hipStream_t, int wcur,
                             double betar) {
  return (wcur >= 0) == (betar != 0.0) ? hipSuccess : hipErrorInvalidValue;
}
}  // namespace solar

// Arguments: the device memory in states of the ensemble, as a decimal number,
// and (optional) how much of it the runtime says is free.
// Prints the stages of a step, then ", " and the states' worth it allocated.
int main(int argc, char** argv) {
  const int nm = 2, n[nm] = {48, 64}, nr[nm] = {40, 30}, sponge[nm] = {3, 3};
  size_t state = 0;
  std::vector<double> gr, c2, rho0, g0;
  for (int m = 0; m < nm; ++m) {
    state += static_cast<size_t>(n[m]) * n[m] * nr[m] * 30 * sizeof(double);
    for (int k = 0; k < nr[m]; ++k) {
      gr.push_back(0.7 + 0.3 * k / (nr[m] - 1));
      c2.push_back(1.0);
      rho0.push_back(1.0);
      g0.push_back(0.0);
    }
  }
  if (argc < 2) return 2;
  if (argc > 2) reported = static_cast<size_t>(std::atof(argv[2]) * static_cast<double>(state));
  stub::device_limit = static_cast<size_t>(std::atof(argv[1]) * static_cast<double>(state));
  const double a_sponge[nm] = {0.1, 0.1}, dt[nm] = {1e-3, 1e-3};
  solar_ens* e = nullptr;
  if (solar_ens_create(&e, nm, n, nr, gr.data(), c2.data(), rho0.data(), g0.data(), sponge, a_sponge, dt)) return 1;
  if (solar_ens_rk4_async(e, 1)) return 1;
  std::printf("%s, %.0f\n", steps.c_str(), std::floor(static_cast<double>(stub::device_used) / static_cast<double>(state)));
  steps.clear();
  if (solar_ens_autotune(e, 1) || solar_ens_finalize(e)) return 1;
  return stub::device_used != 0 || hipGetLastError() != hipSuccess;
}
