// The C ABI's host code (csrc/abi.hip) on a machine without a device: a
// stand-in HIP runtime whose one stream keeps what is launched until it is
// waited for, and stand-in launchers.  Pointers to "device" memory are host
// memory.  Launchers that no scenario reaches stay unresolved.
#pragma once
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <string>
#include <vector>

#include "../../include/pourover_hip.h"
#include "../../pour-over-coffee-lbm_amd/csrc/engine.h"

inline std::deque<std::function<void()>> queued;  // work of the stream, not yet done
inline std::vector<pol::StepArgs> steps;          // every stream-collide launch
inline int blocking_copies = 0;
inline int fail_after = -1;                       // launches that succeed before one fails (-1: all)

inline hipError_t launch(std::function<void()> work) {
  if (fail_after == 0) {
    fail_after = -1;
    return hipErrorLaunchFailure;
  }
  if (fail_after > 0) --fail_after;
  queued.push_back(std::move(work));
  return hipSuccess;
}
inline void wait_all() {
  while (!queued.empty()) {
    queued.front()();
    queued.pop_front();
  }
}

// ---- runtime ---------------------------------------------------------------
extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
// device memory comes as it was left
hipError_t hipMalloc(void** p, size_t n) { *p = memset(malloc(n), 0x5a, n); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipFree(void* p) { wait_all(); free(p); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  ++blocking_copies;
  wait_all();
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return launch([=] { memcpy(d, s, n); });
}
hipError_t hipStreamSynchronize(hipStream_t) { wait_all(); return hipSuccess; }
const char* hipGetErrorName(hipError_t) { return "error"; }
const char* hipGetErrorString(hipError_t) { return "error"; }
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
extern const char __hip_fatbin[1] = {0};
}

// ---- launchers ---------------------------------------------------------------
namespace pol {
hipError_t launch_stream_collide(int, const StepArgs& a, bool, const Grid&, hipStream_t) {
  steps.push_back(a);
  return launch([] {});
}
hipError_t launch_reduce_final(double*, uint32_t, double* out, hipStream_t) {
  return launch([=] { for (int i = 0; i < POL_NRED; ++i) out[i] = i; });
}
hipError_t launch_flux_fold(const double*, uint32_t, double* out, hipStream_t) {
  return launch([=] { *out = 0.5; });
}
hipError_t launch_zero_real(bool dbl, void* p, size_t n, hipStream_t) {
  return launch([=] { memset(p, 0, n * (dbl ? 8 : 4)); });
}
}  // namespace pol

#define CHECK(x)                                                   \
  do {                                                             \
    if (!(x)) {                                                    \
      printf("line %d: %s does not hold\n", __LINE__, #x);         \
      exit(1);                                                     \
    }                                                              \
  } while (0)

// A context of a closed box with cell flags, its buffers in host memory.
struct Box {
  static constexpr int nx = 8, ny = 4, nz = 4;
  static constexpr size_t cells = nx * ny * nz, state_bytes = POL_Q * cells * sizeof(float);
  std::vector<char> mem = std::vector<char>(16 * state_bytes);
  std::vector<uint32_t> flags = std::vector<uint32_t>(cells);
  pol_ctx* c = nullptr;
  char* at(double states) { return mem.data() + (size_t)(states * state_bytes); }
  explicit Box(uint32_t options = 0) {
    pol_desc d{};
    d.nx = nx; d.ny = ny; d.nz = nz;
    d.storage = POL_F32;
    d.options = POL_USE_FLAGS | options;
    d.tau = 0.6;
    CHECK(pol_create(&c, &d) == POL_OK);
    pol_buffers b{};
    b.f[0] = at(0);
    b.f[1] = at(1);
    b.cell_flags = flags.data();
    b.force = at(13);
    b.rho = at(14);
    b.u = at(14.5);
    CHECK(pol_bind(c, &b) == POL_OK);
  }
  ~Box() { pol_destroy(c); }
};
