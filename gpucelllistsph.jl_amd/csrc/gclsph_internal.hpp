// Internal declarations shared by the HIP translation units of libgclsph.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

namespace gclsph {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

// Status codes returned through the C ABI.
enum : int {
  kOk = 0,
  kErrArgument = -1,   // bad argument / dimension / length (reference: error(...))
  kErrHip = -2,        // HIP runtime failure
  kErrState = -3,      // call not valid in the object's state (e.g. pair view past capacity)
  kErrNoDevice = -4,
  kErrUnsupported = -5,
};

#define GCL_HIP(call)                                                                             \
  do {                                                                                            \
    hipError_t e_ = (call);                                                                       \
    if (e_ != hipSuccess)                                                                         \
      throw ::gclsph::Error(::gclsph::kErrHip, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define GCL_CHECK(cond, code, msg)                                 \
  do {                                                             \
    if (!(cond)) throw ::gclsph::Error((code), std::string(msg));  \
  } while (0)

// Message returned by gclsph_last_error() on this thread (api.hip).
void set_last_error(const std::string& m);

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n, int block = kBlock) {
  int64_t g = (n + block - 1) / block;
  return unsigned(g < 1 ? 1 : g);
}

// Per-device control block of an SPH problem.  Lives in device memory so a whole
// batch of steps runs without a host round trip; the host reads it once at the
// end of a `stepsolve` call.
struct StepCtl {
  int parity;         // which of the ping-pong state buffers is current
  int rebuild;        // rebuild the cell order at the start of the next step; within a step
                      // that does, parity and pparity are those before it until the commit
  int synced;         // half-step state equals the main state (no correction ran)
  int pparity;       // which ptype / id buffer is current (flipped by reorders only)
  int iter;          // 1-based iteration inside the running stepsolve call
  int nsteps;        // iterations of the running call
  long long updaten;  // rebuilds in this call
  long long mppcell;  // reference-visible max-particles-per-cell bookkeeping
  double dt;
  double etime;
  double maxcdx_out;  // max over steps of max |cdx|
};

// Device helpers ------------------------------------------------------------
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) {
    double w = __shfl_xor(v, o, 64);
    v = (w > v || w != w) ? w : v;
  }
  return v;
}

// atomic max of a non-negative double (NaN propagates: its bit pattern is larger
// than +Inf's).
__device__ inline void atomic_max_nonneg(unsigned long long* slot, double v) {
  unsigned long long b = __double_as_longlong(v);
  if (b & 0x8000000000000000ull) b = 0;  // -0.0 and negatives clamp to 0
  atomicMax(slot, b);
}

}  // namespace gclsph
