// The part of HIP that csrc/blockscan.hpp and csrc/readback.hpp use, for the host:
// the threads of one block as fibers that run in turn and meet at the
// collectives, and streams and events that do what a test gives them to do.
#pragma once

#include <ucontext.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__ static  // one block at a time
#define __launch_bounds__(...)

// ---- runtime
enum hipError_t { hipSuccess = 0, hipErrorUnknown = 1, hipErrorInvalidHandle = 2 };
inline const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorInvalidHandle ? "invalid resource handle" : "unknown error";
}

struct ihipStream_t {
  std::function<void()> wait;  // until the stream's work is done
  hipError_t result = hipSuccess;  // of that work
  int device = 0;
};
using hipStream_t = ihipStream_t*;
struct ihipEvent_t {
  hipStream_t stream = nullptr;
  int device = 0;
};
using hipEvent_t = ihipEvent_t*;
using hipDevice_t = int;
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocPortable = 1;

inline thread_local int current_device = 0;  // a new thread has device 0
inline hipError_t hipGetDevice(int* d) {
  *d = current_device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  current_device = d;
  return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  *d = s->device;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  if (s->wait) s->wait();
  return s->result;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new ihipEvent_t;
  (*e)->device = current_device;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != s->device) return hipErrorInvalidHandle;
  e->stream = s;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) { return hipStreamSynchronize(e->stream); }
inline std::atomic<int64_t>& pinned_bytes() {
  static std::atomic<int64_t> b{0};
  return b;
}
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  auto* m = static_cast<size_t*>(std::malloc(bytes + 64));
  *m = bytes;
  pinned_bytes() += int64_t(bytes);
  *p = reinterpret_cast<char*>(m) + 64;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  auto* m = reinterpret_cast<size_t*>(static_cast<char*>(p) - 64);
  pinned_bytes() -= int64_t(*m);
  std::free(m);
  return hipSuccess;
}

// ---- device code

struct uint3 {
  unsigned x = 0, y = 0, z = 0;
};
struct int4 {
  int32_t x, y, z, w;
};
inline int4 make_int4(int32_t x, int32_t y, int32_t z, int32_t w) { return {x, y, z, w}; }
inline uint3 threadIdx, blockIdx, gridDim;

namespace block {
struct Fiber {
  ucontext_t ctx;
  std::vector<char> stack = std::vector<char>(128 << 10);
  bool done = false;
};
inline std::vector<Fiber> fibers;
inline ucontext_t scheduler;
inline unsigned current = 0;
inline void (*entry)() = nullptr;

inline void yield() { swapcontext(&fibers[current].ctx, &scheduler); }

// A meeting of `group` threads: the last one to arrive lets all go on.
struct Meeting {
  unsigned arrived = 0, generation = 0;
  void wait(unsigned group) {
    const unsigned g = generation;
    if (++arrived == group) {
      arrived = 0;
      ++generation;
    }
    while (generation == g) yield();
  }
};
inline Meeting whole, wave[16];
inline uint64_t lanes[16][64];

inline void run_fiber() {
  entry();
  fibers[current].done = true;
  yield();
}

// Runs one block of `threads` threads to its end.
inline void run(unsigned threads, void (*f)()) {
  entry = f;
  if (fibers.size() != threads) fibers = std::vector<Fiber>(threads);
  for (Fiber& x : fibers) {
    x.done = false;
    getcontext(&x.ctx);
    x.ctx.uc_stack.ss_sp = x.stack.data();
    x.ctx.uc_stack.ss_size = x.stack.size();
    x.ctx.uc_link = &scheduler;
    makecontext(&x.ctx, run_fiber, 0);
  }
  for (bool any = true; any;) {
    any = false;
    for (current = 0; current < threads; ++current) {
      if (fibers[current].done) continue;
      any = true;
      threadIdx.x = current;
      swapcontext(&scheduler, &fibers[current].ctx);
    }
  }
}

// Every lane's v, seen by all lanes of the wave.
template <typename T>
T exchange(T v, unsigned from) {
  const unsigned w = threadIdx.x / 64, l = threadIdx.x % 64;
  uint64_t bits = 0;
  std::memcpy(&bits, &v, sizeof(T));
  lanes[w][l] = bits;
  wave[w].wait(64);
  T r;
  std::memcpy(&r, &lanes[w][from], sizeof(T));
  wave[w].wait(64);
  return r;
}
}  // namespace block

inline void __syncthreads() { block::whole.wait(unsigned(block::fibers.size())); }
template <typename T>
T __shfl_up(T v, int o, int) {
  const int l = int(threadIdx.x % 64);
  return block::exchange(v, unsigned(l >= o ? l - o : l));
}
template <typename T>
T __shfl_xor(T v, int o, int) {
  return block::exchange(v, (threadIdx.x % 64) ^ unsigned(o));
}
inline unsigned long long __ballot(bool p) {
  const unsigned w = threadIdx.x / 64;
  block::lanes[w][threadIdx.x % 64] = p;
  block::wave[w].wait(64);
  unsigned long long r = 0;
  for (unsigned l = 0; l < 64; ++l) r |= (unsigned long long)(block::lanes[w][l]) << l;
  block::wave[w].wait(64);
  return r;
}
inline bool __any(bool p) { return __ballot(p) != 0; }

template <typename T>
T atomicAdd(T* p, T v) {
  const T old = *p;
  *p = old + v;
  return old;
}
template <typename T>
T atomicMax(T* p, T v) {
  const T old = *p;
  *p = v > old ? v : old;
  return old;
}
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))
#define __hip_atomic_load(p, order, scope) (*(p))
// A thread that sleeps waits for another block: none runs beside this one.
#define __builtin_amdgcn_s_sleep(n)                                                            \
  do {                                                                                         \
    std::printf("block %u waits for a tile that no running block has\n", blockIdx.x);          \
    std::fflush(stdout);                                                                       \
    std::_Exit(3);                                                                             \
  } while (0)
inline long long __double_as_longlong(double v) {
  long long r;
  std::memcpy(&r, &v, 8);
  return r;
}
inline double __longlong_as_double(long long v) {
  double r;
  std::memcpy(&r, &v, 8);
  return r;
}
