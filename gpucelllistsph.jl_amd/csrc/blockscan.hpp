// Scans: within a wave, within a block of 256 threads, and device-wide in one
// launch (used by the cell list, the pair list and the SPH step's rebuild).
#pragma once

#include "gclsph_internal.hpp"

namespace gclsph {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kTile = kScanThreads * kScanItems;  // 4096

constexpr int64_t scan_tiles(int64_t n) { return (n + kTile - 1) / kTile; }
// Words of the scratch array of a device-wide scan: a ticket counter, then one
// status word per tile.
constexpr int64_t scan_words(int64_t n) { return 1 + scan_tiles(n); }

template <typename T>
__device__ inline T wave_inclusive_scan(T v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    T t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// Exclusive block scan over kScanThreads values; returns the thread's exclusive
// prefix and writes the block total to *total.
template <typename T>
__device__ inline T block_exclusive_scan(T v, T* total) {
  __shared__ T wsum[kScanThreads / 64];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  T inc = wave_inclusive_scan(v, lane);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  T pre = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kScanThreads / 64; ++k) {
    if (k < w) pre += wsum[k];
    tot += wsum[k];
  }
  __syncthreads();
  *total = tot;
  return pre + inc - v;
}

// Clears the scratch words of the scan of n items; called by every thread (of
// `threads` in all, this one the i-th) of a kernel before the scan's.
__device__ __forceinline__ void clear_scan_words(uint64_t* words, int64_t n, int64_t i, int64_t threads) {
  for (; i < scan_words(n); i += threads) words[i] = 0;
}

// Exclusive scan of in[0..n) into out[0..n], out[n] = total, by scan_tiles(n)
// blocks of kScanThreads threads in one launch (decoupled look-back).  A block
// takes its tile from a ticket counter, publishes the tile's sum, adds up the
// sums before it, and publishes its prefix; it waits only for tiles of earlier
// tickets, whose blocks run and publish their sums before they wait, so every
// wait ends whatever the order and number of blocks the chip holds.  A status
// word holds its state and its value, so one atomic store publishes both.
// max_out (nullable): atomic maximum of the items.  Clear: the items are zero
// afterwards.  in and out are 16-byte aligned.
//
// One launch instead of three (tile sums, their scan, the tiles again): each
// launch of a step costs 4.4 us however small, and the items are read once.
template <bool Clear, typename O>
__device__ __forceinline__ void scan_tile(int32_t* __restrict__ in, O* __restrict__ out, int64_t n,
                                          uint64_t* __restrict__ words, int32_t* max_out) {
  constexpr uint64_t kSum = uint64_t(1) << 62, kPrefix = uint64_t(2) << 62, kValue = kSum - 1;
  __shared__ uint64_t ticket, before;
  __shared__ int32_t wmax[kScanThreads / 64];
  if (threadIdx.x == 0) ticket = atomicAdd(reinterpret_cast<unsigned long long*>(words), 1ull);
  __syncthreads();
  const int64_t tile = int64_t(ticket);
  const int64_t base = tile * kTile + int64_t(threadIdx.x) * kScanItems;
  const bool whole = base + kScanItems <= n;  // the last tile's tail goes item by item
  int32_t v[kScanItems];
  if (whole) {
    int4* p = reinterpret_cast<int4*>(in + base);
#pragma unroll
    for (int k = 0; k < kScanItems / 4; ++k) {
      const int4 w = p[k];
      v[4 * k] = w.x, v[4 * k + 1] = w.y, v[4 * k + 2] = w.z, v[4 * k + 3] = w.w;
    }
    if constexpr (Clear) {
#pragma unroll
      for (int k = 0; k < kScanItems / 4; ++k) p[k] = make_int4(0, 0, 0, 0);
    }
  } else {
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      v[k] = base + k < n ? in[base + k] : 0;
      if (Clear && base + k < n) in[base + k] = 0;
    }
  }
  O s = 0;
  int32_t mx = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    s += v[k];
    mx = v[k] > mx ? v[k] : mx;
  }
  if (max_out) {
    for (int o = 32; o > 0; o >>= 1) {
      const int32_t t = __shfl_xor(mx, o, 64);
      mx = t > mx ? t : mx;
    }
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
  }
  O total;
  const O mine = block_exclusive_scan<O>(s, &total);
  uint64_t* status = words + 1;
  if (threadIdx.x < 64) {
    const int lane = int(threadIdx.x);
    if (lane == 0) {
      __hip_atomic_store(status + tile, (tile == 0 ? kPrefix : kSum) | uint64_t(total), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      if (max_out) {
        for (int k = 1; k < kScanThreads / 64; ++k) mx = wmax[k] > mx ? wmax[k] : mx;
        if (mx > 0) atomicMax(max_out, mx);
      }
    }
    uint64_t pre = 0;
    for (int64_t j = tile - 1; j >= 0; j -= 64) {  // 64 tiles at a time, nearest first
      const int64_t i = j - lane;
      uint64_t w;
      for (;;) {
        w = i >= 0 ? __hip_atomic_load(status + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : kPrefix;
        if (!__any((w >> 62) == 0)) break;
        __builtin_amdgcn_s_sleep(1);
      }
      const uint64_t full = __ballot((w >> 62) == 2);
      const int last = full ? __builtin_ctzll(full) : 63;  // the nearest tile with its prefix ends the walk
      uint64_t add = lane <= last ? w & kValue : 0;
      for (int o = 32; o > 0; o >>= 1) add += __shfl_xor(add, o, 64);
      pre += add;
      if (full) break;
    }
    if (lane == 0) {
      if (tile > 0)
        __hip_atomic_store(status + tile, kPrefix | (pre + uint64_t(total)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      before = pre;
    }
  }
  __syncthreads();
  O pre = O(before) + mine;
  if (whole) {
    O o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      o[k] = pre;
      pre += v[k];
    }
    int4* p = reinterpret_cast<int4*>(out + base);
#pragma unroll
    for (int k = 0; k < int(kScanItems * sizeof(O) / 16); ++k) {
      int4 w;
      __builtin_memcpy(&w, reinterpret_cast<const char*>(o) + 16 * k, 16);
      p[k] = w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      if (base + k < n) out[base + k] = pre;
      pre += v[k];
    }
  }
  if (tile == scan_tiles(n) - 1 && threadIdx.x == 0) out[n] = O(before) + total;
}

}  // namespace gclsph
