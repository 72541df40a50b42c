// Scans: within a wave, within a block of 256 threads, and device-wide in one
// launch (used by the cell list, the pair list and the SPH step's rebuild).
#pragma once

#include <type_traits>

#include "gclsph_internal.hpp"

namespace gclsph {

constexpr int kScanThreads = 256;
constexpr int kScanRow = 4 * kScanThreads;  // items of one 16-byte load per thread

// A device-wide scan runs in tiles of 4, 8 or 16 rows, a block each: as many
// rows as keep it within kScanTiles blocks, fewest first: a block costs its turn
// at the tile counter (scan_tile below), a long tile its own time.  Limits of
// 256 / 512: 700,000 cells 9.1 / 9.0 us (4 rows both), 2.8 M cells 16.3 (16 rows) /
// 16.5 us (8), the cells of 64 problems, each with a counter, 10.1 (8) / 8.4 us (4).
constexpr int kScanTiles = 512;
constexpr int64_t scan_tiles(int64_t n, int rows) { return (n + rows * kScanRow - 1) / (rows * kScanRow); }
constexpr int scan_rows(int64_t n) {
  return scan_tiles(n, 4) <= kScanTiles ? 4 : (scan_tiles(n, 8) <= kScanTiles ? 8 : 16);
}
// Words of the scratch array of a device-wide scan: a ticket counter, then one
// status word per tile.
constexpr int64_t scan_words(int64_t n) { return 1 + scan_tiles(n, 4); }

template <typename T>
__device__ inline T wave_inclusive_scan(T v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    T t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// Clears the scratch words of the scan of n items; called by every thread (of
// `threads` in all, this one the i-th) of a kernel before the scan's.
__device__ __forceinline__ void clear_scan_words(uint64_t* words, int64_t n, int64_t i, int64_t threads) {
  for (; i < scan_words(n); i += threads) words[i] = 0;
}

// Exclusive scan of in[0..n) into out[0..n], out[n] = total, by
// scan_tiles(n, Rows) blocks of kScanThreads threads in one launch (decoupled
// look-back).  A block publishes its tile's sum, adds up the sums before it,
// 256 tiles at a time, and publishes its prefix.  A status word holds its state
// and its value, so one atomic store publishes both.  max_out (nullable): atomic
// maximum of the items.  Clear: the items are zero afterwards.  in and out are
// 16-byte aligned.
//
// A block waits only for tiles before its own, and takes its tile from a counter
// when it starts: those tiles are then with blocks that run already, whatever
// else the chip runs, so every wait ends.  (A block's place in the grid as its
// tile promises that only while all blocks of all scans in flight fit the chip:
// of 16 rows of 64-bit sums one block fits a CU, 256 the chip.)  A scan of one
// tile needs no counter.  Time with the counter / with places in the grid: 6,000
// and 60,000 cells 2.1 / 2.1 and 4.8 / 4.8 us, 700,000 9.0 / 8.5, 2.8 M 16.5 / 14.8.
//
// One launch instead of three (tile sums, their scan, the tiles again): each
// launch of a step costs 4.4 us however small, and the items are read once.
template <int Rows, bool Clear, typename O>
__device__ __forceinline__ void scan_tile(int32_t* __restrict__ in, O* __restrict__ out, int64_t n,
                                          uint64_t* __restrict__ words, int32_t* max_out) {
  constexpr uint64_t kSum = uint64_t(1) << 62, kPrefix = uint64_t(2) << 62, kValue = kSum - 1;
  constexpr int kWaves = kScanThreads / 64;
  __shared__ uint64_t ticket, wadd[kWaves];
  __shared__ O wsum[Rows][kWaves];
  __shared__ int32_t wmax[kWaves], wfull[kWaves];
  int64_t tile = 0;
  if (scan_tiles(n, Rows) > 1) {  // uniform
    if (threadIdx.x == 0) ticket = atomicAdd(reinterpret_cast<unsigned long long*>(words), 1ull);
    __syncthreads();
    tile = int64_t(ticket);
  }
  const int lane = int(threadIdx.x & 63), wave = int(threadIdx.x >> 6);
  const int64_t base = tile * (Rows * kScanRow) + 4 * int64_t(threadIdx.x);
  int32_t v[Rows][4];
#pragma unroll
  for (int r = 0; r < Rows; ++r) {
    const int64_t i = base + r * kScanRow;
    if (i + 4 <= n) {
      const int4 w = *reinterpret_cast<const int4*>(in + i);
      v[r][0] = w.x, v[r][1] = w.y, v[r][2] = w.z, v[r][3] = w.w;
      if (Clear) *reinterpret_cast<int4*>(in + i) = make_int4(0, 0, 0, 0);
    } else {  // the end of the last tile goes item by item
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[r][k] = i + k < n ? in[i + k] : 0;
        if (Clear && i + k < n) in[i + k] = 0;
      }
    }
  }
  int32_t mx = 0;
  O pre[Rows];  // the thread's prefix in its wave's part of each row
#pragma unroll
  for (int r = 0; r < Rows; ++r) {
    O s = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      s += v[r][k];
      mx = v[r][k] > mx ? v[r][k] : mx;
    }
    const O inc = wave_inclusive_scan<O>(s, lane);
    pre[r] = inc - s;
    if (lane == 63) wsum[r][wave] = inc;
  }
  if (max_out) {
    for (int o = 32; o > 0; o >>= 1) {
      const int32_t t = __shfl_xor(mx, o, 64);
      mx = t > mx ? t : mx;
    }
    if (lane == 0) wmax[wave] = mx;
  }
  __syncthreads();
  O total = 0;
#pragma unroll
  for (int r = 0; r < Rows; ++r) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w == wave) pre[r] += total;
      total += wsum[r][w];
    }
  }
  uint64_t* status = words + 1;
  if (threadIdx.x == 0) {
    __hip_atomic_store(status + tile, (tile == 0 ? kPrefix : kSum) | uint64_t(total), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    if (max_out) {
      for (int w = 1; w < kWaves; ++w) mx = wmax[w] > mx ? wmax[w] : mx;
      if (mx > 0) atomicMax(max_out, mx);
    }
  }
  uint64_t before = 0;
  for (int64_t j = tile - 1; j >= 0; j -= kScanThreads) {  // nearest first; uniform over the block
    const int64_t i = j - threadIdx.x;
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
    if (lane == 0) {
      wadd[wave] = add;
      wfull[wave] = full != 0;
    }
    __syncthreads();
    bool found = false;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
      before += found ? 0 : wadd[k];
      found |= wfull[k] != 0;
    }
    __syncthreads();
    if (found) break;
  }
  if (threadIdx.x == 0 && tile > 0)
    __hip_atomic_store(status + tile, kPrefix | (before + uint64_t(total)), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int r = 0; r < Rows; ++r) {
    const int64_t i = base + r * kScanRow;
    O o[4];
    o[0] = O(before) + pre[r];
#pragma unroll
    for (int k = 1; k < 4; ++k) o[k] = o[k - 1] + v[r][k - 1];
    if (i + 4 <= n) {
      int4* p = reinterpret_cast<int4*>(out + i);
#pragma unroll
      for (int k = 0; k < int(4 * sizeof(O) / 16); ++k) {
        int4 w;
        __builtin_memcpy(&w, reinterpret_cast<const char*>(o) + 16 * k, 16);
        p[k] = w;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (i + k < n) out[i + k] = o[k];
    }
  }
  if (threadIdx.x == 0 && tile == scan_tiles(n, Rows) - 1) out[n] = O(before) + total;
}

// Calls f with the rows per tile as a constant.
template <typename F>
inline void with_scan_rows(int rows, F&& f) {
  if (rows == 4) f(std::integral_constant<int, 4>());
  else if (rows == 8) f(std::integral_constant<int, 8>());
  else f(std::integral_constant<int, 16>());
}

}  // namespace gclsph
