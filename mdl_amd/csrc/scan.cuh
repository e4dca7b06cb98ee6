// Scan of int64 counts by a block, for offsets and chunk bases.
#pragma once

#include "common.cuh"

namespace mdl {

constexpr int kScanItems = 8;  // values of a tile per thread

__device__ __forceinline__ int64_t shfl_i64(int64_t v, int src) {
  const uint32_t lo = (uint32_t)shfl_i((int)(uint32_t)v, src), hi = (uint32_t)shfl_i((int)(v >> 32), src);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Exclusive scan of one value per thread over a block of kThreads: shuffles
// inside each wave, one barrier for the wave totals (256 threads through LDS
// alone took 16 barriers and half the scan's time).  smem holds a word per
// wave.
template <int kThreads>
__device__ __forceinline__ int64_t block_exclusive_scan(int64_t v, int64_t* smem, int64_t* total) {
  constexpr int kWaves = kThreads / kWave;
  const int lane = lane_id(), w = threadIdx.x / kWave;
  int64_t x = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int64_t o = shfl_i64(x, lane >= d ? lane - d : lane);
    if (lane >= d) x += o;
  }
  if (lane == kWave - 1) smem[w] = x;
  __syncthreads();
  int64_t before = 0, all = 0;
#pragma unroll
  for (int q = 0; q < kWaves; ++q) {
    before += q < w ? smem[q] : 0;
    all += smem[q];
  }
  if (total) *total = all;
  __syncthreads();
  return before + x - v;
}

// LDS of a scanned tile: a word per wave, and every wave's 64 x kScanItems
// values with a pad word after each lane's.
template <int kThreads>
struct ScanStage {
  int64_t wave[kThreads / kWave];
  int64_t v[kThreads / kWave][kWave * (kScanItems + 1)];
};

// The values of a tile of kThreads * kScanItems from base, 64 neighbouring
// ones a load: value k of a thread is its wave's k * 64 + lane.
template <int kThreads>
__device__ __forceinline__ void load_scan_tile(const int64_t* __restrict__ in, int64_t n, int64_t base,
                                               int64_t (&v)[kScanItems]) {
  const int64_t first = base + (int64_t)(threadIdx.x / kWave) * (kWave * kScanItems) + lane_id();
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) v[k] = first + k * kWave < n ? in[first + k * kWave] : 0;
}

// offsets[i + 1] = prefix + sum(in[0 .. i]) over the tile v that
// load_scan_tile read from base; returns the tile's sum.  The wave's values
// change places in LDS so that each lane adds up consecutive ones, and back
// for the stores.  (A lane that loads and stores its eight consecutive values
// itself touches 64 lines an instruction: one block took 7.7 us for 8192
// values just written and 14.7 for 16384; so it takes 4.4 and 7.4.)
template <int kThreads>
__device__ __forceinline__ int64_t scan_tile(int64_t (&v)[kScanItems], int64_t n, int64_t base, int64_t prefix,
                                             ScanStage<kThreads>& st, int64_t* __restrict__ offsets) {
  const int lane = lane_id(), w = threadIdx.x / kWave;
  const int64_t first = base + (int64_t)w * (kWave * kScanItems) + lane;
  int64_t* stage = st.v[w];
  auto place = [](int i) { return i + i / kScanItems; };
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) stage[place(k * kWave + lane)] = v[k];
  wave_sync();
  int64_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = stage[place(lane * kScanItems) + k];
    s += v[k];
  }
  int64_t all;
  int64_t ex = block_exclusive_scan<kThreads>(s, st.wave, &all) + prefix;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    ex += v[k];
    stage[place(lane * kScanItems) + k] = ex;
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < kScanItems; ++k)
    if (first + k * kWave < n) offsets[first + k * kWave + 1] = stage[place(k * kWave + lane)];
  wave_sync();  // the next tile restages the values
  return all;
}

// offsets[0 .. n] of n values by one block, the next tile's values on their
// way while one is scanned.  Up to two values a thread are neighbours in
// memory as they are and skip the change of places (512 values 3.8 -> 2.5 us).
template <int kThreads>
__device__ __forceinline__ void scan_in_block(const int64_t* __restrict__ in, int64_t n, ScanStage<kThreads>& st,
                                              int64_t* __restrict__ offsets) {
  constexpr int64_t kTile = (int64_t)kThreads * kScanItems;
  if (threadIdx.x == 0) offsets[0] = 0;
  if (n <= 2 * kThreads) {
    const int64_t i = 2 * (int64_t)threadIdx.x;
    const int64_t a = i < n ? in[i] : 0, b = i + 1 < n ? in[i + 1] : 0;
    const int64_t before = block_exclusive_scan<kThreads>(a + b, st.wave, nullptr);
    if (i < n) offsets[i + 1] = before + a;
    if (i + 1 < n) offsets[i + 2] = before + a + b;
    return;
  }
  int64_t next[kScanItems], carry = 0;
  load_scan_tile<kThreads>(in, n, 0, next);
  for (int64_t base = 0; base < n; base += kTile) {
    int64_t v[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) v[k] = next[k];
    if (base + kTile < n) load_scan_tile<kThreads>(in, n, base + kTile, next);
    carry += scan_tile<kThreads>(v, n, base, carry, st, offsets);
  }
}

}  // namespace mdl
