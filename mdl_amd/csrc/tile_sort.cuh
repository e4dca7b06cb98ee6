// Stable sort of (key, payload) pairs in one or two launches, for the sizes
// where the radix sort's three launches per 8-bit pass cost more than their
// work (a launch takes about 3 us of the stream whatever it does).
//
//   tile_sort   - a block sorts a tile of kMergeTile entries in LDS, on the
//                 bits the tile's own key range needs, and notes its range.
//   rank_merge  - a block places one sorted tile: an entry's position is its
//                 rank in its own tile plus, for every other tile, how many
//                 of that tile's keys go before it.  A tile whose range lies
//                 wholly before or after adds its size or nothing; only
//                 tiles whose ranges overlap are loaded and searched.
//
// The keys of a grouped lookup come feature by feature, so with one table
// per feature a tile overlaps the few tiles of its own table only.  In any
// other order the result is the same and the merge searches every tile.
//
// Keys at or past the last table's rows (the sentinel of ids without a
// gradient) are placed after all others, in input order, as the tables' end.
#pragma once

#include "common.cuh"

namespace mdl {

// A tile is as large as 32 KB of LDS and two blocks per CU allow: smaller
// tiles sort a little sooner and overlap more tiles in the merge (2048: 37 us
// instead of 33 for 32 tables of 12 K entries); sixteen waves of four entries
// a thread, or 8-bit digits, took 1 us longer per call.
constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / kWave;
constexpr int kTileItems = 8;
constexpr int kMergeTile = kTileThreads * kTileItems;
constexpr int kTileBits = 7;  // digit width in LDS at most
constexpr int kTileRadix = 1 << kTileBits;
constexpr int kDigitWaves = kTileRadix / kWave;
// Tiles of one sort at most (the merge's list of overlapping tiles).
constexpr int64_t kMaxMergeTiles = 1024;

static inline int64_t merge_tiles(int64_t n) { return (n + kMergeTile - 1) / kMergeTile; }

struct TileSortArgs {
  const mdl_table* tables;  // ordered by row_base; the last one's end bounds the live keys
  int32_t T;
  const uint32_t* keys_in;
  const uint32_t* vals_in;
  uint32_t* keys_out;
  uint32_t* vals_out;
  int64_t n_cap;
  const int64_t* n_dev;
  uint32_t* tile_min;   // [tiles] smallest live key
  uint32_t* tile_max;   // [tiles] largest live key
  uint32_t* tile_live;  // [tiles] live keys
};

// Entries present: n_cap, or the device count clamped to [0, n_cap].
__device__ __forceinline__ int64_t entries_present(int64_t n_cap, const int64_t* n_dev) {
  if (n_dev == nullptr) return n_cap;
  const int64_t n = *n_dev;
  return n < 0 ? 0 : (n > n_cap ? n_cap : n);
}

// First key no table covers (every key below it belongs to a row).
__device__ __forceinline__ uint64_t live_end(const mdl_table* tables, int32_t T) {
  return (uint64_t)tables[T - 1].row_base + (uint64_t)tables[T - 1].num_rows;
}

struct TileStage {
  uint32_t key[kMergeTile];
  uint32_t val[kMergeTile];
  uint32_t wave_hist[kTileWaves][kTileRadix];
  uint32_t digit_base[kTileRadix];   // entries of smaller digits among its wave's digits
  uint32_t digit_total[kDigitWaves];  // entries of each 64 digits
  uint32_t red[3 * kTileWaves];
};

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
  for (int m = 1; m < kWave; m <<= 1) {
    const uint32_t o = shfl_u(v, lane_id() ^ m);
    v = o < v ? o : v;
  }
  return v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  for (int m = 1; m < kWave; m <<= 1) {
    const uint32_t o = shfl_u(v, lane_id() ^ m);
    v = o > v ? o : v;
  }
  return v;
}

// Sorts entries [tile * kMergeTile, +kMergeTile) of the array.  On return
// st.key holds the tile's live keys in order, as offsets from *key_min
// (dead ones after them), and the sorted pairs have been written out.
// Entry i of wave w, item q, lane l is w * 64 * kItems + q * 64 + l: visited
// in that order, so equal digits keep it (stable).  (kItems is a constant: with
// a tile's own count the loops of a full tile took a fifth longer.)
template <int kItems>
__device__ __forceinline__ void sort_tile(const TileSortArgs& a, int64_t tile, int64_t n, TileStage& st,
                                          uint32_t* live_out, uint32_t* key_min) {
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  const int64_t base = tile * kMergeTile;
  const int m = n - base < kMergeTile ? (int)(n - base) : kMergeTile;
  const uint64_t end = live_end(a.tables, a.T);
  uint32_t k[kItems], v[kItems];
  bool live[kItems];
#pragma unroll
  for (int q = 0; q < kItems; ++q) {
    const int i = w * (kWave * kItems) + q * kWave + lane;
    const int64_t at = base + (i < m ? i : m - 1);
    k[q] = a.keys_in[at];
    v[q] = a.vals_in[at];
  }
  uint32_t lo = 0xffffffffu, hi = 0u, cnt = 0u;
#pragma unroll
  for (int q = 0; q < kItems; ++q) {
    const int i = w * (kWave * kItems) + q * kWave + lane;
    live[q] = i < m && (uint64_t)k[q] < end;
    lo = live[q] && k[q] < lo ? k[q] : lo;
    hi = live[q] && k[q] > hi ? k[q] : hi;
    cnt += (uint32_t)__popcll(__ballot(live[q]));
  }
  lo = wave_min_u32(lo);
  hi = wave_max_u32(hi);
  if (lane == 0) {
    st.red[w] = lo;
    st.red[kTileWaves + w] = hi;
    st.red[2 * kTileWaves + w] = cnt;
  }
  __syncthreads();
  uint32_t tmin = 0xffffffffu, tmax = 0u, tlive = 0u;
#pragma unroll
  for (int q = 0; q < kTileWaves; ++q) {
    tmin = st.red[q] < tmin ? st.red[q] : tmin;
    tmax = st.red[kTileWaves + q] > tmax ? st.red[kTileWaves + q] : tmax;
    tlive += st.red[2 * kTileWaves + q];
  }
  if (tlive == 0) tmin = tmax = 0u;
  // Live keys become offsets from the smallest; dead ones (and the slots
  // past the array) the offset after the largest.  Keys below 2^32 - 1
  // (the tables' rows) leave room for it.
  const uint32_t dead = tmax - tmin + 1u;
  const uint32_t range = (int)tlive == kItems * kTileThreads ? tmax - tmin : (tlive == 0 ? 0u : dead);
#pragma unroll
  for (int q = 0; q < kItems; ++q)
    k[q] = live[q] ? k[q] - tmin : (tlive == 0 ? 0u : dead);
  const int bits = range == 0 ? 0 : 32 - __builtin_clz(range);
  const int passes = (bits + kTileBits - 1) / kTileBits;
  const int per = passes ? (bits + passes - 1) / passes : 0;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
  for (int p = 0; p < passes; ++p) {
    const int shift = p * per;
    const uint32_t mask = (1u << per) - 1u;
    for (int i = tid; i < kTileWaves * kTileRadix; i += kTileThreads) (&st.wave_hist[0][0])[i] = 0u;
    __syncthreads();
    uint32_t rank[kItems];
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
      const uint32_t d = (k[q] >> shift) & mask;
      // lanes that differ from this one in any digit bit (bitop3 0xF6:
      // x | (ballot ^ t), t all ones where the lane's bit is set)
      uint32_t xlo = 0u, xhi = 0u;
#pragma unroll
      for (int b = 0; b < kTileBits; ++b) {
        const uint32_t t = (uint32_t)((int32_t)(d << (31 - b)) >> 31);
        const uint64_t bb = __ballot(t != 0u);
        xlo = __builtin_amdgcn_bitop3_b32(xlo, (uint32_t)bb, t, 0xF6);
        xhi = __builtin_amdgcn_bitop3_b32(xhi, (uint32_t)(bb >> 32), t, 0xF6);
      }
      const uint64_t same = ~(((uint64_t)xhi << 32) | xlo);
      const uint32_t r = (uint32_t)__popcll(same & lt_mask);
      const uint32_t old = st.wave_hist[w][d];
      __builtin_amdgcn_wave_barrier();
      if (r == 0) st.wave_hist[w][d] = old + (uint32_t)__popcll(same);
      __builtin_amdgcn_wave_barrier();
      rank[q] = old + r;
    }
    __syncthreads();
    if (tid < kTileRadix) {
      // thread d: digit d's counts before each wave, then before each digit
      // of its 64
      uint32_t run = 0u;
#pragma unroll
      for (int q = 0; q < kTileWaves; ++q) {
        const uint32_t c = st.wave_hist[q][tid];
        st.wave_hist[q][tid] = run;
        run += c;
      }
      uint32_t x = run;
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t o = shfl_u(x, lane >= d ? lane - d : lane);
        if (lane >= d) x += o;
      }
      st.digit_base[tid] = x - run;
      if (lane == kWave - 1) st.digit_total[w] = x;
    }
    __syncthreads();
    uint32_t group_base[kDigitWaves];
    group_base[0] = 0u;
#pragma unroll
    for (int g = 1; g < kDigitWaves; ++g) group_base[g] = group_base[g - 1] + st.digit_total[g - 1];
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
      const uint32_t d = (k[q] >> shift) & mask;
      uint32_t pos = st.digit_base[d] + st.wave_hist[w][d] + rank[q];
#pragma unroll
      for (int g = 1; g < kDigitWaves; ++g) pos += (int)(d / kWave) == g ? group_base[g] : 0u;
      st.key[pos] = k[q];
      st.val[pos] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
      const int i = w * (kWave * kItems) + q * kWave + lane;
      k[q] = st.key[i];
      v[q] = st.val[i];
    }
  }
  if (passes == 0) {
    // one key value (or none live): the input order stands
#pragma unroll
    for (int q = 0; q < kItems; ++q)
      st.key[w * (kWave * kItems) + q * kWave + lane] = k[q];
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < kItems; ++q) {
    const int i = w * (kWave * kItems) + q * kWave + lane;
    if (i < m) {
      a.keys_out[base + i] = i < (int)tlive ? k[q] + tmin : (uint32_t)end;
      a.vals_out[base + i] = v[q];
    }
  }
  if (a.tile_min != nullptr && tid == 0) {
    a.tile_min[tile] = tmin;
    a.tile_max[tile] = tmax;
    a.tile_live[tile] = tlive;
  }
  *live_out = tlive;
  *key_min = tmin;
}

static __global__ __launch_bounds__(kTileThreads) void tile_sort_kernel(TileSortArgs a) {
  __shared__ TileStage st;
  const int64_t n = entries_present(a.n_cap, a.n_dev);
  if ((int64_t)blockIdx.x * kMergeTile >= n) return;
  uint32_t live, key_min;
  sort_tile<kTileItems>(a, blockIdx.x, n, st, &live, &key_min);
}

// Entries of sorted s[lo, hi) that go before x: those below it, and with
// `ties` also those equal to it; returns lo + their number.
__device__ __forceinline__ int count_before(const uint32_t* s, int lo, int hi, uint32_t x, bool ties) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    const uint32_t y = s[mid];
    if (y < x || (ties && y == x)) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// A block ranks kMergePart entries of one sorted tile, two a thread, against
// two overlapping tiles at a time: a search is a chain of 13 LDS round trips,
// so four of them go side by side in each thread.  (Four tiles at a time need
// 125 VGPRs and 66 KB of LDS: steps of 32 and 64 tables 131 -> 135 and 166 ->
// 171 us; parts of 512 entries change neither.)
constexpr int kMergeThreads = 512;
constexpr int kMergeWaves = kMergeThreads / kWave;
constexpr int kMergePart = 2 * kMergeThreads;
constexpr int kMergeParts = kMergeTile / kMergePart;
constexpr int kMergeLoads = kMergeTile / kMergeThreads;

static __global__ __launch_bounds__(kMergeThreads) void rank_merge_kernel(TileSortArgs a) {
  __shared__ uint32_t s_oth[2][kMergeTile];
  __shared__ uint16_t s_list[kMaxMergeTiles];
  __shared__ uint32_t s_red[3 * kMergeWaves];
  __shared__ uint32_t s_range[2];
  __shared__ int s_count;
  const int64_t n = entries_present(a.n_cap, a.n_dev);
  const int tiles = (int)((n + kMergeTile - 1) / kMergeTile);
  const int tile = (int)blockIdx.x / kMergeParts;
  const int part = ((int)blockIdx.x % kMergeParts) * kMergePart;  // the part's first entry in its tile
  if (tile >= tiles) return;
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  const int64_t base = (int64_t)tile * kMergeTile;
  const int m = n - base < kMergeTile ? (int)(n - base) : kMergeTile;
  if (part >= m) return;
  const int live = (int)a.tile_live[tile];
  const int part_live = live - part < kMergePart ? live - part : kMergePart;  // may be <= 0
  uint32_t x[2], v[2], rank[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = part + q * kMergeThreads + tid;
    const int64_t at = base + (i < m ? i : m - 1);
    x[q] = a.keys_in[at];
    v[q] = a.vals_in[at];
    if (i == part) s_range[0] = x[q];
    if (i == part + part_live - 1) s_range[1] = x[q];
  }
  if (tid == 0) s_count = 0;
  __syncthreads();
  const uint32_t kmin = s_range[0], kmax = s_range[1];
  uint32_t before = 0u, dead_before = 0u, all_live = 0u;
  for (int j = tid; j < tiles; j += kMergeThreads) {
    const uint32_t lj = a.tile_live[j];
    const int64_t left = n - (int64_t)j * kMergeTile;
    all_live += lj;
    if (j < tile) dead_before += (uint32_t)(left < kMergeTile ? left : kMergeTile) - lj;
    if (j == tile || lj == 0 || part_live <= 0) continue;
    const uint32_t jmin = a.tile_min[j], jmax = a.tile_max[j];
    if (j < tile ? jmax <= kmin : jmax < kmin) before += lj;
    else if (j < tile ? jmin <= kmax : jmin < kmax) s_list[atomicAdd(&s_count, 1)] = (uint16_t)j;
  }
  for (int d = 1; d < kWave; d <<= 1) {
    before += shfl_u(before, lane ^ d);
    dead_before += shfl_u(dead_before, lane ^ d);
    all_live += shfl_u(all_live, lane ^ d);
  }
  if (lane == 0) {
    s_red[w] = before;
    s_red[kMergeWaves + w] = dead_before;
    s_red[2 * kMergeWaves + w] = all_live;
  }
  __syncthreads();
  before = dead_before = all_live = 0u;
#pragma unroll
  for (int q = 0; q < kMergeWaves; ++q) {
    before += s_red[q];
    dead_before += s_red[kMergeWaves + q];
    all_live += s_red[2 * kMergeWaves + q];
  }
  const int others = s_count;
#pragma unroll
  for (int q = 0; q < 2; ++q) rank[q] = before + (uint32_t)(part + q * kMergeThreads + tid);
  // The next two tiles' keys are on their way while two are searched.
  uint32_t next[2][kMergeLoads], next_ties[2];
  auto fetch = [&](int at) {
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const bool there = at + o < others;
      const int j = s_list[there ? at + o : at];
      const int live_j = there ? (int)a.tile_live[j] : 0;
      next_ties[o] = j < tile ? 1u : 0u;
#pragma unroll
      for (int q = 0; q < kMergeLoads; ++q) {
        // past the tile's live keys: a key that goes before none
        const int i = q * kMergeThreads + tid;
        next[o][q] = i < live_j ? a.keys_in[(int64_t)j * kMergeTile + i] : 0xffffffffu;
      }
    }
  };
  if (others > 0) fetch(0);
  for (int o = 0; o < others; o += 2) {
    // Keys below `bound` go before the entry: equal keys of an earlier tile
    // do, those of a later one do not (live keys lie below 2^32 - 1).
    uint32_t bound[2][2];
    __syncthreads();  // the previous searches are done
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int q = 0; q < 2; ++q) bound[t][q] = x[q] + next_ties[t];
#pragma unroll
      for (int q = 0; q < kMergeLoads; ++q) s_oth[t][q * kMergeThreads + tid] = next[t][q];
    }
    __syncthreads();
    if (o + 2 < others) fetch(o + 2);
    uint32_t at[2][2] = {{0u, 0u}, {0u, 0u}};
#pragma unroll
    for (uint32_t step = kMergeTile / 2; step >= 1; step >>= 1) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q) at[t][q] += s_oth[t][at[t][q] + step - 1] < bound[t][q] ? step : 0u;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 2; ++q) rank[q] += at[t][q] + (s_oth[t][at[t][q]] < bound[t][q] ? 1u : 0u);
  }
  const uint32_t dead_at = all_live + dead_before;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = part + q * kMergeThreads + tid;
    if (i < m) {
      const uint32_t to = i < live ? rank[q] : dead_at + (uint32_t)(i - live);
      a.keys_out[to] = x[q];
      a.vals_out[to] = v[q];
    }
  }
}

}  // namespace mdl
