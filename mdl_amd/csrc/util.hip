// Error state, bucketing and the lengths -> offsets scan.
#include "common.cuh"
#include "scan.cuh"

#include <cstdio>

namespace mdl {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int code, const std::string& msg) {
  set_error(msg);
  return code;
}

int check_hip(hipError_t err, const char* what) {
  if (err == hipSuccess) return MDL_OK;
  return fail(MDL_ERR_HIP, std::string(what) + ": " + hipGetErrorString(err));
}

// ------------------------------------------------------------ bucketing --

// Bucket of one raw value (0 for a null).  mod_magic = ceil(2^64 / m) for
// the mod rule's m = num_buckets - 1 >= 2.
__device__ __forceinline__ int64_t bucket_of(int64_t v, bool present, int64_t num_buckets, int32_t mode,
                                             int32_t validate_nonzero, uint64_t mod_magic, int& bad) {
  if (!present) return 0;
  if (mode == MDL_BUCKET_NONE) return v;
  if (mode == MDL_BUCKET_PRE_HASHED) {
    // Unsigned low bits of the signed hash: identical to the signed modulo
    // for a power-of-two bucket count, INT64_MIN included.
    bad += (validate_nonzero && v == 0);
    return (int64_t)(((uint64_t)v & (uint64_t)(num_buckets - 1)) + 1u);
  }
  // 1 + floormod(v - 1, m) without forming v - 1 or dividing: the sign goes
  // first (x = v or ~v = -v - 1, both below 2^63, INT64_MIN included), and
  // mulhi(x, ceil(2^64 / m)) is floor(x / m) or one more, which one add of m
  // corrects.
  const uint64_t m = (uint64_t)(num_buckets - 1);
  uint64_t fm1 = 0;  // floormod(v - 1, m)
  if (m > 1) {
    const bool neg = v < 0;
    const uint64_t x = neg ? ~(uint64_t)v : (uint64_t)v;
    uint64_t rem = x - __umul64hi(x, mod_magic) * m;
    if ((int64_t)rem < 0) rem += m;
    const uint64_t fm = neg ? m - 1 - rem : rem;  // floormod(v, m)
    fm1 = fm == 0 ? m - 1 : fm - 1;
  }
  return (int64_t)(1 + fm1);
}

__global__ void bucketize_kernel(const int64_t* __restrict__ raw, const uint8_t* __restrict__ valid,
                                 int64_t n, int64_t num_buckets, int32_t mode,
                                 int32_t validate_nonzero, int64_t* __restrict__ out,
                                 int32_t* __restrict__ error_count, uint64_t mod_magic) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  int bad = 0;
  for (; i < n; i += stride) {
    const bool present = valid == nullptr || valid[i] != 0;
    out[i] = bucket_of(raw[i], present, num_buckets, mode, validate_nonzero, mod_magic, bad);
  }
  if (error_count != nullptr && bad) atomicAdd(error_count, bad);
}

static uint64_t mod_magic_for(int32_t mode, int64_t num_buckets) {
  const uint64_t m = (uint64_t)(num_buckets - 1);
  return mode == MDL_BUCKET_MOD && m > 1 ? UINT64_MAX / m + 1 : 0;  // ceil(2^64 / m)
}

static int validate_bucket_mode(const char* who, int32_t mode, int64_t num_buckets) {
  if (mode == MDL_BUCKET_PRE_HASHED) {
    if (num_buckets <= 0 || (num_buckets & (num_buckets - 1)) != 0)
      return fail(MDL_ERR_INVALID, "pre_hashed num_buckets must be a positive power of two");
  } else if (mode == MDL_BUCKET_MOD) {
    if (num_buckets <= 1) return fail(MDL_ERR_INVALID, "mod bucketing needs num_buckets > 1");
  } else {
    return fail(MDL_ERR_INVALID, std::string(who) + ": unknown bucketing mode");
  }
  return MDL_OK;
}

// ----------------------------------------------------------------- scan --

constexpr int kScanThreads = 256;
constexpr int kScanTile = kScanThreads * kScanItems;
// A scan of up to kScanOneBlock lengths is one block's, in one launch: for
// 16384 lengths 7.4 us when they were just written and 8.5 from HBM, for 24576
// 10.7 and 12.0; the tile sums and the scan of the tiles take 9.3 us with the
// gap between them for either.
constexpr int kScanOneThreads = 1024;
constexpr int64_t kScanOneBlock = 2 * kScanOneThreads * kScanItems;

// Sum over a block of kScanThreads, valid in its first thread.
__device__ __forceinline__ int64_t block_sum_i64(int64_t v, int64_t* smem) {
  for (int m = 1; m < kWave; m <<= 1) v += shfl_i64(v, lane_id() ^ m);
  if (lane_id() == 0) smem[threadIdx.x / kWave] = v;
  __syncthreads();
  int64_t t = 0;
#pragma unroll
  for (int q = 0; q < kScanThreads / kWave; ++q) t += smem[q];
  return t;
}

__global__ __launch_bounds__(kScanOneThreads) void scan_one_block(const int64_t* __restrict__ in, int64_t n,
                                                                  int64_t* __restrict__ offsets) {
  __shared__ ScanStage<kScanOneThreads> st;
  scan_in_block<kScanOneThreads>(in, n, st, offsets);
}

__global__ __launch_bounds__(kScanThreads) void scan_tile_sums(const int64_t* __restrict__ in, int64_t n,
                                                               int64_t* __restrict__ sums) {
  __shared__ int64_t smem[kScanThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int64_t v[kScanItems];
  int64_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + (int64_t)k * kScanThreads + threadIdx.x;
    v[k] = i < n ? in[i] : 0;
  }
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) s += v[k];
  const int64_t t = block_sum_i64(s, smem);
  if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

// Exclusive scan of the per-tile sums in place, one block, any count.
__global__ __launch_bounds__(kScanThreads) void scan_sums_single(int64_t* __restrict__ sums, int64_t m) {
  __shared__ int64_t smem[kScanThreads / kWave];
  int64_t carry = 0;
  for (int64_t base = 0; base < m; base += kScanThreads) {
    int64_t i = base + threadIdx.x;
    int64_t v = i < m ? sums[i] : 0;
    int64_t total;
    int64_t ex = block_exclusive_scan<kScanThreads>(v, smem, &total);
    if (i < m) sums[i] = carry + ex;
    carry += total;
  }
}

// offsets[i+1] = sum(in[0..i]); offsets[0] = 0.  The tile's prefix is
// sums[b] after scan_sums_single, or, with prefix_self (few tiles), the sum
// of the raw tile sums before it, added up here: one launch fewer.
__global__ __launch_bounds__(kScanThreads) void scan_tiles_final(const int64_t* __restrict__ in, int64_t n,
                                                                 const int64_t* __restrict__ sums,
                                                                 int64_t* __restrict__ offsets, int prefix_self) {
  __shared__ ScanStage<kScanThreads> st;
  int64_t tile_prefix;
  if (prefix_self) {
    int64_t p = 0;
    for (int64_t j = threadIdx.x; j < (int64_t)blockIdx.x; j += kScanThreads) p += sums[j];
    block_exclusive_scan<kScanThreads>(p, st.wave, &tile_prefix);
  } else {
    tile_prefix = sums[blockIdx.x];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) offsets[0] = 0;
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int64_t v[kScanItems];
  load_scan_tile<kScanThreads>(in, n, base, v);
  scan_tile<kScanThreads>(v, n, base, tile_prefix, st, offsets);
}

// ------------------------------------------------------ list truncation --

struct TakeArgs {
  const int64_t* in_offsets;
  const uint8_t* row_valid;
  int64_t rows, n_in, max_length;
  int32_t truncation;
  int64_t* lengths;
  int64_t* starts;
  int32_t* error_count;
};

// The rows of one scan tile: kept counts, first kept elements, and the tile's
// sum for the offsets scan that follows (rows and sums in a launch each took
// 8.4 us for 409600 rows; together 4.9).  Offsets outside [0, n_in] or
// decreasing are clamped (and counted); a null row keeps nothing.
__global__ __launch_bounds__(kScanThreads) void bag_take_kernel(TakeArgs a, int64_t* __restrict__ sums) {
  __shared__ int64_t smem[kScanThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int64_t lo[kScanItems], hi[kScanItems];
  bool present[kScanItems];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t r = base + (int64_t)k * kScanThreads + threadIdx.x;
    const int64_t rc = r < a.rows ? r : a.rows - 1;
    lo[k] = ld_policy(a.in_offsets + rc);
    hi[k] = ld_policy(a.in_offsets + rc + 1);
    present[k] = a.row_valid == nullptr || ld_policy(a.row_valid + rc) != 0;
  }
  // A null row keeps nothing, except under tail truncation: the reference
  // rebuilds tail-truncated lists from the raw offsets (src/dataloader.py:
  // 8583-8604), so a null row with a non-empty span keeps its last elements.
  const bool tail_cut = a.truncation == MDL_TRUNCATE_TAIL && a.max_length >= 0;
  int64_t s = 0;
  int bad = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t r = base + (int64_t)k * kScanThreads + threadIdx.x;
    if (r >= a.rows) continue;
    bool wrong = false;
    if (lo[k] < 0 || lo[k] > a.n_in) {
      lo[k] = lo[k] < 0 ? 0 : a.n_in;
      wrong = true;
    }
    if (hi[k] < lo[k] || hi[k] > a.n_in) {
      hi[k] = hi[k] < lo[k] ? lo[k] : a.n_in;
      wrong = true;
    }
    const int64_t len = present[k] || tail_cut ? hi[k] - lo[k] : 0;
    const int64_t take = a.max_length >= 0 && len > a.max_length ? a.max_length : len;
    a.lengths[r] = take;
    a.starts[r] = a.truncation == MDL_TRUNCATE_HEAD ? lo[k] : hi[k] - take;
    s += take;
    bad += wrong;
  }
  if (bad && a.error_count != nullptr) atomicAdd(a.error_count, bad);
  const int64_t t = block_sum_i64(s, smem);
  if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

constexpr int kGatherThreads = 256;  // rows per block pass, one thread each to stage them
constexpr int kGatherFlight = 4;     // kept entries a thread has in flight

// Each block pass takes 256 consecutive rows: it stages their kept offsets
// and first source elements in LDS (coalesced), then walks their kept
// entries -- one contiguous stretch of the output -- 256 at a time, each
// thread finding its row by a search in LDS.  A thread's search and its
// element's load are one dependent chain, so four entries go side by side
// (one at a time: 55 us for 8.5 M kept of 9.8 M ids; four: 31,
// 5.0 TB/s).
// The grid then zeroes the entries past the kept total.
__global__ __launch_bounds__(kGatherThreads) void bag_gather_kernel(
    const int64_t* __restrict__ out_offsets, const int64_t* __restrict__ starts, int64_t rows,
    const int64_t* __restrict__ raw, const uint8_t* __restrict__ elem_valid, int64_t num_buckets, int32_t mode,
    int32_t validate_nonzero, uint64_t mod_magic, int64_t* __restrict__ values, int64_t capacity,
    int32_t* __restrict__ error_count) {
  // kept offsets relative to the pass's first entry; past its last row, and
  // past 2^30 entries, a bound no searched entry reaches
  __shared__ int32_t s_off[kGatherThreads];
  __shared__ int64_t s_src[kGatherThreads];  // first source element of the row less its offset
  constexpr int64_t kFar = 1ll << 30;
  const int tid = threadIdx.x;
  int bad = 0;
  for (int64_t r0 = (int64_t)blockIdx.x * kGatherThreads; r0 < rows; r0 += (int64_t)gridDim.x * kGatherThreads) {
    const int nr = rows - r0 < kGatherThreads ? (int)(rows - r0) : kGatherThreads;
    const int64_t b = out_offsets[r0];
    const int64_t end = out_offsets[r0 + nr];
    const int64_t e = end < capacity ? end : capacity;
    // a stretch of more than 2^30 entries goes in windows
    for (int64_t w0 = b; w0 < e; w0 += kFar) {
      const int m = (int)(e - w0 < kFar ? e - w0 : kFar);
      const int64_t off = tid < nr ? out_offsets[r0 + tid] - w0 : kFar;
      s_off[tid] = (int32_t)(off > kFar ? kFar : (off < -1 ? -1 : off));
      s_src[tid] = tid < nr ? starts[r0 + tid] - off : 0;
      __syncthreads();
      for (int j0 = tid; j0 < m; j0 += kGatherThreads * kGatherFlight) {
        int row[kGatherFlight];
#pragma unroll
        for (int q = 0; q < kGatherFlight; ++q) row[q] = 0;
        // last row whose offset is at or before the entry
#pragma unroll
        for (int step = kGatherThreads / 2; step >= 1; step >>= 1) {
#pragma unroll
          for (int q = 0; q < kGatherFlight; ++q)
            row[q] += s_off[row[q] + step] <= j0 + q * kGatherThreads ? step : 0;
        }
        int64_t v[kGatherFlight];
        bool present[kGatherFlight];
#pragma unroll
        for (int q = 0; q < kGatherFlight; ++q) {
          const int j = j0 + q * kGatherThreads;
          const int64_t src = j < m ? s_src[row[q]] + j : s_src[row[0]] + j0;
          v[q] = ld_policy(raw + src);
          present[q] = elem_valid == nullptr || ld_policy(elem_valid + src) != 0;
        }
#pragma unroll
        for (int q = 0; q < kGatherFlight; ++q) {
          const int j = j0 + q * kGatherThreads;
          if (j < m) {
            const int64_t out = bucket_of(v[q], present[q], num_buckets, mode, validate_nonzero, mod_magic, bad);
            st_policy<kOutPolicy>(values + w0 + j, out);
          }
        }
      }
      __syncthreads();  // the next window or pass restages the LDS
    }
  }
  const int64_t total = out_offsets[rows];
  for (int64_t j = total + (int64_t)blockIdx.x * kGatherThreads + tid; j < capacity;
       j += (int64_t)gridDim.x * kGatherThreads)
    values[j] = 0;
  if (error_count != nullptr && bad) atomicAdd(error_count, bad);
}

// Window entries of every row of up to kLenFeatures sequence features: the
// rows' lengths clamped to [0, cap], one feature after the other.
constexpr int kLenFeatures = 16;
struct LenArgs {
  const int64_t* lengths[kLenFeatures];
  int64_t cap[kLenFeatures];
  int64_t end[kLenFeatures];  // rows of the features up to and with this one
  int32_t features;
};

__global__ __launch_bounds__(256) void clamp_lengths_kernel(LenArgs a, int64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int64_t start = 0;
  for (int f = 0; f < a.features; ++f) {
    if (i < a.end[f]) {
      const int64_t n = a.lengths[f][i - start];
      out[i] = n < 0 ? 0 : (n > a.cap[f] ? a.cap[f] : n);
      return;
    }
    start = a.end[f];
  }
}

static __global__ void zero_offset_kernel(int64_t* p) { *p = 0; }

// Tiles whose prefix the final kernel adds up itself.
constexpr int64_t kScanSelfPrefixTiles = 1024;

// The offsets of n lengths whose tile sums are in sums.
static int scan_from_sums(const int64_t* lengths, int64_t n, int64_t* sums, int64_t* offsets, hipStream_t s) {
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  const int self = tiles <= kScanSelfPrefixTiles ? 1 : 0;
  if (!self) {
    hipLaunchKernelGGL(scan_sums_single, dim3(1), dim3(kScanThreads), 0, s, sums, tiles);
    MDL_CHECK_LAUNCH("scan_sums_single");
  }
  hipLaunchKernelGGL(scan_tiles_final, dim3((unsigned)tiles), dim3(kScanThreads), 0, s, lengths, n, sums, offsets,
                     self);
  MDL_CHECK_LAUNCH("scan_tiles_final");
  return MDL_OK;
}

}  // namespace mdl

using namespace mdl;

extern "C" {

const char* mdl_last_error(void) { return g_last_error.c_str(); }

int32_t mdl_abi_version(void) { return 6; }

int mdl_bucketize(const int64_t* raw, const uint8_t* valid, int64_t n, int64_t num_buckets,
                  int32_t mode, int32_t validate_nonzero, int64_t* out, int32_t* error_count,
                  void* stream) {
  if (n < 0) return fail(MDL_ERR_INVALID, "mdl_bucketize: negative n");
  int rc = validate_bucket_mode("mdl_bucketize", mode, num_buckets);
  if (rc) return rc;
  if (n == 0) return MDL_OK;
  if (raw == nullptr || out == nullptr) return fail(MDL_ERR_INVALID, "mdl_bucketize: null pointer");
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(bucketize_kernel, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), raw,
                     valid, n, num_buckets, mode, validate_nonzero, out, error_count,
                     mod_magic_for(mode, num_buckets));
  MDL_CHECK_LAUNCH("bucketize_kernel");
  return MDL_OK;
}

int mdl_clamp_lengths(const uint64_t* lengths, const int64_t* rows, const int64_t* caps, int32_t num_features,
                      int64_t* clamped, void* stream) {
  if (num_features < 0) return fail(MDL_ERR_INVALID, "mdl_clamp_lengths: negative count");
  if (num_features > 0 && (!lengths || !rows || !caps || !clamped))
    return fail(MDL_ERR_INVALID, "mdl_clamp_lengths: null pointer");
  for (int32_t f0 = 0; f0 < num_features; f0 += kLenFeatures) {
    LenArgs a{};
    int64_t n = 0;
    a.features = num_features - f0 < kLenFeatures ? num_features - f0 : kLenFeatures;
    for (int32_t f = 0; f < a.features; ++f) {
      if (rows[f0 + f] < 0) return fail(MDL_ERR_INVALID, "mdl_clamp_lengths: negative rows");
      n += rows[f0 + f];
      a.lengths[f] = reinterpret_cast<const int64_t*>(lengths[f0 + f]);
      a.cap[f] = caps[f0 + f];
      a.end[f] = n;
    }
    const int64_t blocks = (n + 255) / 256;
    if (blocks > 0xffffff) return fail(MDL_ERR_UNSUPPORTED, "mdl_clamp_lengths: too many rows");
    if (n > 0) {
      hipLaunchKernelGGL(clamp_lengths_kernel, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), a, clamped);
      MDL_CHECK_LAUNCH("clamp_lengths_kernel");
    }
    clamped += n;
  }
  return MDL_OK;
}

size_t mdl_bag_truncate_workspace_bytes(int64_t rows) {
  const size_t scan = (mdl_offsets_workspace_bytes(rows) + 255) & ~size_t(255);
  return scan + (size_t)(rows > 0 ? rows : 1) * sizeof(int64_t);
}

int mdl_bag_truncate(const int64_t* in_offsets, const uint8_t* row_valid, int64_t rows, const int64_t* raw,
                     const uint8_t* elem_valid, int64_t n_in, int64_t max_length, int32_t truncation,
                     int32_t bucket_mode, int64_t num_buckets, int32_t validate_nonzero, int64_t* lengths,
                     int64_t* out_offsets, int64_t* values, int64_t values_capacity, int32_t* error_count,
                     void* workspace, size_t workspace_bytes, void* stream) {
  if (rows < 0 || n_in < 0 || values_capacity < 0)
    return fail(MDL_ERR_INVALID, "mdl_bag_truncate: negative count");
  if (truncation != MDL_TRUNCATE_HEAD && truncation != MDL_TRUNCATE_TAIL)
    return fail(MDL_ERR_INVALID, "mdl_bag_truncate: truncation must be head or tail");
  if (bucket_mode != MDL_BUCKET_NONE) {
    const int ok = validate_bucket_mode("mdl_bag_truncate", bucket_mode, num_buckets);
    if (ok) return ok;
  }
  if (out_offsets == nullptr || (rows > 0 && (in_offsets == nullptr || lengths == nullptr)) ||
      (values_capacity > 0 && values == nullptr) || (values_capacity > 0 && n_in > 0 && raw == nullptr))
    return fail(MDL_ERR_INVALID, "mdl_bag_truncate: null pointer");
  if (workspace_bytes < mdl_bag_truncate_workspace_bytes(rows) || workspace == nullptr)
    return fail(MDL_ERR_WORKSPACE, "mdl_bag_truncate: workspace too small");
  hipStream_t s = as_stream(stream);
  const size_t scan_bytes = (mdl_offsets_workspace_bytes(rows) + 255) & ~size_t(255);
  int64_t* starts = reinterpret_cast<int64_t*>(static_cast<char*>(workspace) + scan_bytes);
  int rc = MDL_OK;
  if (rows > 0) {
    TakeArgs t{in_offsets, row_valid, rows, n_in, max_length, truncation, lengths, starts, error_count};
    int64_t* sums = static_cast<int64_t*>(workspace);
    hipLaunchKernelGGL(bag_take_kernel, dim3((unsigned)((rows + kScanTile - 1) / kScanTile)), dim3(kScanThreads), 0, s,
                       t, sums);
    MDL_CHECK_LAUNCH("bag_take_kernel");
    rc = scan_from_sums(lengths, rows, sums, out_offsets, s);
  } else {
    rc = mdl_lengths_to_offsets(lengths, rows, out_offsets, workspace, scan_bytes, stream);
  }
  if (rc) return rc;
  if (values_capacity == 0) return MDL_OK;
  int64_t blocks = (rows + kGatherThreads - 1) / kGatherThreads;
  if (blocks < 256) blocks = 256;  // the zero fill past the kept total needs a grid of its own size
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(bag_gather_kernel, dim3((unsigned)blocks), dim3(kGatherThreads), 0, s, out_offsets, starts,
                     rows, raw,
                     elem_valid, num_buckets, bucket_mode, validate_nonzero, mod_magic_for(bucket_mode, num_buckets),
                     values, values_capacity, error_count);
  MDL_CHECK_LAUNCH("bag_gather_kernel");
  return MDL_OK;
}

size_t mdl_offsets_workspace_bytes(int64_t n) {
  int64_t tiles = (n + kScanTile - 1) / kScanTile;
  return (size_t)(tiles + 1) * sizeof(int64_t);
}

int mdl_lengths_to_offsets(const int64_t* lengths, int64_t n, int64_t* offsets, void* workspace,
                           size_t workspace_bytes, void* stream) {
  if (n < 0) return fail(MDL_ERR_INVALID, "mdl_lengths_to_offsets: negative n");
  hipStream_t s = as_stream(stream);
  if (n == 0) {
    // a kernel, not a memset: callers may capture this call in a graph
    hipLaunchKernelGGL(zero_offset_kernel, dim3(1), dim3(1), 0, s, offsets);
    MDL_CHECK_LAUNCH("zero_offset_kernel");
    return MDL_OK;
  }
  if (workspace_bytes < mdl_offsets_workspace_bytes(n))
    return fail(MDL_ERR_WORKSPACE, "mdl_lengths_to_offsets: workspace too small");
  if (n <= kScanOneBlock) {
    hipLaunchKernelGGL(scan_one_block, dim3(1), dim3(kScanOneThreads), 0, s, lengths, n, offsets);
    MDL_CHECK_LAUNCH("scan_one_block");
    return MDL_OK;
  }
  int64_t tiles = (n + kScanTile - 1) / kScanTile;
  int64_t* sums = static_cast<int64_t*>(workspace);
  hipLaunchKernelGGL(scan_tile_sums, dim3((unsigned)tiles), dim3(kScanThreads), 0, s, lengths, n, sums);
  MDL_CHECK_LAUNCH("scan_tile_sums");
  return scan_from_sums(lengths, n, sums, offsets, s);
}

}  // extern "C"
