// Lower-bound search of int32 needles in a sorted int32 array
// (torch.searchsorted(sorted, values, side='left', out_int32=True)), as the
// reference's run_searchsorted (src/torch/torch_searchsorted.h:33-82,
// tests/test_searchsorted.py).
//
// Each workgroup first stages every B-th haystack element in LDS
// (B = ceil(len / kSamples), so at most kSamples of them; the whole
// haystack when it fits).  A needle's lower bound c among the samples
// brackets its answer: sorted[(c-1)B] < key <= sorted[cB], so the answer
// lies in [(c-1)B + 1, min(cB, len)] (0 when c = 0), and a binary search
// over that window of fewer than B elements in global memory finishes it.
// The LDS stage replaces the upper levels of the search, whose probes all
// needles share; the lower levels are random probes into the haystack and
// bound the kernel.
#include "tcs_common.hpp"

namespace tcs {

constexpr int kSsThreads = 1024;
constexpr int kSsSamples = 16384;  // 64 KiB of LDS per workgroup

// The samples of `sorted` in LDS: every B-th element, at most kSsSamples.
struct SsSamples {
  int32_t B, ns;
};

__device__ __forceinline__ SsSamples stage_samples(int32_t* s_samp, const int32_t* __restrict__ sorted,
                                                   int32_t len) {
  const int32_t B = (int32_t)(((int64_t)len + kSsSamples - 1) / kSsSamples);
  const int32_t ns = len > 0 ? (int32_t)(((int64_t)len + B - 1) / B) : 0;  // <= kSsSamples
  for (int i = threadIdx.x; i < ns; i += kSsThreads) s_samp[i] = sorted[(int64_t)i * B];
  __syncthreads();
  return SsSamples{B, ns};
}

// Lower bound of key in sorted[lo, lo + count] (the answer is known to lie
// there): a binary search in global memory.
__device__ __forceinline__ int32_t lower_bound_in(const int32_t* __restrict__ sorted, int32_t lo, int32_t count,
                                                  int32_t key) {
  while (count > 0) {
    const int32_t half = count >> 1;
    const bool right = sorted[lo + half] < key;
    lo = right ? lo + half + 1 : lo;
    count = right ? count - half - 1 : half;
  }
  return lo;
}

// Lower bound of key in sorted[0, len): the samples bracket it, then a
// search over the window of fewer than B elements between two samples.
__device__ __forceinline__ int32_t lower_bound_staged(const int32_t* s_samp, SsSamples sm,
                                                      const int32_t* __restrict__ sorted, int32_t len,
                                                      int32_t key) {
  // Invariant of both searches: the answer lies in [lo, lo + count].
  int32_t lo = 0, count = sm.ns;
  while (count > 0) {
    const int32_t half = count >> 1;
    const bool right = s_samp[lo + half] < key;
    lo = right ? lo + half + 1 : lo;
    count = right ? count - half - 1 : half;
  }
  const int64_t hi = (int64_t)lo * sm.B < len ? (int64_t)lo * sm.B : len;
  const int32_t glo = lo == 0 ? 0 : (lo - 1) * sm.B + 1;
  return lower_bound_in(sorted, glo, lo == 0 ? 0 : (int32_t)hi - glo, key);
}

__global__ __launch_bounds__(kSsThreads) void searchsorted_kernel(const int32_t* __restrict__ sorted, int32_t len,
                                                                  const int32_t* __restrict__ values,
                                                                  int32_t* __restrict__ out, int64_t nv) {
  __shared__ int32_t s_samp[kSsSamples];
  const SsSamples sm = stage_samples(s_samp, sorted, len);
  const int64_t stride = (int64_t)gridDim.x * kSsThreads;
  for (int64_t i = (int64_t)blockIdx.x * kSsThreads + threadIdx.x; i < nv; i += stride)
    out[i] = lower_bound_staged(s_samp, sm, sorted, len, values[i]);
}

// ---------------------------------------------------------------------------
// Few needles: sixteen lanes a needle.  Each step compares the needle with 15
// evenly spaced elements of the range that holds its answer and keeps one
// sixteenth of it, so 2^24 elements take six dependent reads, with nothing
// staged first.  Bound by the reads' latency (2^12 needles into 2^24: 5.4 us,
// the sampled search 29).
// ---------------------------------------------------------------------------
constexpr int kSfThreads = 256, kSfLanes = 16;
__global__ __launch_bounds__(kSfThreads) void searchsorted_few_kernel(const int32_t* __restrict__ sorted, int32_t len,
                                                                      const int32_t* __restrict__ values,
                                                                      int32_t* __restrict__ out, int64_t nv) {
  const int lane = __lane_id(), q = lane % kSfLanes, g = lane / kSfLanes;
  const int64_t i = ((int64_t)blockIdx.x * kSfThreads + threadIdx.x) / kSfLanes;
  const int32_t key = values[i < nv ? i : nv - 1];
  // The answer lies in [lo, lo + count].
  int32_t lo = 0, count = len;
  while (__ballot(count > 0) != 0) {
    // Lane q < 15 looks at the last element of part q; parts of equal size
    // but the last, which takes what is left (up to `part` elements).
    const int32_t part = count / kSfLanes + 1;
    const int32_t at = (q + 1) * part - 1;
    const bool less = q < kSfLanes - 1 && at < count && sorted[lo + at] < key;
    const int32_t c = __builtin_popcount((uint32_t)(__ballot(less) >> (g * kSfLanes)) & 0xffffu);
    // Parts before c lie below the needle; the answer is in part c, at most
    // the index of its last element.
    lo += c * part;
    const int32_t left = count - c * part;
    count = left < part ? left : part - 1;
  }
  if (q == 0 && i < nv) out[i] = lo;
}

// ---------------------------------------------------------------------------
// Bucket index (tcs_searchsorted_indexed).  Keys map to order keys
// u = bits ^ 0x80000000 (unsigned order = signed order); the haystack's
// order keys span [umin, umax] (its two ends).  Bucket of u:
// (u - umin) >> shift, with shift the smallest that leaves at most 2^bits
// buckets.  start[k] = first index whose bucket is >= k (k <= the number of
// buckets used), so a needle in bucket k has its lower bound in [start[k],
// start[k + 1]]: elements before start[k] are in lower buckets, hence
// smaller, and elements from start[k + 1] on are in higher buckets, hence
// larger.  With keys spread over their range a bucket holds 4 to 8 elements
// and the search is one table read and one or two 16-byte reads; when more
// than a sixteenth of the haystack lies in buckets of over kSsWide elements
// (clustered keys), every needle takes the sampled search instead.
// ---------------------------------------------------------------------------
constexpr int kSsBuildBlocks = 512;  // build workgroups: one count word each, before the table
constexpr int32_t kSsWide = 64;
constexpr int kSsLongGaps = 256;     // table gaps above kSsLongGap: at most 2^22 / kSsLongGap in all
constexpr uint32_t kSsLongGap = 16384;

struct BucketMap {
  uint32_t umin, umax;
  int shift;
  uint32_t used;  // buckets that hold order keys of [umin, umax]
};

__device__ __forceinline__ uint32_t order_key(int32_t v) { return (uint32_t)v ^ 0x80000000u; }

__device__ __forceinline__ BucketMap bucket_map(const int32_t* __restrict__ sorted, int32_t len, int bits) {
  BucketMap m;
  m.umin = order_key(sorted[0]);
  m.umax = order_key(sorted[len - 1]);
  const uint32_t range = m.umax - m.umin;
  const int width = range == 0 ? 0 : 32 - __builtin_clz(range);
  m.shift = width > bits ? width - bits : 0;
  m.used = (range >> m.shift) + 1u;  // <= 2^bits
  return m;
}

// The table in one pass over the haystack: element i starts the buckets after
// its predecessor's up to its own (2^24 elements 24 us; a search per entry took
// 86).  A wave takes 256 consecutive elements at a time, four rows of 64, so an element's predecessor is the lane's below
// (or the last lane's of the row before) and the element 64 places back the
// lane's own of the row before.  Few buckets start at one element as a rule;
// a wave fills gaps of more than 8 together, the workgroup those above
// kSsLongGap.  wide[block] = the block's elements whose bucket holds the
// element kSsWide places back too.
__global__ __launch_bounds__(kSsThreads) void bucket_start_kernel(const int32_t* __restrict__ sorted, int32_t len,
                                                                  int32_t per_block, int bits,
                                                                  int32_t* __restrict__ wide,
                                                                  int32_t* __restrict__ start) {
  static_assert(kSsWide == kWave, "the element kSsWide places back is the row before's");
  constexpr int R = 4;
  __shared__ uint32_t s_first[kSsLongGaps], s_last[kSsLongGaps];
  __shared__ int32_t s_at[kSsLongGaps];
  __shared__ int s_gaps, s_wide;
  if (threadIdx.x == 0) s_gaps = s_wide = 0;
  const BucketMap m = bucket_map(sorted, len, bits);
  __syncthreads();
  const int lane = __lane_id(), wid = threadIdx.x / kWave;
  const int64_t b0 = (int64_t)blockIdx.x * per_block;
  const int64_t b1 = b0 + per_block < len ? b0 + per_block : len;
  auto bucket = [&](int32_t v) { return (order_key(v) - m.umin) >> m.shift; };
  int nwide = 0;
  for (int64_t w = b0 + (int64_t)wid * (R * kWave); w < b1; w += (int64_t)kSsThreads * R) {
    // Row -1 first; rows past the end repeat the haystack's last element.
    int32_t v[R + 1];
#pragma unroll
    for (int j = 0; j <= R; ++j) {
      const int64_t p = w + (j - 1) * kWave + lane;
      v[j] = sorted[p < 0 ? 0 : (p < len ? p : len - 1)];
    }
    uint32_t b[R + 1];
#pragma unroll
    for (int j = 0; j <= R; ++j) b[j] = bucket(v[j]);
#pragma unroll
    for (int j = 1; j <= R; ++j) {
      const int64_t p = w + (j - 1) * kWave + lane;
      const uint32_t left = dpp_mov<kWaveShr1>(b[j]);
      const uint32_t above = (uint32_t)readlane((int)b[j - 1], kWave - 1);
      const uint32_t prev = lane > 0 ? left : above;
      const uint32_t first = p == 0 ? 0u : prev + 1u;
      const uint32_t gap = p < b1 ? b[j] + 1u - first : 0u;  // entries [first, first + gap) start here
      nwide += p < b1 && p >= kSsWide && b[j - 1] == b[j] ? 1 : 0;
      if (gap <= 8u) {
        for (uint32_t k = 0; k < gap; ++k) start[first + k] = (int32_t)p;
      }
      uint64_t more = __ballot(gap > 8u);
      while (more != 0) {
        const int l = __builtin_ctzll(more);
        more &= more - 1;
        const uint32_t f = (uint32_t)readlane((int)first, l), g = (uint32_t)readlane((int)gap, l);
        const int32_t at = (int32_t)(w + (j - 1) * kWave) + l;
        if (g > kSsLongGap) {
          if (lane == 0) {
            const int q = atomicAdd(&s_gaps, 1);
            s_first[q] = f;
            s_last[q] = f + g;
            s_at[q] = at;
          }
        } else {
          for (uint32_t k = lane; k < g; k += kWave) start[f + k] = at;
        }
      }
    }
  }
  nwide = wave_sum(nwide);
  if (lane == 0 && nwide) atomicAdd(&s_wide, nwide);
  __syncthreads();
  for (int q = 0; q < s_gaps; ++q) {
    for (uint32_t k = s_first[q] + threadIdx.x; k < s_last[q]; k += kSsThreads) start[k] = s_at[q];
  }
  if (threadIdx.x == 0) {
    wide[blockIdx.x] = s_wide;
    if (blockIdx.x == 0) start[m.used] = len;
  }
}

// Four or two 32-bit elements from an address of 4-byte alignment.
typedef int32_t i32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef int32_t i32x2u __attribute__((ext_vector_type(2), aligned(4)));

// Lower bounds of U needles by the table.  `sorted` holds at least four
// elements.
template <int U>
__device__ __forceinline__ void bucket_search(const int32_t* __restrict__ sorted, int32_t len, const BucketMap& m,
                                              const int32_t* __restrict__ start, const int32_t (&key)[U],
                                              int32_t (&r)[U]) {
  int32_t lo[U], hi[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t o = order_key(key[u]);
    const uint32_t k = (o - m.umin) >> m.shift;
    const bool in = o >= m.umin && o <= m.umax;
    const uint32_t q = in ? k : 0u;
    const i32x2u se = *reinterpret_cast<const i32x2u*>(start + q);
    lo[u] = se[0];
    hi[u] = se[1];
    if (!in) lo[u] = hi[u] = o < m.umin ? 0 : len;
    // A bucket of one order key: its start is the answer.
    if (m.shift == 0) hi[u] = lo[u];
  }
  int32_t at[U], c[U];
  i32x4u e[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    while (hi[u] - lo[u] > 32) {
      const int32_t mid = lo[u] + (hi[u] - lo[u]) / 2;
      if (sorted[mid] < key[u]) {
        lo[u] = mid + 1;
      } else {
        hi[u] = mid;
      }
    }
    // Elements before lo are smaller than the needle and those from hi on
    // are not, so counting the smaller ones from any index <= lo is right.
    at[u] = lo[u] < len - 4 ? lo[u] : len - 4;
    e[u] = *reinterpret_cast<const i32x4u*>(sorted + at[u]);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    c[u] = (e[u][0] < key[u]) + (e[u][1] < key[u]) + (e[u][2] < key[u]) + (e[u][3] < key[u]);
    while (c[u] == 4 && at[u] + 4 < hi[u]) {
      at[u] = at[u] + 4 < len - 4 ? at[u] + 4 : len - 4;
      e[u] = *reinterpret_cast<const i32x4u*>(sorted + at[u]);
      c[u] = (e[u][0] < key[u]) + (e[u][1] < key[u]) + (e[u][2] < key[u]) + (e[u][3] < key[u]);
    }
    r[u] = lo[u] == hi[u] ? lo[u] : at[u] + c[u];
  }
}

// More than a sixteenth of the haystack in wide buckets (every workgroup
// sums the build's counts).  Ends with a barrier.
__device__ __forceinline__ bool bucket_clustered(const int32_t* __restrict__ wide, int32_t len, const BucketMap& m,
                                                 int* s_sum) {
  if (threadIdx.x == 0) *s_sum = 0;
  __syncthreads();
  const int t = threadIdx.x;
  int v = t < kSsBuildBlocks ? wide[t] : 0;
  if (t < kSsBuildBlocks) {
    v = wave_sum(v);
    if (__lane_id() == 0 && v) atomicAdd(s_sum, v);
  }
  __syncthreads();
  return m.shift > 0 && *s_sum > len / 16;
}

// Needles in input order, four per thread in flight.
constexpr int kSsU = 4;
__global__ __launch_bounds__(kSsThreads) void searchsorted_indexed_kernel(const int32_t* __restrict__ sorted,
                                                                          int32_t len, int bits,
                                                                          const int32_t* __restrict__ wide,
                                                                          const int32_t* __restrict__ start,
                                                                          const int32_t* __restrict__ values,
                                                                          int32_t* __restrict__ out, int64_t nv) {
  __shared__ int32_t s_samp[kSsSamples];
  const BucketMap m = bucket_map(sorted, len, bits);
  const int64_t stride = (int64_t)gridDim.x * kSsThreads;
  const int64_t first = (int64_t)blockIdx.x * kSsThreads + threadIdx.x;
  if (bucket_clustered(wide, len, m, s_samp)) {
    __syncthreads();  // s_samp is rewritten
    const SsSamples sm = stage_samples(s_samp, sorted, len);
    for (int64_t i = first; i < nv; i += stride) out[i] = lower_bound_staged(s_samp, sm, sorted, len, values[i]);
    return;
  }
  for (int64_t i = first; i < nv; i += stride * kSsU) {
    int32_t key[kSsU], r[kSsU];
#pragma unroll
    for (int u = 0; u < kSsU; ++u) key[u] = values[i + u * stride < nv ? i + u * stride : nv - 1];
    bucket_search<kSsU>(sorted, len, m, start, key, r);
#pragma unroll
    for (int u = 0; u < kSsU; ++u)
      if (i + u * stride < nv) out[i + u * stride] = r[u];
  }
}

// Haystacks beyond an XCD's L2: a workgroup takes 8192 needles at a time and
// searches them grouped by the top eight bits of their place in the key
// range, lowest group first, so that all workgroups sweep the haystack and
// the table in the same direction and a line fetched into an L2 serves the
// needles of every workgroup of that XCD.  2^24 needles into 2^24 keys: 520
// us, in input order 650 (each needle fetches two lines past the L2s).
constexpr int kSgThreads = 512, kSgRows = 16, kSgTile = kSgThreads * kSgRows;
__global__ __launch_bounds__(kSgThreads) void searchsorted_grouped_kernel(const int32_t* __restrict__ sorted,
                                                                          int32_t len, int bits,
                                                                          const int32_t* __restrict__ wide,
                                                                          const int32_t* __restrict__ start,
                                                                          const int32_t* __restrict__ values,
                                                                          int32_t* __restrict__ out, int64_t nv) {
  static_assert(kSgThreads >= kSsBuildBlocks && kSgTile <= 65536, "one count word per thread; 16-bit positions");
  __shared__ int32_t s_key[kSgTile];
  __shared__ uint16_t s_at[kSgTile];
  __shared__ uint32_t s_cnt[256];
  __shared__ uint32_t s_wsum[4];
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  const BucketMap m = bucket_map(sorted, len, bits);
  if (bucket_clustered(wide, len, m, reinterpret_cast<int*>(s_cnt))) {
    __syncthreads();
    const int32_t B = (int32_t)(((int64_t)len + kSgTile - 1) / kSgTile);
    const int32_t ns = (int32_t)(((int64_t)len + B - 1) / B);
    for (int i = tid; i < ns; i += kSgThreads) s_key[i] = sorted[(int64_t)i * B];
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * kSgThreads + tid; i < nv; i += (int64_t)gridDim.x * kSgThreads)
      out[i] = lower_bound_staged(s_key, SsSamples{B, ns}, sorted, len, values[i]);
    return;
  }
  const uint32_t range = m.umax - m.umin;
  const int width = range == 0 ? 0 : 32 - __builtin_clz(range);
  const int gshift = width > 8 ? width - 8 : 0;
  for (int64_t t0 = (int64_t)blockIdx.x * kSgTile; t0 < nv; t0 += (int64_t)gridDim.x * kSgTile) {
    const int tvalid = t0 + kSgTile <= nv ? kSgTile : (int)(nv - t0);
    __syncthreads();  // the previous tile's counts and results have been read
    if (tid < 256) s_cnt[tid] = 0;
    int32_t key[kSgRows];
    uint32_t gr[kSgRows];  // group << 16 | rank in it (in no particular order)
#pragma unroll
    for (int i = 0; i < kSgRows; ++i) {
      const int p = i * kSgThreads + tid;
      key[i] = values[t0 + (p < tvalid ? p : tvalid - 1)];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSgRows; ++i) {
      const uint32_t o = order_key(key[i]);
      const uint32_t g = o <= m.umin ? 0u : (o >= m.umax ? range >> gshift : (o - m.umin) >> gshift);
      gr[i] = g << 16;
      if (i * kSgThreads + tid < tvalid) gr[i] |= atomicAdd(&s_cnt[g], 1u);
    }
    __syncthreads();
    uint32_t cnt = 0, incl = 0;
    if (tid < 256) {
      cnt = s_cnt[tid];
      incl = wave_incl_scan(cnt);
      if (lane == kWave - 1) s_wsum[wid] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t before = incl - cnt;
      for (int w = 0; w < wid; ++w) before += s_wsum[w];
      s_cnt[tid] = before;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSgRows; ++i) {
      const int p = i * kSgThreads + tid;
      if (p < tvalid) {
        const uint32_t q = s_cnt[gr[i] >> 16] + (gr[i] & 0xffffu);
        s_key[q] = key[i];
        s_at[q] = (uint16_t)p;
      }
    }
    __syncthreads();
    int32_t r[kSgRows];
#pragma unroll
    for (int i = 0; i < kSgRows; i += kSsU) {
      int32_t k4[kSsU], r4[kSsU];
#pragma unroll
      for (int u = 0; u < kSsU; ++u) {
        const int q = (i + u) * kSgThreads + tid;
        k4[u] = s_key[q < tvalid ? q : tvalid - 1];
      }
      bucket_search<kSsU>(sorted, len, m, start, k4, r4);
#pragma unroll
      for (int u = 0; u < kSsU; ++u) r[i + u] = r4[u];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSgRows; ++i) {
      const int q = i * kSgThreads + tid;
      if (q < tvalid) s_key[s_at[q]] = r[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSgRows; ++i) {
      const int p = i * kSgThreads + tid;
      if (p < tvalid) out[t0 + p] = s_key[p];
    }
  }
}

// The grouped kernel from these sizes on: below, the grouping costs more than
// the lines it saves (2^20 elements, 2^24 needles: 238 us against 205; 2^22
// elements, 2^24 needles: 338 against 502; 2^24 elements, 2^20 needles: 87
// against 65).
constexpr int64_t kSgMinLen = (int64_t)1 << 20, kSgMinNeedles = (int64_t)3 << 19;

// Whether the needles are too few to pay for staging samples in every
// workgroup, or for a table (2^14 needles into 2^20 elements: 5.3 us against
// 14.7 sampled; 2^15 into 2^24: 16 us, with a table 28).
static bool searchsorted_few(int64_t len, int64_t nv) {
  if (len <= kSsSamples) return nv <= (int64_t)1 << 13;
  return nv <= (len > ((int64_t)1 << 22) ? (int64_t)1 << 16 : (int64_t)1 << 15);
}

// Four workgroups per CU of the current device (two are resident at a
// time with 64 KiB of LDS each; the second pair evens out the tail).
static uint32_t searchsorted_grid() {
  static std::atomic<int> cached[kMaxCachedDevices];
  return (uint32_t)device_cached(cached, [](int dev) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    return 4 * cus;
  });
}

}  // namespace tcs

extern "C" {

int tcs_searchsorted(const int32_t* sorted, int64_t sorted_len, const int32_t* values, int32_t* out,
                     int64_t num_values, void* stream) {
  using namespace tcs;
  if (sorted_len < 0 || num_values < 0 || sorted_len >= ((int64_t)1 << 31)) return TCS_ERR_INVALID_ARG;
  if (num_values == 0) return TCS_OK;
  if (!values || !out || (sorted_len > 0 && !sorted)) return TCS_ERR_INVALID_ARG;
  if (searchsorted_few(sorted_len, num_values)) {
    constexpr int64_t per = kSfThreads / kSfLanes;
    hipLaunchKernelGGL(searchsorted_few_kernel, dim3((uint32_t)((num_values + per - 1) / per)), dim3(kSfThreads), 0,
                       static_cast<hipStream_t>(stream), sorted, (int32_t)sorted_len, values, out, num_values);
    TCS_CHECK_LAUNCH();
    return TCS_OK;
  }
  const uint64_t need = (uint64_t)((num_values + kSsThreads - 1) / kSsThreads);
  const uint64_t cap = searchsorted_grid();
  const uint32_t blocks = (uint32_t)(need < cap ? need : cap);
  hipLaunchKernelGGL(searchsorted_kernel, dim3(blocks), dim3(kSsThreads), 0, static_cast<hipStream_t>(stream),
                     sorted, (int32_t)sorted_len, values, out, num_values);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

static int floor_log2(int64_t v) {
  int b = 0;
  while (b < 62 && ((int64_t)1 << (b + 1)) <= v) ++b;
  return b;
}

static int clamp_int(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// The least and the preferred workspace.  The build's counts and a table of
// 2^bits + 1 entries go into whatever is given: 4 to 8 elements a bucket
// (2^22 buckets at most) with the preferred one.
size_t tcs_searchsorted_workspace_bytes(int64_t sorted_len) {
  if (sorted_len <= 0) return 0;
  return (((size_t)1 << clamp_int(floor_log2(sorted_len) - 4, 10, 20)) + 1) * sizeof(int32_t);
}

static int bucket_bits(int64_t len) { return clamp_int(floor_log2(len) - 2, 10, 22); }

size_t tcs_searchsorted_preferred_bytes(int64_t sorted_len) {
  if (sorted_len <= 0) return 0;
  return (tcs::kSsBuildBlocks + ((size_t)1 << bucket_bits(sorted_len)) + 1) * sizeof(int32_t);
}

int tcs_searchsorted_indexed(const int32_t* sorted, int64_t sorted_len, const int32_t* values, int32_t* out,
                             int64_t num_values, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace tcs;
  if (sorted_len < 0 || num_values < 0 || sorted_len >= ((int64_t)1 << 31)) return TCS_ERR_INVALID_ARG;
  if (num_values == 0) return TCS_OK;
  if (!values || !out || (sorted_len > 0 && !sorted)) return TCS_ERR_INVALID_ARG;
  if (sorted_len == 0) return tcs_searchsorted(sorted, sorted_len, values, out, num_values, stream);
  if (!workspace || workspace_bytes < tcs_searchsorted_workspace_bytes(sorted_len)) return TCS_ERR_WORKSPACE;
  // A haystack that fits in LDS needs no table.
  if (sorted_len <= kSsSamples || searchsorted_few(sorted_len, num_values))
    return tcs_searchsorted(sorted, sorted_len, values, out, num_values, stream);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t entries = (int64_t)(workspace_bytes / sizeof(int32_t)) - kSsBuildBlocks - 1;
  const int bits = clamp_int(bucket_bits(sorted_len), 1, floor_log2(entries));
  auto* wide = static_cast<int32_t*>(workspace);
  int32_t* start = wide + kSsBuildBlocks;
  const int32_t len = (int32_t)sorted_len;
  const int32_t per_block = (len + kSsBuildBlocks - 1) / kSsBuildBlocks;
  hipLaunchKernelGGL(bucket_start_kernel, dim3(kSsBuildBlocks), dim3(kSsThreads), 0, st, sorted, len, per_block, bits,
                     wide, start);
  TCS_CHECK_LAUNCH();
  const uint64_t cap = searchsorted_grid();
  if (sorted_len > kSgMinLen && num_values > kSgMinNeedles) {
    const uint64_t tiles = (uint64_t)((num_values + kSgTile - 1) / kSgTile);
    const uint64_t resident = cap / 4 * 3;  // three workgroups of 49 KiB of LDS on each CU
    hipLaunchKernelGGL(searchsorted_grouped_kernel, dim3((uint32_t)(tiles < resident ? tiles : resident)),
                       dim3(kSgThreads), 0, st, sorted, len, bits, wide, start, values, out, num_values);
  } else {
    const uint64_t need = (uint64_t)((num_values + kSsThreads - 1) / kSsThreads);
    hipLaunchKernelGGL(searchsorted_indexed_kernel, dim3((uint32_t)(need < cap ? need : cap)), dim3(kSsThreads), 0, st,
                       sorted, len, bits, wide, start, values, out, num_values);
  }
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

}  // extern "C"
