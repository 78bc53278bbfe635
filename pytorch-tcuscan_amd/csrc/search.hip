// Lower-bound search of int32 needles in a sorted int32 array
// (torch.searchsorted(sorted, values, side='left', out_int32=True)), as the
// reference's run_searchsorted (src/torch/torch_searchsorted.h:33-82,
// tests/test_searchsorted.py).
//
// Four ways, by size: sixteen lanes a needle (few needles); a search tree of
// samples in LDS (short haystacks, or no workspace); a table of buckets over
// the key range; and, for many needles, needles grouped by slices of the
// haystack that are searched in LDS.
#include "tcs_common.hpp"

namespace tcs {

constexpr int kSsThreads = 1024;
constexpr int kSsLog = 14, kSsNodes = 1 << kSsLog;  // 64 KiB of LDS per workgroup
constexpr int kSsU = 4;                             // needles of a thread in flight

// A search tree of 2^log - 1 nodes over the sorted samples p[0], p[step],
// ..., p[(ns - 1) * step] in breadth-first order (children of node k: 2k and
// 2k + 1): the first steps of a wave's lanes fall on distinct banks, where
// the halving of a sorted array puts them on one.  Nodes past the samples
// hold INT32_MAX, which no key exceeds.  A workgroup of kSsThreads.
__device__ __forceinline__ void stage_tree(int32_t* tree, int log, const int32_t* __restrict__ p, int64_t step,
                                           int32_t ns) {
  constexpr int R = 8;  // loads in flight
  const int32_t nodes = 1 << log;
  for (int32_t r0 = threadIdx.x; r0 < nodes; r0 += R * kSsThreads) {
    int32_t v[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int32_t r = r0 + i * kSsThreads - 1;
      v[i] = ns > 0 ? p[(r < 0 ? 0 : (r < ns ? r : ns - 1)) * step] : 0;
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int32_t r = r0 + i * kSsThreads;  // rank of the sample, from 1
      if (r > 0 && r < nodes) {
        const int z = __builtin_ctz(r);
        tree[(nodes >> (z + 1)) + (r >> (z + 1))] = r <= ns ? v[i] : 0x7fffffff;
      }
    }
  }
}

// c[u] = number of samples of the tree below key[u].  Three vector
// instructions a step: the node's byte offset, not its number, is carried.
template <int U>
__device__ __forceinline__ void tree_count(const int32_t* tree, int log, const int32_t (&key)[U], int32_t (&c)[U]) {
  const char* t = reinterpret_cast<const char*>(tree);
#pragma unroll
  for (int u = 0; u < U; ++u) c[u] = 4;
  for (int s = 0; s < log; ++s) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      c[u] = (c[u] << 1) + (*reinterpret_cast<const int32_t*>(t + c[u]) < key[u] ? 4 : 0);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) c[u] = (c[u] >> 2) - (1 << log);
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

// All needles by samples: every B-th element, B the least that leaves the
// tree room for them, then the window of fewer than B elements between two
// samples.  2^24 needles into 2^14 elements: 40.7 us (4.1e11 needles a
// second; bound by the steps' LDS reads), 187 with one needle a thread at a
// time and a sorted array of samples.
//
// narrow(key, lo, hi) may move the ends of the window [lo, hi] that the answer
// lies in closer together.
template <int U, class F>
__device__ __forceinline__ void search_staged(int32_t* s_tree, const int32_t* __restrict__ sorted, int32_t len,
                                              const int32_t* __restrict__ values, int32_t* __restrict__ out,
                                              int64_t nv, F narrow) {
  if (len == 0) {
    for (int64_t i = (int64_t)blockIdx.x * kSsThreads + threadIdx.x; i < nv; i += (int64_t)gridDim.x * kSsThreads)
      out[i] = 0;
    return;
  }
  const int32_t B = (int32_t)(((int64_t)len + kSsNodes - 1) / kSsNodes);
  const int32_t ns = (int32_t)(((int64_t)len + B - 1) / B);  // at most kSsNodes: the first apart, the rest in the tree
  const int log = ns > 1 ? 32 - __builtin_clz(ns - 1) : 0;
  stage_tree(s_tree, log, sorted + B, B, ns - 1);
  const int32_t first = sorted[0];
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * kSsThreads;
  for (int64_t i = (int64_t)blockIdx.x * kSsThreads + threadIdx.x; i < nv; i += U * stride) {
    int32_t key[U], c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) key[u] = values[i + u * stride < nv ? i + u * stride : nv - 1];
    tree_count<U>(s_tree, log, key, c);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      c[u] += first < key[u] ? 1 : 0;
      int32_t lo = c[u];
      if (B > 1 && lo > 0) {
        // sorted[(c - 1) B] < key <= sorted[c B].
        int32_t hi = (int64_t)c[u] * B < len ? c[u] * B : len;
        lo = (c[u] - 1) * B + 1;
        narrow(key[u], lo, hi);
        lo = lower_bound_in(sorted, lo, hi - lo, key[u]);
      }
      if (i + u * stride < nv) out[i + u * stride] = lo;
    }
  }
}

// U needles of a thread in flight.
template <int U>
__global__ __launch_bounds__(kSsThreads) void searchsorted_kernel(const int32_t* __restrict__ sorted, int32_t len,
                                                                  const int32_t* __restrict__ values,
                                                                  int32_t* __restrict__ out, int64_t nv) {
  __shared__ int32_t s_tree[kSsNodes];
  search_staged<U>(s_tree, sorted, len, values, out, nv, [](int32_t, int32_t&, int32_t&) {});
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
// From this length on the sampled search that the table falls back to also
// looks its window up in the table: between two samples lie 512 elements and
// more, in a bucket often fewer (2^24 needles into 2^24 clustered elements with
// the least workspace: 1524 us by samples alone, 626 so, 644 by a search of
// every bucket of up to 2048; 2^19 with the preferred one 108, 73, 133).
constexpr int32_t kSsNarrowLen = 1 << 22;
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
// its predecessor's up to its own (2^24 elements 25 us; a search per entry took
// 86).  A wave takes 256 consecutive elements at a time, four rows of 64, so an element's predecessor is the lane's below
// (or the last lane's of the row before) and the element 64 places back the
// lane's own of the row before.  Few buckets start at one element as a rule;
// a wave fills gaps of more than 8 together, the workgroup those above
// kSsLongGap.  wide[block] = the block's elements whose bucket holds the
// element kSsWide places back too.
__global__ __launch_bounds__(kSsThreads) void bucket_start_kernel(const int32_t* __restrict__ sorted, int32_t len,
                                                                  int64_t per_block, int bits,
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
  // A haystack that is not sorted may hold keys outside [umin, umax] and
  // buckets that fall.  Buckets end at m.used - 1 and only a rise writes
  // entries, so every write lies in the table; and as the first element's
  // bucket is 0 and the last one's m.used - 1, every entry is crossed by a
  // rise and holds an index of the haystack.
  auto bucket = [&](int32_t v) {
    const uint32_t k = (order_key(v) - m.umin) >> m.shift;
    return k < m.used ? k : m.used - 1u;
  };
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
      // Entries [first, first + gap) start here; below zero after a bucket
      // above, which the comparisons take for a long gap.
      const uint32_t gap = p < b1 ? b[j] + 1u - first : 0u;
      nwide += p < b1 && p >= kSsWide && b[j - 1] == b[j] ? 1 : 0;
      if (gap <= 8u) {
        for (uint32_t k = 0; k < gap; ++k) start[first + k] = (int32_t)p;
      }
      uint64_t more = __ballot(gap > 8u);
      while (more != 0) {
        const int l = __builtin_ctzll(more);
        more &= more - 1;
        const uint32_t f = (uint32_t)readlane((int)first, l), g = (uint32_t)readlane((int)gap, l);
        if ((int32_t)g <= 0) continue;  // buckets are at most 2^22
        const int32_t at = (int32_t)(w + (j - 1) * kWave) + l;
        if (g > kSsLongGap) {
          int q = 0;
          if (lane == 0) {
            q = atomicAdd(&s_gaps, 1);
            if (q < kSsLongGaps) {
              s_first[q] = f;
              s_last[q] = f + g;
              s_at[q] = at;
            }
          }
          // Rises of a sorted haystack have room for all of theirs.
          if (__builtin_amdgcn_readfirstlane(q) < kSsLongGaps) continue;
        }
        for (uint32_t k = lane; k < g; k += kWave) start[f + k] = at;
      }
    }
  }
  nwide = wave_sum(nwide);
  if (lane == 0 && nwide) atomicAdd(&s_wide, nwide);
  __syncthreads();
  const int gaps = s_gaps < kSsLongGaps ? s_gaps : kSsLongGaps;
  for (int q = 0; q < gaps; ++q) {
    for (uint32_t k = s_first[q] + threadIdx.x; k < s_last[q]; k += kSsThreads) start[k] = s_at[q];
  }
  if (threadIdx.x == 0) {
    if (wide) wide[blockIdx.x] = s_wide;
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

// Needles in input order, kSsU per thread in flight.
__global__ __launch_bounds__(kSsThreads) void searchsorted_indexed_kernel(const int32_t* __restrict__ sorted,
                                                                          int32_t len, int bits,
                                                                          const int32_t* __restrict__ wide,
                                                                          const int32_t* __restrict__ start,
                                                                          const int32_t* __restrict__ values,
                                                                          int32_t* __restrict__ out, int64_t nv) {
  __shared__ int32_t s_tree[kSsNodes];
  const BucketMap m = bucket_map(sorted, len, bits);
  const int64_t stride = (int64_t)gridDim.x * kSsThreads;
  const int64_t first = (int64_t)blockIdx.x * kSsThreads + threadIdx.x;
  if (!wide || bucket_clustered(wide, len, m, s_tree)) {
    __syncthreads();  // the sum has been read
    if (len < kSsNarrowLen) {
      search_staged<kSsU>(s_tree, sorted, len, values, out, nv, [](int32_t, int32_t&, int32_t&) {});
    } else {
      search_staged<kSsU>(s_tree, sorted, len, values, out, nv, [&](int32_t key, int32_t& lo, int32_t& hi) {
        const uint32_t o = order_key(key);
        if (o < m.umin || o > m.umax) return;
        const i32x2u se = *reinterpret_cast<const i32x2u*>(start + ((o - m.umin) >> m.shift));
        lo = lo > se[0] ? lo : se[0];
        hi = hi < se[1] ? hi : se[1];
      });
    }
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

// ---------------------------------------------------------------------------
// Large haystacks with many needles: the needles go to the haystack.  The
// haystack is cut into slices of 16384 samples (every B-th element; B = 1 up
// to 2^24 elements), at most 1024 of them, whose samples fit in LDS as a
// search tree.  Four kernels over batches of at most 1024 tiles of 16384
// needles:
//   split:   a tile's needles, grouped by slice, into its part of `out`, with
//            every needle's place in the tile (16 bits) and the start of
//            every slice's group;
//   columns: a workgroup per slice scans its groups' sizes over the tiles;
//   sweep:   a workgroup per slice, or per share of the needles of one that
//            many need, searches them in LDS and writes the answers in their
//            place;
//   unsplit: a tile's answers back to the needles' order.
// A tile whose needles are all in one slice (needles in order, few values) is
// answered by the split, its groups empty (2^24 needles in order into 2^20
// elements: 163 us through all four kernels, 100 so, 144 by a table of the
// bounds).
// All memory is read and written in runs of a group (64 bytes for 2^24
// elements) or longer, where a search per needle reads a line of the haystack
// and one of a table for each.  Slices hold equal numbers of elements and
// shares equal numbers of needles, whatever the keys.  2^24 needles into 2^24
// elements: 162 us, 172 on inputs that change from call to call (split 47,
// columns 11, sweep 77, unsplit 27 alone; a table searched by groups of 8192
// needles 551).  Split and unsplit run at 3.1 and 5.9
// TB/s; the sweep is bound by its vector instructions (112 a row of 64
// needles, 70% busy) and by the tree's LDS reads (50% busy).
// ---------------------------------------------------------------------------
constexpr int kSwThreads = kSsThreads, kSwRows = 16, kSwTile = kSwThreads * kSwRows;
constexpr int kSwSlices = 1024, kSwSamples = kSsNodes;
// Most needles of a share (us with 10240, 20480 and 40960 at most: 2^24 random
// needles into 2^24 elements 179, 162, 162, clustered ones 173, 166, 173, into 2^22
// 142, 130, 125; 2^23 into 98304 79, 72, 75); and where there are few slices, of a slice with few
// needles left (the split has answered the rest), which would keep one
// compute unit busy and the others waiting (2^22 needles in order into 98305
// elements: sweep 15.7 us, 8.8 so).
constexpr int kSwShare = 20480, kSwFewSlices = 16, kSwFewNeedles = 65536, kSwFewShare = 4096;
__host__ __device__ constexpr int32_t sweep_shares(int32_t needles, int nb) {
  const int32_t share = nb <= kSwFewSlices && needles <= kSwFewNeedles ? kSwFewShare : kSwShare;
  return (needles + share - 1) / share;
}

// Inclusive maximum scan over a wave's lanes of values >= 0.
__device__ __forceinline__ int32_t wave_incl_max(int32_t v) {
  v = max(v, dpp_mov<kRowShr1>(v));
  v = max(v, dpp_mov<kRowShr2>(v));
  v = max(v, dpp_mov<kRowShr4>(v));
  v = max(v, dpp_mov<kRowShr8>(v));
  v = max(v, dpp_mov<kRowBcast15, 0xa>(v));
  return max(v, dpp_mov<kRowBcast31, 0xc>(v));
}

// Exclusive scan of one value per thread over a workgroup of kSwThreads, and
// the total; s_w holds a word per wave.  Ends with a barrier.
__device__ __forceinline__ int32_t sw_block_scan(int32_t v, int32_t* s_w, int32_t* total) {
  constexpr int W = kSwThreads / kWave;
  const int lane = __lane_id(), wid = threadIdx.x / kWave;
  const int32_t incl = wave_incl_scan(v);
  if (lane == kWave - 1) s_w[wid] = incl;
  __syncthreads();
  int32_t before = incl - v, all = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    before += w < wid ? s_w[w] : 0;
    all += s_w[w];
  }
  *total = all;
  __syncthreads();
  return before;
}

// The lower bound of a key of the slice from element e0 that c samples lie
// below: with B = 1, no more than the samples (c is 0 in slice 0 only),
// otherwise between samples c - 1 and c.
__device__ __forceinline__ int32_t slice_answer(const int32_t* __restrict__ sorted, int32_t len, int32_t B, int64_t e0,
                                                int32_t c, int32_t key) {
  if (B == 1 || c == 0) return (int32_t)e0 + c;
  const int64_t l = e0 + (int64_t)(c - 1) * B + 1;
  const int64_t hi = l + B - 1 < len ? l + B - 1 : len;
  return lower_bound_in(sorted, (int32_t)l, (int32_t)(hi - l), key);
}

__global__ __launch_bounds__(kSwThreads) __attribute__((amdgpu_waves_per_eu(8))) void searchsorted_split_kernel(
    const int32_t* __restrict__ sorted, int64_t slice, int nb, int log, const int32_t* values, int32_t* out,
    int64_t nv, uint16_t* __restrict__ pos, uint16_t* __restrict__ start, int32_t len, int32_t B) {
  __shared__ int32_t s_key[kSwTile];  // or the samples of the one slice that all needles are in
  __shared__ int32_t s_tree[kSwSlices];
  __shared__ int32_t s_cnt[kSwSlices + 1];
  __shared__ int32_t s_w[kSwThreads / kWave];
  __shared__ int32_t s_one;
  const int tid = threadIdx.x;
  stage_tree(s_tree, log, sorted + slice, slice, nb - 1);
  const int64_t t0 = (int64_t)blockIdx.x * kSwTile;
  const int tvalid = t0 + kSwTile <= nv ? kSwTile : (int)(nv - t0);
  values += t0;
  out += t0;
  pos += t0;
  s_cnt[tid] = 0;
  if (tid == 0) {
    s_cnt[kSwSlices] = 0;
    s_one = -1;
  }
  int32_t key[kSwRows], br[kSwRows];  // slice << 16 | rank in it (in no particular order)
#pragma unroll
  for (int i = 0; i < kSwRows; ++i) {
    const int p = i * kSwThreads + tid;
    key[i] = values[p < tvalid ? p : tvalid - 1];
  }
  int again = tid;  // places are found anew in each phase, not kept in registers
  asm volatile("" : "+v"(again));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSwRows; i += 4) {
    const int32_t k4[4] = {key[i], key[i + 1], key[i + 2], key[i + 3]};
    int32_t c4[4];
    tree_count<4>(s_tree, log, k4, c4);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      // Rows past the end count in a word of their own.
      const int32_t b = (i + u) * kSwThreads + again < tvalid ? c4[u] : kSwSlices;
      // A wave whose needles are in one slice (needles in order) counts them
      // with one add: 64 to one word follow one another.
      const int32_t b0 = __builtin_amdgcn_readfirstlane(b);
      if (__ballot(b != b0) == 0) {
        int32_t at = 0;
        if (__lane_id() == 0) at = atomicAdd(&s_cnt[b0], kWave);
        br[i + u] = b << 16 | (__builtin_amdgcn_readfirstlane(at) + (int32_t)__lane_id());
      } else {
        br[i + u] = b << 16 | atomicAdd(&s_cnt[b], 1);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  int32_t all;
  if (s_cnt[tid] == tvalid) s_one = tid;
  const int32_t first = sw_block_scan(s_cnt[tid], s_w, &all);
  if (s_one >= 0) {
    // All needles in one slice (needles in order, or few values): answered
    // here, the slice's samples in the place of the needles.  The tile's groups
    // are empty, starting at its end, which unsplit knows it by.
    if (tid < nb) start[(int64_t)blockIdx.x * nb + tid] = (uint16_t)tvalid;
    const int64_t e0 = (int64_t)s_one * slice, rest = (len - e0 + B - 1) / B;
    stage_tree(s_key, kSsLog, sorted + e0 + B, B, (int32_t)(rest < kSwSamples ? rest : kSwSamples) - 1);
    const int32_t least = sorted[e0];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSwRows; i += 4) {
      const int32_t k4[4] = {key[i], key[i + 1], key[i + 2], key[i + 3]};
      int32_t c4[4];
      tree_count<4>(s_key, kSsLog, k4, c4);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int32_t lo = slice_answer(sorted, len, B, e0, c4[u] + (least < k4[u] ? 1 : 0), k4[u]);
        const int p = (i + u) * kSwThreads + tid;
        if (p < tvalid) out[p] = lo;
      }
    }
    return;
  }
  s_cnt[tid] = first;
  if (tid == 0) s_cnt[kSwSlices] = tvalid;
  if (tid < nb) start[(int64_t)blockIdx.x * nb + tid] = (uint16_t)first;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSwRows; ++i) {
    br[i] = s_cnt[br[i] >> 16] + (br[i] & 0xffff);
    s_key[br[i]] = key[i];
    if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  asm volatile("" : "+v"(again));
#pragma unroll
  for (int i = 0; i < kSwRows; ++i) {
    const int p = i * kSwThreads + again;
    if (p < tvalid) {
      pos[p] = (uint16_t)br[i];
      out[p] = s_key[p];
    }
    if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
}

// groups[slice][tile] = {needles of the slice in earlier tiles, place of the
// group in `out` less that}; total[slice].
__global__ __launch_bounds__(kSwThreads) void searchsorted_columns_kernel(const uint16_t* __restrict__ start, int nb,
                                                                          int nt, int64_t nv,
                                                                          i32x2u* __restrict__ groups,
                                                                          int32_t* __restrict__ total) {
  __shared__ int32_t s_w[kSwThreads / kWave];
  const int t = threadIdx.x, b = blockIdx.x;
  int32_t s = 0, e = 0;
  if (t < nt) {
    const int64_t left = nv - (int64_t)t * kSwTile;
    s = start[(int64_t)t * nb + b];
    e = b + 1 < nb ? start[(int64_t)t * nb + b + 1] : (left < kSwTile ? (int)left : kSwTile);
  }
  int32_t all;
  const int32_t before = sw_block_scan(e - s, s_w, &all);
  if (t < nt) groups[(int64_t)b * nt + t] = i32x2u{before, t * kSwTile + s - before};
  if (t == 0) total[b] = all;
}

__global__ __launch_bounds__(kSwThreads) __attribute__((amdgpu_waves_per_eu(8))) void searchsorted_sweep_kernel(
    const int32_t* __restrict__ sorted, int32_t len, int32_t B, int nb, int nt, const i32x2u* __restrict__ groups,
    const int32_t* __restrict__ total, int32_t* __restrict__ out) {
  constexpr int W = kSwThreads / kWave, U = 4;
  __shared__ int32_t s_tree[kSwSamples];
  __shared__ int32_t s_before[kSwThreads + 1];  // needles of the slice in earlier tiles
  __shared__ int32_t s_at[kSwThreads];      // place of the tile's group less that
  __shared__ uint8_t s_own[W][U * kWave] __attribute__((aligned(4)));
  __shared__ int32_t s_w[W];
  __shared__ int32_t s_first[W];
  __shared__ int32_t s_slice, s_share, s_shares;
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  if (tid == 0) s_shares = 0;
  const int32_t tot = tid < nb ? total[tid] : 0;
  const int32_t shares = sweep_shares(tot, nb);
  int32_t all;
  const int32_t before = sw_block_scan(shares, s_w, &all);
  const int32_t me = (int32_t)blockIdx.x - before;
  if (me >= 0 && me < shares) {
    s_slice = tid;
    s_share = me;
    s_shares = shares;
    s_w[0] = tot;
  }
  __syncthreads();
  if (s_shares == 0) return;
  const int b = s_slice;
  const int32_t btot = s_w[0];
  const int32_t j0 = (int32_t)((int64_t)btot * s_share / s_shares);
  const int32_t j1 = (int32_t)((int64_t)btot * (s_share + 1) / s_shares);
  const int32_t per = ((j1 - j0 + W - 1) / W + kWave - 1) / kWave * kWave;  // needles of a wave
  // The slice's samples: 0 apart (only slice 0 has needles that do not exceed
  // it), the rest in the tree.
  const int64_t e0 = (int64_t)b * kSwSamples * B;
  const int64_t rest = (len - e0 + B - 1) / B;
  stage_tree(s_tree, kSsLog, sorted + e0 + B, B, (int32_t)(rest < kSwSamples ? rest : kSwSamples) - 1);
  const int32_t first = sorted[e0];
  // This thread's tile holds the slice's needles [p0, p1).
  int32_t p0 = btot, p1 = btot;
  if (tid < nt) {
    const i32x2u g = groups[(int64_t)b * nt + tid];
    p0 = g[0];
    s_at[tid] = g[1];
    if (tid + 1 < nt) p1 = groups[(int64_t)b * nt + tid + 1][0];
  }
  s_before[tid] = p0;
  if (tid == 0) s_before[kSwThreads] = btot;
  if (p0 < p1) {
    // The tile of each wave's first needle.
    int32_t w = p0 > j0 ? (p0 - j0 + per - 1) / per : 0;
    for (; w < W && j0 + w * per < p1; ++w) s_first[w] = tid;
  }
  __syncthreads();
  const int32_t w0 = j0 + wid * per;
  const int32_t w1 = w0 + per < j1 ? w0 + per : j1;
  if (w0 >= w1) return;
  // Places of the wave's next rows of needles, from `r0` on: up to U rows, and
  // no further than the 64 tiles from `cur` reach (one a lane).  Each tile
  // marks its first needle; the nearest mark at or before a needle names its
  // tile, tile `cur` where there is none.
  int32_t cur = __builtin_amdgcn_readfirstlane(s_first[wid]), r0 = w0;
  uint8_t* own = s_own[wid];
  auto place = [&](int32_t (&at)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) at[u] = -1;
    while (r0 < w1) {
      const int32_t t = cur + lane;
      const int32_t q0 = s_before[t < nt ? t : nt], q1 = s_before[t + 1 < nt ? t + 1 : nt];
      const int32_t reach = readlane(q1, kWave - 1);
      int32_t r1 = w1 < r0 + U * kWave ? w1 : r0 + U * kWave;
      r1 = reach < r1 ? reach : r1;
      if (r1 <= r0) {  // tiles without needles
        cur += kWave;
        continue;
      }
      reinterpret_cast<uint32_t*>(own)[lane] = 0;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (q0 >= r0 && q0 < r1 && q0 < q1) own[q0 - r0] = (uint8_t)lane;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      int32_t m[U];
#pragma unroll
      for (int u = 0; u < U; ++u) m[u] = own[u * kWave + lane];
      int32_t carry = 0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        m[u] = max(wave_incl_max(m[u]), carry);
        carry = readlane(m[u], kWave - 1);
        const int32_t j = r0 + u * kWave + lane;
        const int32_t a = s_at[cur + m[u]] + j;
        at[u] = j < r1 ? a : -1;
      }
      cur += __builtin_popcountll(__ballot(q1 <= r1));
      r0 = r1;
      break;
    }
  };
  int32_t at[U], key[U];
  place(at);
#pragma unroll
  for (int u = 0; u < U; ++u) key[u] = out[at[u] >= 0 ? at[u] : 0];
  for (bool more = true; more;) {
    // The next rows are on their way during the search.
    int32_t nat[U], nkey[U], c[U];
    more = r0 < w1;
    if (more) {
      place(nat);
#pragma unroll
      for (int u = 0; u < U; ++u) nkey[u] = out[nat[u] >= 0 ? nat[u] : 0];
    }
    tree_count<U>(s_tree, kSsLog, key, c);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      c[u] += first < key[u] ? 1 : 0;  // samples below the needle
      const int32_t lo = slice_answer(sorted, len, B, e0, c[u], key[u]);
      if (at[u] >= 0) out[at[u]] = lo;
      if (more) {
        at[u] = nat[u];
        key[u] = nkey[u];
      }
    }
  }
}

__global__ __launch_bounds__(kSwThreads) __attribute__((amdgpu_waves_per_eu(8))) void searchsorted_unsplit_kernel(
    const uint16_t* __restrict__ pos, const uint16_t* __restrict__ start, int nb, int32_t* __restrict__ out, int64_t nv) {
  __shared__ int32_t s_r[kSwTile];
  const int tid = threadIdx.x;
  const int64_t t0 = (int64_t)blockIdx.x * kSwTile;
  const int tvalid = t0 + kSwTile <= nv ? kSwTile : (int)(nv - t0);
  if (start[(int64_t)blockIdx.x * nb] != 0) return;  // the split has answered the tile
  int32_t r[kSwRows];
  uint32_t q[kSwRows];
#pragma unroll
  for (int i = 0; i < kSwRows; ++i) {
    const int p = i * kSwThreads + tid;
    r[i] = out[t0 + (p < tvalid ? p : tvalid - 1)];
    q[i] = pos[t0 + (p < tvalid ? p : tvalid - 1)];
  }
#pragma unroll
  for (int i = 0; i < kSwRows; ++i) {
    const int p = i * kSwThreads + tid;
    if (p < tvalid) s_r[p] = r[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSwRows; ++i) {
    const int p = i * kSwThreads + tid;
    if (p < tvalid) out[t0 + p] = s_r[q[i]];
  }
}

// The sweep from these sizes on; below, its four launches and the slices read
// by workgroups with few needles cost more than a table does (us, table and
// sweep; 65537 elements: 2^22 needles 41 and 50, in order 16 and 37, 2^24 143 and
// 131; 2^18: 2^22 needles 46 and 47, 2^23 83 and 69; 2^20: 2^21 needles 35 and 44,
// 2^22 60 and 48; 2^21: 2^20 32 and 34, 2^21 52 and 44; 2^22 and above: 2^19 27 and
// 27, 2^20 41 and 33).
// From kSwLongLen elements on the sampled search is taken up to one needle for
// kSwLongShare elements (searchsorted_sampled), and the slices beyond.
constexpr int64_t kSwMinLen = (int64_t)1 << 16;
constexpr int64_t kSwLongLen = (int64_t)1 << 25, kSwLongShare = 256;
static int64_t sweep_min_needles(int64_t len) {
  if (len <= (int64_t)3 << 15) return (int64_t)6 << 20;
  if (len <= (int64_t)1 << 20) return (int64_t)3 << 20;
  if (len > kSwLongLen) return len / kSwLongShare;
  return len <= (int64_t)1 << 21 ? (int64_t)1 << 20 : (int64_t)1 << 19;
}

// Slices, elements between samples, and the scratch of a batch of nt tiles:
// groups, slice totals, group starts, places.
struct SweepLayout {
  int32_t B;
  int nb, log;
  size_t total, start, pos, end;
};

static SweepLayout sweep_layout(int64_t len, int64_t nt) {
  SweepLayout l;
  l.B = (int32_t)((len + (int64_t)kSwSamples * kSwSlices - 1) / ((int64_t)kSwSamples * kSwSlices));
  const int64_t slice = (int64_t)kSwSamples * l.B;
  l.nb = (int)((len + slice - 1) / slice);
  l.log = 0;
  while ((1 << l.log) < l.nb) ++l.log;
  l.total = (size_t)l.nb * nt * sizeof(i32x2u);
  l.start = l.total + (size_t)l.nb * sizeof(int32_t);
  l.pos = l.start + ((size_t)l.nb * nt * sizeof(uint16_t) + 15) / 16 * 16;
  l.end = l.pos + (size_t)nt * kSwTile * sizeof(uint16_t);
  return l;
}

// Tiles of a batch in `bytes` of scratch; 0 where the sweep does not pay:
// each batch reads the haystack, so it wants 256 tiles (or all there are).
static int64_t sweep_tiles(int64_t len, int64_t nv, size_t bytes) {
  if (len <= kSwMinLen || nv <= sweep_min_needles(len)) return 0;
  const int64_t all = (nv + kSwTile - 1) / kSwTile;
  int64_t nt = all < kSwThreads ? all : kSwThreads;
  const int64_t least = nt < 256 ? nt : 256;
  const SweepLayout one = sweep_layout(len, 1), two = sweep_layout(len, 2);
  const size_t per_tile = two.end - one.end + 16;
  if (sweep_layout(len, nt).end > bytes) nt = bytes > one.end ? (int64_t)((bytes - one.end) / per_tile) : 0;
  return nt >= least ? nt : 0;
}

// Whether the needles are too few to pay for staging samples in every
// workgroup, or for a table.  us, sixteen lanes and the other way: 2^16 needles
// into 2^16 elements 7.4 and 9.1 sampled, 2^17 needles 12.2 and 9.2; 2^16 into
// 2^18 9.9 and 10.0 by a table, 8.7 and 17.2 where the elements are clustered;
// into 2^21 16.9 and 13.1, clustered 12.9 and 33; into 2^24 28 and 30.  A
// needle's fifteen lines a step are the more, the less of the haystack the
// caches hold: 2^15 into 5e7 elements 26.6 and 30.8 sampled, 2^16 49 and 31; 2^15
// into 2e8 42 and 32.
static bool searchsorted_few(int64_t len, int64_t nv) {
  const int64_t k = (int64_t)1 << 13;
  return nv <= (len <= (int64_t)1 << 24 ? 8 * k : len <= (int64_t)1 << 26 ? 5 * k : len <= (int64_t)1 << 27 ? 4 * k : 2 * k);
}

// Whether the sampled search is taken where there is a workspace too: few
// needles into a haystack not much longer than the samples (2^18 into 65537
// elements 8.4 us, 9.6 by a table), and haystacks that cost more to read, for
// a table or by slices, than their needles to search (us, sampled, by a
// table, by slices; 2^18 needles into 5e7 elements 61, 75, 58, clustered 51, 121,
// 50; 2^18 into 1.3e8 70, 195, 136; 2^19 into 2e8 135, 307, 181, 2^20 239, 337,
// 198).
static bool searchsorted_sampled(int64_t len, int64_t nv) {
  if (len <= kSsNodes || (len <= (int64_t)3 << 15 && nv <= (int64_t)1 << 18)) return true;
  return len > kSwLongLen && nv <= len / kSwLongShare;
}

// Workgroups for `rows` rows of kSsThreads needles: one for each CU of the
// current device first, then kSsU needles a thread before more of them, up to
// the two a CU that are resident with 64 KiB of LDS each, since every workgroup
// of the sampled search stages the samples (2^20 needles into 2^14 elements:
// 16.4 us with one needle a thread, 7.4 with four; 2^20 into 2^20 clustered
// elements, by the table's sampled search: 99 and 49; 2^24 into 2^18: 297 us
// with four workgroups a CU, 283 with two).
// The sampled search of many needles with reads past the samples takes four a
// CU, which even out the tail (2^24 into 16385 elements: 60 us with two, 56).
static uint32_t searchsorted_grid(uint64_t rows, bool reads) {
  static std::atomic<int> cached[kMaxCachedDevices];
  const uint64_t cus = (uint64_t)device_cached(cached, [](int dev) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    return n;
  });
  const uint64_t few = rows < cus ? rows : cus, need = (rows + kSsU - 1) / kSsU;
  const uint64_t cap = reads && need >= 16 * cus ? 4 * cus : 2 * cus;
  return (uint32_t)(need < few ? few : (need < cap ? need : cap));
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
  // While no thread has more than one needle, one in flight: the steps of
  // three copies of it would be LDS reads as well (2^18 needles into 2^14: 7.1
  // us with four, 5.9 with one; 2^19 7.1 and 7.9).
  const uint64_t rows = (uint64_t)((num_values + kSsThreads - 1) / kSsThreads);
  const uint32_t blocks = searchsorted_grid(rows, sorted_len > kSsNodes);
  hipLaunchKernelGGL(blocks == rows ? searchsorted_kernel<1> : searchsorted_kernel<kSsU>, dim3(blocks),
                     dim3(kSsThreads), 0, static_cast<hipStream_t>(stream), sorted, (int32_t)sorted_len, values, out,
                     num_values);
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

size_t tcs_searchsorted_preferred_bytes(int64_t sorted_len, int64_t num_values) {
  using namespace tcs;
  if (sorted_len <= 0) return 0;
  const int64_t nt = sweep_tiles(sorted_len, num_values, SIZE_MAX);
  const size_t least = tcs_searchsorted_workspace_bytes(sorted_len);
  if (searchsorted_few(sorted_len, num_values) || searchsorted_sampled(sorted_len, num_values)) return least;
  if (nt > 0) {
    const size_t sweep = sweep_layout(sorted_len, nt).end;
    return sweep > least ? sweep : least;
  }
  return (kSsBuildBlocks + ((size_t)1 << bucket_bits(sorted_len)) + 1) * sizeof(int32_t);
}

static int sweep_batch(const int32_t* sorted, int64_t len, const int32_t* values, int32_t* out, int64_t nv,
                       void* workspace, hipStream_t st) {
  using namespace tcs;
  const int64_t nt = (nv + kSwTile - 1) / kSwTile;
  const SweepLayout l = sweep_layout(len, nt);
  char* w = static_cast<char*>(workspace);
  auto* groups = reinterpret_cast<i32x2u*>(w);
  auto* total = reinterpret_cast<int32_t*>(w + l.total);
  auto* start = reinterpret_cast<uint16_t*>(w + l.start);
  auto* pos = reinterpret_cast<uint16_t*>(w + l.pos);
  hipLaunchKernelGGL(searchsorted_split_kernel, dim3((uint32_t)nt), dim3(kSwThreads), 0, st, sorted,
                     (int64_t)kSwSamples * l.B, l.nb, l.log, values, out, nv, pos, start, (int32_t)len, l.B);
  TCS_CHECK_LAUNCH();
  hipLaunchKernelGGL(searchsorted_columns_kernel, dim3(l.nb), dim3(kSwThreads), 0, st, start, l.nb, (int)nt, nv, groups,
                     total);
  TCS_CHECK_LAUNCH();
  // At most one share more than full ones for each slice, and those of a slice
  // with few needles.
  const int64_t more = l.nb <= kSwFewSlices ? kSwFewNeedles / kSwFewShare : 1;
  hipLaunchKernelGGL(searchsorted_sweep_kernel, dim3((uint32_t)(l.nb * more + nv / kSwShare)), dim3(kSwThreads), 0, st, sorted,
                     (int32_t)len, l.B, l.nb, (int)nt, groups, total, out);
  TCS_CHECK_LAUNCH();
  hipLaunchKernelGGL(searchsorted_unsplit_kernel, dim3((uint32_t)nt), dim3(kSwThreads), 0, st, pos, start, l.nb,
                     out, nv);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

int tcs_searchsorted_indexed(const int32_t* sorted, int64_t sorted_len, const int32_t* values, int32_t* out,
                             int64_t num_values, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace tcs;
  if (sorted_len < 0 || num_values < 0 || sorted_len >= ((int64_t)1 << 31)) return TCS_ERR_INVALID_ARG;
  if (num_values == 0) return TCS_OK;
  if (!values || !out || (sorted_len > 0 && !sorted)) return TCS_ERR_INVALID_ARG;
  if (sorted_len == 0) return tcs_searchsorted(sorted, sorted_len, values, out, num_values, stream);
  if (!workspace || workspace_bytes < tcs_searchsorted_workspace_bytes(sorted_len)) return TCS_ERR_WORKSPACE;
  if (searchsorted_few(sorted_len, num_values) || searchsorted_sampled(sorted_len, num_values))
    return tcs_searchsorted(sorted, sorted_len, values, out, num_values, stream);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t nt = sweep_tiles(sorted_len, num_values, workspace_bytes);
  if (nt > 0) {
    for (int64_t i = 0; i < num_values; i += nt * kSwTile) {
      const int64_t n = num_values - i < nt * kSwTile ? num_values - i : nt * kSwTile;
      if (const int rc = sweep_batch(sorted, sorted_len, values + i, out + i, n, workspace, st)) return rc;
    }
    return TCS_OK;
  }
  // The counts before the table; where they would halve it (the least
  // workspace) and buckets are wide by then, the table alone, every needle
  // by samples and table (2^24 needles into 2^26 elements: 3307 us with the
  // counts, 1703 without; into 2^24, of 32 a bucket: 1023 and 1056).
  const int64_t entries = (int64_t)(workspace_bytes / sizeof(int32_t)) - 1;
  const int most = clamp_int(bucket_bits(sorted_len), 1, floor_log2(entries));
  const int counted = clamp_int(most, 1, floor_log2(entries - kSsBuildBlocks));
  const bool alone = counted < most && sorted_len >= kSsNarrowLen && (sorted_len >> counted) > kSsWide / 2;
  const int bits = alone ? most : counted;
  auto* wide = alone ? nullptr : static_cast<int32_t*>(workspace);
  int32_t* start = static_cast<int32_t*>(workspace) + (alone ? 0 : kSsBuildBlocks);
  const int32_t len = (int32_t)sorted_len;
  const int64_t per_block = (sorted_len + kSsBuildBlocks - 1) / kSsBuildBlocks;
  hipLaunchKernelGGL(bucket_start_kernel, dim3(kSsBuildBlocks), dim3(kSsThreads), 0, st, sorted, len, per_block, bits,
                     wide, start);
  TCS_CHECK_LAUNCH();
  hipLaunchKernelGGL(searchsorted_indexed_kernel,
                     dim3(searchsorted_grid((uint64_t)((num_values + kSsThreads - 1) / kSsThreads), false)), dim3(kSsThreads), 0, st,
                     sorted, len, bits, wide, start, values, out, num_values);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

}  // extern "C"
