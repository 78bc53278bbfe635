// Stable LSD radix sort on gfx950 with 8-bit digits, returning the sorted
// values and their original positions (the reference's run_radix_sort,
// src/torch/torch_sort.h:21-81, src/radix_sort.cpp: a 1-bit split per bit,
// 16 passes, after an order-preserving re-encoding of fp16).
//
// Order: torch.sort(stable=True): ascending (or descending) by value, ties in
// input order; floats order -0.0 and +0.0 as equal and every NaN after +inf
// (before everything when descending).  Values move unchanged, so the
// output holds the input's exact bits; the order key is recomputed from
// them in every pass.
//
// The keys are cut into at most kSortMaxChunks contiguous chunks, one
// resident workgroup each.  Every digit position is a count kernel (the 256
// digit counts of each chunk, or of each of a chunk's parts), for many counts
// a kernel that sums them up to each part's first output index per digit,
// and a scatter kernel: a workgroup walks its chunk tile by tile with the
// 256 output indices in registers, ranks a tile's keys by digit, reorders
// the tile in LDS and writes each digit's run contiguously.  There is no
// look-back: no tile waits for another.  At most kSortBlockMax keys are
// sorted by one workgroup in one launch.
#include "tcs_common.hpp"
#include "tcs_device.hpp"
#include "tcs_sortkey.hpp"

namespace tcs {

constexpr int kSortThreads = 512;     // of a count workgroup
constexpr int kSortNW = kSortThreads / kWave;
constexpr int kSortMaxChunks = 512;   // scatter workgroups
constexpr int kSortMaxRows = 1024;    // count workgroups
constexpr int kSortFusedRows = 64;    // up to here the scatter kernel sums the counts itself

// Digit of an order key (or of the order key in the low or high half of a
// pair, with 16 added to the shift).
__device__ __forceinline__ uint32_t sort_digit(uint32_t key, uint32_t shift) {
  return __builtin_amdgcn_ubfe(key, shift, 8);
}

// Order keys of two consecutive rows: the pair of a 16-bit type in one word
// (row 0 in the low half), or the two keys.  Descending order inverts every
// key bit (flip = ~0).
template <int DT>
struct KeyPair {
  using KT = SortKey<DT>;
  static constexpr bool kPacked = KT::kBits == 16;
  uint32_t k[kPacked ? 1 : 2];
  __device__ __forceinline__ void set(uint32_t r0, uint32_t r1, uint32_t flip) {
    if constexpr (kPacked) {
      k[0] = KT::pair(r0 | (r1 << 16)) ^ flip;
    } else {
      k[0] = KT::key((typename KT::Raw)r0) ^ flip;
      k[1] = KT::key((typename KT::Raw)r1) ^ flip;
    }
  }
  __device__ __forceinline__ uint32_t word(int h) const { return kPacked ? k[0] : k[h]; }
  __device__ __forceinline__ uint32_t shift(uint32_t s, int h) const { return kPacked ? s + 16u * (uint32_t)h : s; }
};

// N values of `BITS` bits, 16-bit ones two to a register.
template <int N, int BITS>
struct RowRegs {
  static constexpr bool kPacked = BITS <= 16;
  uint32_t w[kPacked ? N / 2 : N];
  // Sets rows i and i + 1 (i even).
  __device__ __forceinline__ void set2(int i, uint32_t a, uint32_t b) {
    if constexpr (kPacked) {
      w[i / 2] = a | (b << 16);
    } else {
      w[i] = a;
      w[i + 1] = b;
    }
  }
  __device__ __forceinline__ uint32_t get(int i) const {
    if constexpr (kPacked) return i % 2 ? w[i / 2] >> 16 : w[i / 2] & 0xffffu;
    else return w[i];
  }
};

// Counts one row into the wave's `hist` and returns the number of keys of
// this lane's digit d that the wave has met before this key (earlier rows,
// then lower lanes).  Eight ballots, one per digit bit from bit `at` of
// `word`, leave in (lo, hi) the lanes of `vmask` with the same digit: a
// sign-extended bit, its ballot and two three-input logic operations a bit.
// A wave's LDS operations execute in order, so the rows' reads and the adds
// of the first lane of each digit follow one another without a wait.
__device__ __forceinline__ uint32_t sort_rank_row(uint32_t* hist, uint32_t word, uint32_t at, uint32_t d,
                                                  bool valid, uint64_t vmask) {
  uint32_t lo = (uint32_t)vmask, hi = (uint32_t)(vmask >> 32);
#pragma unroll
  for (uint32_t b = 0; b < 8; ++b) {
    const int s = __builtin_amdgcn_sbfe((int)word, at + b, 1);
    const uint64_t m = __ballot(s != 0);
    lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)m, (uint32_t)s, 0x90);          // lo & ~(m ^ s)
    hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(m >> 32), (uint32_t)s, 0x90);
  }
  const uint32_t rank = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
  uint32_t base = 0;
  if (valid) {
    base = __hip_atomic_load(&hist[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    if (rank == 0)
      (void)__hip_atomic_fetch_add(&hist[d], (uint32_t)(__builtin_popcount(lo) + __builtin_popcount(hi)),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
  return base + rank;
}

// ---------------------------------------------------------------------------
// Digit counts: counts[r * 256 + d] = keys of digit d among the `part` keys
// from r * part.  Per
// wave C copies of the 256 bins, lane l adding into copy l % C: lanes whose
// keys share a digit (skewed data) then contend C times less.  Bound by the
// read: 2^26 int32 keys 45 us (5.9 TB/s) in the first pass; the later passes'
// counts take about 95 us, since reading what the scatter before them wrote
// makes room in the last-level cache for which that write has to drain.
// ---------------------------------------------------------------------------
template <int DT, int C>
__global__ __launch_bounds__(kSortThreads) void sort_count_kernel(const typename SortKey<DT>::Raw* __restrict__ x,
                                                                  int64_t n, int64_t part, uint32_t shift,
                                                                  uint32_t flip, uint32_t* __restrict__ counts) {
  using Raw = typename SortKey<DT>::Raw;
  constexpr int V = 16 / (int)sizeof(Raw);
  constexpr int NH = kSortNW * C;
  // One word of padding per copy: the copies of one bin fall in different
  // LDS banks.
  __shared__ uint32_t h[NH][257];
  const int tid = threadIdx.x, wid = tid / kWave;
  for (int k = tid; k < NH * 257; k += kSortThreads) (&h[0][0])[k] = 0;
  uint32_t* hc = h[wid * C + (__lane_id() % C)];
  __syncthreads();
  const int64_t c0 = (int64_t)blockIdx.x * part;
  const int64_t c1 = c0 + part < n ? c0 + part : n;
  // Four 16-byte loads in flight per thread per step; steps that lie wholly
  // inside the chunk skip the per-element bounds checks.
  constexpr int U = 4;
  constexpr int64_t STEP = (int64_t)kSortThreads * V;
  auto add = [&](const Raw(&r)[V], auto all, int64_t left) {
    constexpr bool ALL = decltype(all)::value;
#pragma unroll
    for (int i = 0; i < V; i += 2) {
      KeyPair<DT> kp;
      kp.set(r[i], r[i + 1], flip);
#pragma unroll
      for (int e = 0; e < 2; ++e)
        if (ALL || i + e < left) atomicAdd(&hc[sort_digit(kp.word(e), kp.shift(shift, e))], 1u);
    }
  };
  int64_t b0 = c0 + (int64_t)tid * V;
  const int64_t full_end = c0 + ((c1 - c0) / (U * STEP)) * (U * STEP);  // steps [c0, full_end) are whole
  for (; b0 < full_end; b0 += U * STEP) {
    Raw r[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u) load_items<Raw, V, true>(x, b0 + u * STEP, c1, r[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) add(r[u], std::integral_constant<bool, true>{}, V);
  }
  for (; b0 < c1; b0 += STEP) {
    Raw r[V];
    load_items<Raw, V, false>(x, b0, c1, r);
    add(r, std::integral_constant<bool, false>{}, c1 - b0);
  }
  __syncthreads();
  if (tid < 256) {
    uint32_t s = 0;
#pragma unroll
    for (int w = 0; w < NH; ++w) s += h[w][tid];
    counts[(size_t)blockIdx.x * 256 + tid] = s;
  }
}

// In place: counts[r * 256 + d] = keys of digit d in the rows before r, and
// totals[d] = keys of digit d.  A workgroup takes 16 digits; its threads are
// 64 groups of kSortMaxRows / 64 consecutive rows.
constexpr int kSortScanThreads = 1024, kSortScanDigits = 16;
__global__ __launch_bounds__(kSortScanThreads) void sort_row_scan_kernel(uint32_t* __restrict__ counts, int rows,
                                                                           uint32_t* __restrict__ totals) {
  constexpr int NG = kSortScanThreads / kSortScanDigits, PER = kSortMaxRows / NG;
  __shared__ uint32_t s_sum[kSortScanDigits][NG + 1];
  const int q = threadIdx.x % kSortScanDigits, g = threadIdx.x / kSortScanDigits;
  const int d = blockIdx.x * kSortScanDigits + q;
  uint32_t v[PER], sum = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) v[i] = g * PER + i < rows ? counts[(size_t)(g * PER + i) * 256 + d] : 0u;
#pragma unroll
  for (int i = 0; i < PER; ++i) sum += v[i];
  s_sum[q][g] = sum;
  __syncthreads();
  // Wave w scans digit w's 64 group sums.
  const int w = threadIdx.x / kWave, lane = __lane_id();
  const uint32_t mine = s_sum[w][lane];
  const uint32_t incl = wave_incl_scan(mine);
  s_sum[w][lane] = incl - mine;
  if (lane == kWave - 1) totals[blockIdx.x * kSortScanDigits + w] = incl;
  __syncthreads();
  uint32_t run = s_sum[q][g];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (g * PER + i < rows) counts[(size_t)(g * PER + i) * 256 + d] = run;
    run += v[i];
  }
}

// ---------------------------------------------------------------------------
// One digit position.  Workgroup c walks its chunk in tiles of 64 NW IT keys:
// wave w, row i, lane l is tile element w * 64 IT + i * 64 + l, so the
// (row, lane) order of a wave is the input order (the chunk's last tile
// takes the fewest rows a wave that hold it).  Each wave ranks its rows
// with its own 256 counters; 256 threads turn the counters into tile
// positions and advance the chunk's output indices, which thread d keeps in
// a register; the tile is reordered in LDS and each digit's run written
// contiguously, while the next tile's keys are already being loaded.
//
// GEN: positions are generated (the first pass without given indices); a
// 16-bit key then shares a word with its tile-local position, and the tile
// takes half the LDS.  BIG: 2^30 keys or more, whose outputs 32-bit byte
// offsets do not reach.  LIMIT: the outputs past the first `limit` are not
// written.
//
// Bound by the write requests of the runs and by the ranking: 2^28 fp16
// normals, first pass 0.73 ms and second 0.79 (8-wave workgroups with
// 8192-key tiles 1.07 and 0.92; with their writes made linear 0.66 and 0.70;
// without any write 0.50).  The look-back passes before took 1.34 and 1.25 ms.
// Plain loads: nontemporal ones measured the same.
// ---------------------------------------------------------------------------
template <int DT, bool GEN, int NW, int IT, bool BIG, bool LIMIT>
__global__ __launch_bounds__(NW * kWave, 4) void sort_scatter_kernel(
    const typename SortKey<DT>::Raw* __restrict__ kin, const int32_t* __restrict__ vin,
    typename SortKey<DT>::Raw* __restrict__ kout, int32_t* __restrict__ vout, const uint32_t* __restrict__ counts,
    const uint32_t* __restrict__ totals, int rows, int parts, uint32_t shift, uint32_t flip, int64_t n,
    int64_t chunk, uint32_t limit) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int NT = NW * kWave, TILE = NT * IT;
  constexpr bool kNarrow = KT::kBits <= 16;
  constexpr bool kWord = GEN && kNarrow;  // key and tile-local position in one word
  static_assert(TILE <= 65536 && IT % 2 == 0, "16-bit tile positions, rows in pairs");
  using Item = typename std::conditional<kWord, uint32_t, uint64_t>::type;
  __shared__ uint32_t s_whist[NW][256];  // per wave: digit counts, then the tile position of its first key per digit
  __shared__ uint32_t s_gofs[256];       // output index of tile position 0 for each digit
  __shared__ uint32_t s_wsum[4];
  __shared__ Item s_item[TILE];
  // A word holds no digit beside key and position: the digits beside it, read
  // back instead of the key's order computed again.
  constexpr bool kDig = kWord && TILE < 32768;
  __shared__ uint8_t s_dig[kDig ? TILE : 1];

  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  const int64_t c0 = (int64_t)blockIdx.x * chunk;
  const int64_t c1 = c0 + chunk < n ? c0 + chunk : n;
  uint32_t* whist = s_whist[wid];

  uint32_t kr[IT];
  int32_t vv[GEN ? 1 : IT];
  const uint32_t len = (uint32_t)(c1 - c0);
  const Raw* kc = kin + c0;
  const int32_t* vc = GEN ? nullptr : vin + c0;
  const uint32_t wl = (uint32_t)(wid * (kWave * IT) + lane);  // whole tile: position of the lane's row 0
  // A whole tile's loads share one uniform base and one lane offset.
  auto load = [&](uint32_t t) {
    const char* kt = reinterpret_cast<const char*>(kc + t);
#pragma unroll
    for (int i = 0; i < IT; ++i)
      kr[i] = *reinterpret_cast<const Raw*>(kt + wl * (uint32_t)sizeof(Raw) + i * kWave * sizeof(Raw));
    if constexpr (!GEN) {
      const char* vt = reinterpret_cast<const char*>(vc + t);
#pragma unroll
      for (int i = 0; i < IT; ++i) vv[i] = *reinterpret_cast<const int32_t*>(vt + wl * 4u + i * kWave * 4);
    }
  };
  // The chunk's last tile, when it is not whole, has `part_rows` rows a wave.
  // Loads past the chunk's end take its last key, so that none waits behind
  // a branch.
  auto load_part = [&](uint32_t t, uint32_t part_rows) {
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const uint32_t p = t + (uint32_t)wid * kWave * part_rows + lane + i * kWave;
      const uint32_t q = p < len ? p : len - 1;
      kr[i] = kc[q];
      if constexpr (!GEN) vv[i] = vc[q];
    }
  };
  if (len >= (uint32_t)TILE) load(0);

  // Output index of the chunk's first key of digit tid.
  uint32_t ofs = 0;
  {
    uint32_t total = 0, incl = 0;
    if (tid < 256) {
      if (totals) {
        ofs = counts[(size_t)blockIdx.x * parts * 256 + tid];
        total = totals[tid];
      } else {
        constexpr int U = 16;  // loads in flight
        for (int g0 = 0; g0 < rows; g0 += U) {
          uint32_t v[U];
#pragma unroll
          for (int u = 0; u < U; ++u) v[u] = counts[(size_t)(g0 + u < rows ? g0 + u : 0) * 256 + tid];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            ofs += g0 + u < (int)blockIdx.x * parts ? v[u] : 0u;
            total += g0 + u < rows ? v[u] : 0u;
          }
        }
      }
      incl = wave_incl_scan(total);
      if (lane == kWave - 1) s_wsum[wid] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      for (int w = 0; w < wid; ++w) ofs += s_wsum[w];
      ofs += incl - total;
    }
  }

  auto do_tile = [&](uint32_t t, uint32_t part_rows, auto full_c) {
    constexpr bool FULL = decltype(full_c)::value;
    const int nrows = FULL ? IT : (int)part_rows;
    const uint32_t wt = FULL ? wl : (uint32_t)wid * kWave * part_rows + lane;  // tile position of the lane's row 0
    const int tvalid = FULL ? TILE : (int)(len - t);
    const uint32_t first = (uint32_t)c0 + t;  // input position of the tile
#pragma unroll
    for (int k = 0; k < 256 / kWave; ++k) whist[k * kWave + lane] = 0;
    KeyPair<DT> kp[IT / 2];
    RowRegs<IT, KT::kBits> raw;
    RowRegs<IT, 16> rk;
    uint32_t pr[2];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      if (i % 2 == 0) {
        raw.set2(i, kr[i], kr[i + 1]);
        kp[i / 2].set(kr[i], kr[i + 1], flip);
      }
      const uint32_t word = kp[i / 2].word(i % 2), at = kp[i / 2].shift(shift, i % 2);
      if (FULL || i < nrows) {
        const bool valid = FULL || wt + i * kWave < (uint32_t)tvalid;
        pr[i % 2] = sort_rank_row(whist, word, at, sort_digit(word, at), valid, FULL ? ~0ull : __ballot(valid));
      } else {
        pr[i % 2] = 0;
      }
      if (i % 2 == 1) {
        rk.set2(i - 1, pr[0], pr[1]);
        asm volatile("" : "+v"(rk.w[i / 2]));
      }
    }
    __syncthreads();

    // Thread d: its digit's keys per wave, their tile positions, and the
    // output index that tile position 0 stands for.
    uint32_t before[NW], cnt = 0, incl = 0;
    if (tid < 256) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        before[w] = cnt;
        cnt += s_whist[w][tid];
      }
      incl = wave_incl_scan(cnt);
      if (lane == kWave - 1) s_wsum[wid] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t excl = incl - cnt;
      for (int w = 0; w < wid; ++w) excl += s_wsum[w];
#pragma unroll
      for (int w = 0; w < NW; ++w) s_whist[w][tid] = excl + before[w];
      s_gofs[tid] = ofs - excl;
      ofs += cnt;
    }
    __syncthreads();

    constexpr int RB = 16;  // rows whose tile positions are read at once
    uint32_t pos[RB];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      if (i % RB == 0) {
#pragma unroll
        for (int j = 0; j < RB && j < IT; ++j)
          pos[j] = whist[sort_digit(kp[(i + j) / 2].word(j % 2), kp[(i + j) / 2].shift(shift, j % 2))];
      }
      const uint32_t local = wt + i * kWave;
      if (FULL || (i < nrows && local < (uint32_t)tvalid)) {
        const uint32_t d = sort_digit(kp[i / 2].word(i % 2), kp[i / 2].shift(shift, i % 2));
        const uint32_t p = pos[i % RB] + rk.get(i);
        if constexpr (kWord) {
          s_item[p] = (raw.get(i) << 16) | local;
          if constexpr (kDig) s_dig[p] = (uint8_t)d;
        } else {
          const uint32_t val = GEN ? first + local : (uint32_t)vv[i];
          s_item[p] = ((uint64_t)val << 32) | (kNarrow ? (d << 16) | raw.get(i) : raw.get(i));
        }
      }
    }
    if (FULL && t + 2 * TILE <= len) load(t + TILE);
    __syncthreads();

    auto put = [&](int p, uint32_t d, uint32_t raw, uint32_t val) {
      const uint32_t dst = s_gofs[d] + (uint32_t)p;
      if (LIMIT && dst >= limit) return;
      if constexpr (!BIG) {
        *reinterpret_cast<Raw*>(reinterpret_cast<char*>(kout) + dst * (uint32_t)sizeof(Raw)) = (Raw)raw;
        *reinterpret_cast<int32_t*>(reinterpret_cast<char*>(vout) + dst * 4u) = (int32_t)val;
      } else {
        kout[dst] = (Raw)raw;
        vout[dst] = (int32_t)val;
      }
    };
#pragma unroll
    for (int i = 0; i < IT; i += 2) {
      Item e[2];
      uint32_t d[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int p = (i + h) * NT + tid;
        const bool in = FULL || (i < nrows && p < tvalid);
        e[h] = in ? s_item[p] : Item(0);
        if constexpr (kDig) d[h] = in ? s_dig[p] : 0u;
      }
      if constexpr (!kWord && kNarrow) {
        d[0] = ((uint32_t)e[0] >> 16) & 0xffu;
        d[1] = ((uint32_t)e[1] >> 16) & 0xffu;
      } else if constexpr (!kDig) {
        KeyPair<DT> q;
        if constexpr (kWord) q.set((uint32_t)e[0] >> 16, (uint32_t)e[1] >> 16, flip);
        else q.set((uint32_t)e[0], (uint32_t)e[1], flip);
        d[0] = sort_digit(q.word(0), q.shift(shift, 0));
        d[1] = sort_digit(q.word(1), q.shift(shift, 1));
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int p = (i + h) * NT + tid;
        if (FULL || (i < nrows && p < tvalid)) {
          if constexpr (kWord) {
            put(p, d[h], (uint32_t)e[h] >> 16, first + ((uint32_t)e[h] & 0xffffu));
          } else {
            put(p, d[h], (uint32_t)e[h], (uint32_t)(e[h] >> 32));
          }
        }
      }
    }
  };
  // Everything loaded so far has arrived when the loop starts (vmcnt 0), so
  // that inside it a tile's first use waits for its own loads only, not for
  // the stores issued after them.
  __builtin_amdgcn_s_waitcnt(0x0f70);
  uint32_t t = 0;
  for (; t + TILE <= len; t += TILE) do_tile(t, IT, std::integral_constant<bool, true>{});
  if (t < len) {
    const uint32_t part_rows = (len - t + NT - 1) / NT;
    load_part(t, part_rows);
    do_tile(t, part_rows, std::integral_constant<bool, false>{});
  }
}

// ---------------------------------------------------------------------------
// At most kSortBlockMax keys: every digit position in one workgroup, keys
// and positions in LDS between passes: one launch (3000 fp16 keys 7.5 us, 8000
// int32 keys 21 us; a histogram, two sums and a look-back pass per digit took
// 29 and 53).  Twice as many keys in one workgroup are slower than the
// chunked form (16000 fp16: 22 against 15 us).  Wave w holds elements
// [64 w rows, 64 (w + 1) rows), rows = ceil(n / 1024).
// ---------------------------------------------------------------------------
constexpr int kSortBlockThreads = 1024, kSortBlockIT = 8;
constexpr int64_t kSortBlockMax = (int64_t)kSortBlockThreads * kSortBlockIT;
template <int DT>
__global__ __launch_bounds__(kSortBlockThreads) void sort_block_kernel(
    const typename SortKey<DT>::Raw* __restrict__ x, const int32_t* __restrict__ idx_in,
    typename SortKey<DT>::Raw* __restrict__ out_x, int32_t* __restrict__ out_idx, int n, uint32_t flip,
    int limit) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int NW = kSortBlockThreads / kWave, IT = kSortBlockIT, P = KT::kBits / 8;
  __shared__ uint32_t s_whist[NW][256];
  __shared__ uint32_t s_wsum[4];
  __shared__ uint64_t s_item[kSortBlockMax];
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  const int rows = (n + kSortBlockThreads - 1) / kSortBlockThreads;
  const int wb = wid * rows * kWave + lane;
  uint32_t* whist = s_whist[wid];
  uint32_t kr[IT], vv[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int p = wb + i * kWave;
    const bool valid = i < rows && p < n;
    kr[i] = valid ? (uint32_t)x[p] : 0u;
    vv[i] = valid && idx_in ? (uint32_t)idx_in[p] : (uint32_t)p;
  }
  for (int pass = 0; pass < P; ++pass) {
    const uint32_t shift = 8u * (uint32_t)pass;
#pragma unroll
    for (int k = 0; k < 256 / kWave; ++k) whist[k * kWave + lane] = 0;
    uint32_t dr[IT];  // digit << 16 | rank
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      if (i < rows) {
        const bool valid = wb + i * kWave < n;
        const uint32_t key = KT::key((Raw)kr[i]) ^ flip;
        const uint32_t d = sort_digit(key, shift);
        dr[i] = (d << 16) | sort_rank_row(whist, key, shift, d, valid, __ballot(valid));
      }
    }
    __syncthreads();
    uint32_t before[NW], cnt = 0, incl = 0;
    if (tid < 256) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        before[w] = cnt;
        cnt += s_whist[w][tid];
      }
      incl = wave_incl_scan(cnt);
      if (lane == kWave - 1) s_wsum[wid] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t excl = incl - cnt;
      for (int w = 0; w < wid; ++w) excl += s_wsum[w];
#pragma unroll
      for (int w = 0; w < NW; ++w) s_whist[w][tid] = excl + before[w];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      if (i < rows && wb + i * kWave < n)
        s_item[whist[dr[i] >> 16] + (dr[i] & 0xffffu)] = ((uint64_t)vv[i] << 32) | kr[i];
    }
    __syncthreads();
    if (pass + 1 < P) {
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        if (i < rows && wb + i * kWave < n) {
          const uint64_t e = s_item[wb + i * kWave];
          kr[i] = (uint32_t)e;
          vv[i] = (uint32_t)(e >> 32);
        }
      }
    }
  }
  for (int p = tid; p < limit; p += kSortBlockThreads) {
    const uint64_t e = s_item[p];
    out_x[p] = (Raw)e;
    out_idx[p] = (int32_t)(uint32_t)(e >> 32);
  }
}

// Scratch: one temporary copy of keys and positions, the digit counts and
// their totals (any contents).  The workspace is only its header: no pass
// looks back.
struct SortLayout {
  size_t tmpv_off, counts_off, totals_off, scratch;
  bool wide;            // 16-wave scatter workgroups, else 8-wave ones
  int chunks, parts;    // scatter workgroups, count rows per chunk
  int64_t chunk;
};

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

inline int sort_passes(int dt) {
  switch (dt) {
    case TCS_I8: return 1;
    case TCS_F16: case TCS_BF16: case TCS_I16: return 2;
    case TCS_F32: case TCS_I32: case TCS_U32: return 4;
    default: return 0;
  }
}

inline int sort_elem_bytes(int dt) { return dt == TCS_I8 ? 1 : (sort_passes(dt) == 2 ? 2 : 4); }

// Above kSortWideMin keys the scatter workgroups take 16 waves, and 16384 or
// 32768 keys a tile (the LDS of a whole compute unit), one workgroup on each:
// a tile's runs are then twice or four times as long, and fewer of the lines
// that the 256 runs write are left partial between tiles.  Below it 8-wave
// workgroups with 4096-key tiles, two to a compute unit, divide the keys more
// evenly (fp16 keys, 4e6: 46 against 53 us, 5e6: 56 against 61, 8e6: 73
// either way; int32, 4e6: 101 against 106, 8e6: 176 against 161).
inline SortLayout sort_layout(int64_t n, int dt) {
  SortLayout L{};
  L.wide = n > kSortWideMin;
  const int64_t least = 2048, most = L.wide ? kSortMaxChunks / 2 : kSortMaxChunks, unit = L.wide ? 4096 : 512;
  int64_t chunks = (n + least - 1) / least;
  if (chunks > most) chunks = most;
  if (chunks < 1) chunks = 1;
  L.chunk = ((n + chunks - 1) / chunks + unit - 1) / unit * unit;
  if (L.chunk < unit) L.chunk = unit;
  L.chunks = n > 0 ? (int)((n + L.chunk - 1) / L.chunk) : 1;
  L.parts = 1;
  while (L.wide && L.parts < 4 && L.chunk / L.parts > 16384) L.parts *= 2;
  L.tmpv_off = align256((size_t)n * sort_elem_bytes(dt));
  L.counts_off = align256(L.tmpv_off + (size_t)n * 4);
  // Room for the most rows of counts up to this many keys: rounding chunks
  // up to whole units can leave fewer chunks for more keys, and scratch of a
  // larger n is to serve a smaller one.
  const int64_t rows = L.wide ? (int64_t)kSortMaxRows : (n + least - 1) / least;
  L.totals_off = align256(L.counts_off + (size_t)(rows < most || L.wide ? rows : most) * 256 * 4);
  L.scratch = align256(L.totals_off + 256 * 4);
  return L;
}

template <int DT>
struct SortArgs {
  using Raw = typename SortKey<DT>::Raw;
  const Raw* kin;
  const int32_t* vin;
  Raw* kout;
  int32_t* vout;
  const uint32_t *counts, *totals;
  uint32_t shift, flip;
  int64_t n;
  uint32_t limit;  // outputs of the last pass, n of the others
};

template <int DT, bool GEN, int NW, int IT, bool BIG = false, bool LIMIT = false>
static void sort_scatter_launch(const SortLayout& L, const SortArgs<DT>& a, hipStream_t st) {
  hipLaunchKernelGGL((sort_scatter_kernel<DT, GEN, NW, IT, BIG, LIMIT>), dim3(L.chunks), dim3(NW * kWave), 0, st, a.kin,
                     a.vin, a.kout, a.vout, a.counts, a.totals, L.chunks * L.parts, L.parts, a.shift, a.flip, a.n,
                     L.chunk, a.limit);
}

// A tile as large as the LDS of a compute unit allows for the wide form:
// 32768 16-bit keys whose positions are generated, 16384 others.
template <int DT, bool GEN>
static void sort_scatter(const SortLayout& L, const SortArgs<DT>& a, hipStream_t st) {
  constexpr int IT = GEN && SortKey<DT>::kBits <= 16 ? 32 : 16;
  if (!L.wide && a.limit < a.n) {
    sort_scatter_launch<DT, GEN, 8, 8, false, true>(L, a, st);
  } else if (!L.wide) {
    sort_scatter_launch<DT, GEN, 8, 8>(L, a, st);
  } else if (a.n < ((int64_t)1 << 30)) {
    sort_scatter_launch<DT, GEN, 16, IT>(L, a, st);
  } else {
    sort_scatter_launch<DT, GEN, 16, IT, true>(L, a, st);
  }
}

// The first k outputs to out_x and out_idx; passes before the last alternate
// between scratch and mid_x / mid_idx, of n elements each (out_x and out_idx
// themselves when k == n).  k < n only for keys that do not take the wide
// form.
template <int DT>
static int sort_run(const void* x, const int32_t* idx_in, void* mid_x, int32_t* mid_idx, void* out_x,
                    int32_t* out_idx, int64_t n, int64_t k, bool desc, void* scratch, hipStream_t st) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int P = KT::kBits / 8;
  SortArgs<DT> a{};
  a.flip = desc ? ~0u : 0u;
  a.n = n;
  a.kin = static_cast<const Raw*>(x);
  a.vin = idx_in;
  if (n <= kSortBlockMax) {
    hipLaunchKernelGGL((sort_block_kernel<DT>), dim3(1), dim3(kSortBlockThreads), 0, st, a.kin, idx_in,
                       static_cast<Raw*>(out_x), out_idx, (int)n, a.flip, (int)k);
    TCS_CHECK_LAUNCH();
    return TCS_OK;
  }
  const SortLayout L = sort_layout(n, DT);
  const int rows = L.chunks * L.parts;
  char* sc = static_cast<char*>(scratch);
  auto* counts = reinterpret_cast<uint32_t*>(sc + L.counts_off);
  auto* totals = rows > kSortFusedRows ? reinterpret_cast<uint32_t*>(sc + L.totals_off) : nullptr;
  a.counts = counts;
  a.totals = totals;
  for (int p = 0; p < P; ++p) {
    // The last pass writes the outputs; earlier ones alternate so that it
    // does not read what it writes.
    const bool last = p == P - 1, mid = (P - 1 - p) % 2 == 0;
    a.kout = last ? static_cast<Raw*>(out_x) : (mid ? static_cast<Raw*>(mid_x) : reinterpret_cast<Raw*>(sc));
    a.vout = last ? out_idx : (mid ? mid_idx : reinterpret_cast<int32_t*>(sc + L.tmpv_off));
    a.limit = (uint32_t)(last ? k : n);
    a.shift = 8u * (uint32_t)p;
    if (L.wide) {
      hipLaunchKernelGGL((sort_count_kernel<DT, 4>), dim3(rows), dim3(kSortThreads), 0, st, a.kin, n,
                         L.chunk / L.parts, a.shift, a.flip, counts);
    } else {
      hipLaunchKernelGGL((sort_count_kernel<DT, 1>), dim3(rows), dim3(kSortThreads), 0, st, a.kin, n,
                         L.chunk / L.parts, a.shift, a.flip, counts);
    }
    TCS_CHECK_LAUNCH();
    if (totals) {
      hipLaunchKernelGGL(sort_row_scan_kernel, dim3(256 / kSortScanDigits), dim3(kSortScanThreads), 0, st, counts,
                         rows, totals);
      TCS_CHECK_LAUNCH();
    }
    if (p == 0 && !idx_in) {
      sort_scatter<DT, true>(L, a, st);
    } else {
      sort_scatter<DT, false>(L, a, st);
    }
    TCS_CHECK_LAUNCH();
    a.kin = a.kout;
    a.vin = a.vout;
  }
  return TCS_OK;
}

static int sort_any(const void* x, int dtype, const int32_t* idx_in, void* mid_x, int32_t* mid_idx, void* out_x,
                    int32_t* out_idx, int64_t n, int64_t k, bool desc, void* scratch, hipStream_t st) {
  auto run = [&](auto f) { return f(x, idx_in, mid_x, mid_idx, out_x, out_idx, n, k, desc, scratch, st); };
  switch (dtype) {
    case TCS_F16: return run(sort_run<TCS_F16>);
    case TCS_BF16: return run(sort_run<TCS_BF16>);
    case TCS_F32: return run(sort_run<TCS_F32>);
    case TCS_I8: return run(sort_run<TCS_I8>);
    case TCS_I16: return run(sort_run<TCS_I16>);
    case TCS_I32: return run(sort_run<TCS_I32>);
    default: return run(sort_run<TCS_U32>);
  }
}

// The second temporary copy follows the sort's own scratch.
size_t sort_first_scratch_bytes(int64_t n, int dtype) {
  return sort_layout(n, dtype).scratch + align256((size_t)n * sort_elem_bytes(dtype)) + (size_t)n * 4;
}

int sort_first(const void* x, int dtype, void* out_x, int32_t* out_idx, int64_t n, int64_t k, bool descending,
               void* scratch, hipStream_t st) {
  char* mid = static_cast<char*>(scratch) + sort_layout(n, dtype).scratch;
  if (k < n && n > kSortWideMin) return TCS_ERR_INVALID_ARG;
  return sort_any(x, dtype, nullptr, mid, reinterpret_cast<int32_t*>(mid + align256((size_t)n * sort_elem_bytes(dtype))),
                  out_x, out_idx, n, k, descending, scratch, st);
}

}  // namespace tcs

extern "C" {

size_t tcs_sort_workspace_bytes(int64_t n, int dtype) {
  if (n < 0 || tcs::sort_passes(dtype) == 0) return 0;
  return tcs::lookback_ws_bytes(0);
}

size_t tcs_sort_scratch_bytes(int64_t n, int dtype) {
  if (n < 0 || tcs::sort_passes(dtype) == 0) return 0;
  return tcs::sort_layout(n, dtype).scratch;
}

int tcs_sort(const void* x, int dtype, const int32_t* idx_in, void* out_x, int32_t* out_idx, int64_t n,
             int descending, void* workspace, size_t workspace_bytes, void* scratch, size_t scratch_bytes,
             void* stream) {
  using namespace tcs;
  if (sort_passes(dtype) == 0) return TCS_ERR_UNSUPPORTED_DTYPE;
  if (n < 0 || n >= ((int64_t)1 << 31)) return TCS_ERR_INVALID_ARG;
  if (n == 0) return TCS_OK;
  if (!x || !out_x || !out_idx) return TCS_ERR_INVALID_ARG;
  if (!aligned16(x) || (idx_in && !aligned16(idx_in))) return TCS_ERR_INVALID_ARG;
  const SortLayout L = sort_layout(n, dtype);
  if (!workspace || workspace_bytes < lookback_ws_bytes(0) || !scratch || scratch_bytes < L.scratch) return TCS_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return sort_any(x, dtype, idx_in, out_x, out_idx, out_x, out_idx, n, n, descending != 0, scratch, st);
}

}  // extern "C"
