// Top-k on gfx950 by radix select, and the reference's sampled estimator
// of the k-th largest value.
//
// tcs_topk replaces run_topk_fp16 / run_topk_int16 (src/torch/torch_topk.h:
// 69-207; the reference narrows [x_min, x_max] with parallel splits).  By
// size (topk_run):
//
// Few keys: the radix sort, whose last pass writes the first k only.
//
// Many keys, k <= kTkRankMax: one pass over the keys keeps the largest order
// key of every sub-chunk and of every group of sub-chunks.  The k-th largest
// group maximum, ties to the lowest sub-chunk, bounds the k-th key from below
// (k groups each hold a key at or above it), so only the sub-chunks whose
// maximum reaches it are read again, and their keys at or above it, about
// 1.15 k of them when the keys are in no particular order, are ranked by
// counting.  If they do not fit (the largest keys lie together), the radix
// select below runs instead, over the sub-chunks that reach the bound: its
// kernels are launched behind this path and leave at once when it has
// succeeded, so nothing waits for the host.  2^28 fp16 normals, k = 2048: 124
// us, of which the read takes 82, the select's two reads and eleven launches
// 278; sorted keys, which give too many candidates, 183 against 429 (2^25 of
// them 89 against 116; fp32 112 against 157).
//
// Otherwise radix select: the k-th largest order key T is found one 8-bit
// digit at a time, from the top: a histogram of digit r over the keys whose
// higher digits equal the digits chosen so far, then one workgroup picks the
// bin holding the k-th largest.  State passes between launches in the
// workspace, so no result reaches the host until the end.  An ordered
// selection then takes every key above T and the first `need` keys equal to
// T in input order (per-tile counts, their scan, and placement by the tiles
// that hold any of them), and those k are ranked by counting or, when they
// are many, by the radix sort (ties by input position).  The per-tile counts
// of keys of two or more bytes come from a record the last digit round keeps
// (keys above the higher digits, low bytes of the few matching them), so
// reads are one pass per key byte plus the tiles that hold selected keys
// (one-byte keys: one more pass for the tile counts).
//
// tcs_topk_pivot follows run_topk_pivot_fp16 (src/torch/torch_topk.h:
// 23-60, src/kernels/kernel_topk_pivot.h): per block, over its first eight
// tiles of num_samples * 32 elements, the 8th largest of each 32, then the
// 4th largest of those per tile, then the largest over the tiles.  At least
// 32 elements of the tile are >= that estimate.
#include "tcs_common.hpp"
#include "tcs_device.hpp"
#include "tcs_sortkey.hpp"

namespace tcs {

constexpr int kTkThreads = 512, kTkMaxGroups = 1024, kTkPickThreads = 1024;
constexpr int kTkNW = 8, kTkG = 8;

template <int DT>
struct TopkGeom {
  using Raw = typename SortKey<DT>::Raw;
  static constexpr int J = sizeof(Raw) <= 2 ? 4 : 2;
  static constexpr int64_t kTile = (int64_t)kTkNW * J * kWave * kTkG;
};
constexpr int64_t kTkTileMin = (int64_t)kTkNW * 2 * kWave * kTkG;  // 8192

// The last digit round of a key of two or more bytes also records, per tile
// (one unrolled step of a histogram workgroup covers one tile), the number
// of keys whose higher digits are above the chosen ones and the low bytes of
// up to kTkListMax keys whose higher digits equal them.  Once the last digit
// is chosen, each tile's counts above and at the threshold follow from that
// record without reading the keys again; a tile with more matching keys than
// were recorded is counted from its keys (topk_tilefix_kernel).
constexpr int kTkListMax = 16;
// Placement reads only the sub-chunks of a tile that hold selected keys
// (their record's mask bits): a selected key is above or matches the
// higher digits.
constexpr int64_t kTkSubChunk = 2048;
// Tiles of a histogram workgroup, in a chunk of whole tiles or (behind a gate)
// apart: at most ceil(n / kTkMaxGroups) <= 2^21 keys for n < 2^31, so 256 of 8192.
constexpr int kTkMaxChunkTiles = 256;

inline int64_t topk_tile(int key_bytes) { return (int64_t)kTkNW * (key_bytes <= 2 ? 4 : 2) * kWave * kTkG; }

// The kernels of the radix select take `gate`: null, or the candidate count
// of the maxima path, which has succeeded when the count fits.
constexpr uint32_t kTkCandMax = 8192;  // 64 KiB of LDS
// Words of the maxima path's state: candidates, the bound's T and P, arrivals
// and digit counts of the gated launches.
constexpr int kTkArrived = 8, kTkBins = 64, kTkStateWords = kTkBins + 256;
// Workgroups of a gated launch: one a CU, so that few arrive at one word (2^25
// sorted fp32 keys, k = 2048: 112 us with 256, 118 with 512 or 1024; the select
// before it, with a range of keys a workgroup and every workgroup's digit counts
// read by the last, 225).
constexpr uint32_t kTkGatedGroups = 256;
__device__ __forceinline__ bool topk_done(const uint32_t* gate) { return gate && *gate <= kTkCandMax; }

// Behind a gate the last workgroup of a launch also runs the small step that
// follows (a launch that leaves at once still takes about 4 us in the
// stream).  What the workgroups leave for it they write, and it reads, with
// device-scope accesses, which need no fence (a fence in every workgroup
// writes back and invalidates the L2s: 2^28 keys, 1300 us); a workgroup
// arrives when its own writes have left.  `arrived` is zero at the launch's
// start and again after it.
__device__ __forceinline__ bool topk_last_arrival(uint32_t* arrived) {
  __shared__ uint32_t s_ticket;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    s_ticket = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (s_ticket == gridDim.x - 1) __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return s_ticket == gridDim.x - 1;
}
template <bool SHARED>
__device__ __forceinline__ uint64_t topk_read(const uint64_t* p) {
  return SHARED ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
}
__device__ __forceinline__ void topk_leave(uint64_t* p, uint64_t v, bool shared) {
  if (shared) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    *p = v;
  }
}

// Picks digit r of the k-th largest key: the bin b where the count of keys
// in bins >= b first reaches the number still to take.  One workgroup of NT
// threads; count(d, q, nq) is thread q's share of digit d's keys, of nq threads
// a digit.
template <int NT, class F>
__device__ __forceinline__ void topk_pick(F count, int r, int first, int64_t k, uint64_t* state) {
  constexpr int NQ = NT / 256;
  const int tid = threadIdx.x, d = tid & 255, q = tid >> 8;
  const uint32_t s = count(d, q, NQ);
  __shared__ uint32_t sr[NQ][256];
  __shared__ uint32_t ws[4];
  __shared__ uint64_t s_state[2];
  sr[q][d] = s;
  if (tid == 0) {
    s_state[0] = first ? 0 : state[0];
    s_state[1] = first ? (uint64_t)k : state[1];
  }
  __syncthreads();
  // suffix[b] = keys in bins >= b: an inclusive scan over b' = 255 - b.
  uint32_t cnt = 0, incl = 0;
  if (tid < 256) {
#pragma unroll
    for (int e = 0; e < NQ; ++e) cnt += sr[e][255 - tid];
    incl = wave_incl_scan(cnt);
    if (__lane_id() == kWave - 1) ws[tid / kWave] = incl;
  }
  __syncthreads();
  if (tid < 256) {
    uint32_t before = 0;
    for (int w = 0; w < tid / kWave; ++w) before += ws[w];
    const uint64_t suffix = before + incl;  // keys in bins >= 255 - tid
    const uint64_t need = s_state[1];
    if (suffix >= need && suffix - cnt < need) {
      const uint32_t b = 255u - (uint32_t)tid;
      state[0] = s_state[0] | ((uint64_t)b << (8 * r));
      state[1] = need - (suffix - cnt);
    }
  }
}

// ---------------------------------------------------------------------------
// Digit histogram among the keys matching the chosen higher digits.
// state[0]: key digits chosen so far; state[1]: how many of the keys
// matching them are still to be taken.  64-bit words, high half zero.
// ---------------------------------------------------------------------------
// FUSE (the last round, r = 0, of keys of two or more bytes): also record
// per tile the keys above the chosen higher digits, which of its
// kTkSubChunk-key sub-chunks hold any key above or matching them, and the
// low bytes of up to kTkListMax keys matching them: tstat[tile] = above <<
// 32 | sub-chunk mask << 16 | matching, tlist[tile * kTkListMax + j] = low
// byte (any order).
template <int DT, bool FUSE>
__global__ __launch_bounds__(kTkThreads) void topk_hist_kernel(const typename SortKey<DT>::Raw* __restrict__ x,
                                                               int64_t n, int64_t chunk, uint32_t flip, int r,
                                                               int64_t k_all, uint64_t* state, uint64_t* partial,
                                                               uint64_t* __restrict__ tstat,
                                                               uint8_t* __restrict__ tlist,
                                                               const uint32_t* __restrict__ gate,
                                                               uint32_t* __restrict__ arrived,
                                                               uint32_t* __restrict__ bins,
                                                               const uint32_t* __restrict__ submax, int sub_shift) {
  if (topk_done(gate)) return;
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int NWV = kTkThreads / kWave, C = 4, NH = NWV * C;
  constexpr int V = 16 / (int)sizeof(Raw);
  // Four 16-byte loads in flight per thread per step; steps that lie wholly
  // inside the chunk skip the per-element bounds checks.
  constexpr int U = 4;
  constexpr int64_t STEP = (int64_t)kTkThreads * V;
  constexpr int64_t TILE = TopkGeom<DT>::kTile;
  static_assert(!FUSE || (U * STEP == TILE && KT::kBits > 8), "one whole step per tile");
  static_assert(TILE < 65536, "packed 16-bit tile counts");
  static_assert(TILE / kTkSubChunk <= 16, "sub-chunk mask in 16 bits");
  constexpr int NT = FUSE ? kTkMaxChunkTiles : 1;
  // 257 words per copy: the copies of one bin fall in different LDS banks.
  __shared__ uint32_t h[NH][257];
  __shared__ uint32_t s_am[NT];                         // per tile: above << 16 | matching
  __shared__ uint32_t s_sub[NT];                        // per tile: sub-chunks holding either
  __shared__ uint8_t s_list[NT][FUSE ? kTkListMax : 1];  // low bytes of matching keys
  const int tid = threadIdx.x, wid = tid / kWave;
  const int hc = wid * C + (__lane_id() % C);
  for (int k = tid; k < NH * 257; k += kTkThreads) (&h[0][0])[k] = 0;
  if constexpr (FUSE)
    for (int k = tid; k < NT; k += kTkThreads) s_am[k] = s_sub[k] = 0;
  __syncthreads();
  const int hs = 8 * (r + 1);  // bits above digit r
  const uint32_t want = hs >= KT::kBits ? 0u : (uint32_t)(state[0] >> hs);
  auto count = [&](const Raw (&v)[V]) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const uint32_t k = KT::key(v[i]) ^ flip;
      if (hs >= KT::kBits || (k >> hs) == want) atomicAdd(&h[hc][(k >> (8 * r)) & 0xffu], 1u);
    }
  };
  // FUSE: histogram one step's keys (Q groups of V, valid: in range) and add
  // them to the record of local tile lt; off: the tile offset of group 0's
  // first key (group u starts u * STEP later, inside one sub-chunk).  The
  // low bytes are taken group by group, so only one group's keys are live
  // at a time.
  auto count_record = [&](auto& v, int lt, int64_t off, auto valid) {
    constexpr int Q = (int)(sizeof(v) / sizeof(v[0]));
    uint32_t above = 0, subm = 0;
#pragma unroll
    for (int u = 0; u < Q; ++u) {
      uint32_t eqm = 0, abv = 0;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const uint32_t k = KT::key(v[u][i]) ^ flip;
        const bool ok = valid(u, i);
        const bool eq = ok && (k >> 8) == want;
        if (eq) atomicAdd(&h[hc][k & 0xffu], 1u);
        abv += ok && (k >> 8) > want ? 1u : 0u;
        eqm |= (eq ? 1u : 0u) << i;
      }
      above += abv;
      if ((eqm | abv) != 0) subm |= 1u << (int)((off + u * STEP) / kTkSubChunk);
      if (eqm != 0) {
        uint32_t slot = atomicAdd(&s_am[lt], (uint32_t)__builtin_popcount(eqm)) & 0xffffu;
        if (slot < (uint32_t)kTkListMax) {
#pragma unroll
          for (int i = 0; i < V; ++i) {
            if ((eqm >> i) & 1u) {
              if (slot < (uint32_t)kTkListMax) s_list[lt][slot] = (uint8_t)((KT::key(v[u][i]) ^ flip) & 0xffu);
              ++slot;
            }
          }
        }
      }
    }
    if (above != 0) atomicAdd(&s_am[lt], above << 16);
    if (subm != 0) atomicOr(&s_sub[lt], subm);
  };
  // Whole steps of this workgroup: step0, step0 + stride, ..., nst of them,
  // and a last one that is not whole where `end` cuts it.  Without a gate a
  // range of its own.  Behind one, steps that lie apart: a wave leaves out
  // those whose sub-chunks all lie below the bound (no key there is selected,
  // and the digits chosen count only keys at or above the k-th), and the
  // rest may lie together.
  constexpr int64_t SPAN = U * STEP;
  const int64_t step0 = gate ? (int64_t)blockIdx.x * SPAN : (int64_t)blockIdx.x * chunk;
  const int64_t stride = gate ? (int64_t)gridDim.x * SPAN : SPAN;
  const int64_t end = gate || step0 + chunk > n ? n : step0 + chunk;
  const int nst = end - step0 >= SPAN ? (int)((end - step0 - SPAN) / stride) + 1 : 0;
  const uint32_t bound = gate ? gate[1] : 0u;
  const int64_t wave0 = (int64_t)__builtin_amdgcn_readfirstlane(wid) * (kWave * V);
  for (int j0 = 0; j0 < nst; j0 += kWave) {
    uint64_t todo = nst - j0 < kWave ? (1ull << (nst - j0)) - 1ull : ~0ull;
    if (gate) {
      // Lane l looks at step j0 + l.
      const int j = j0 + (int)__lane_id();
      uint32_t m = 0;
      if (j < nst) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t q = submax[(step0 + j * stride + u * STEP + wave0) >> sub_shift];
          m = m > q ? m : q;
        }
      }
      todo &= __ballot(m >= bound);
    }
    while (todo != 0) {
      // In a vector register: for a uniform tile the compiler would join the
      // lanes' LDS adds one lane at a time.
      int j = j0 + __builtin_ctzll(todo);
      asm volatile("" : "+v"(j));
      todo &= todo - 1;
      const int64_t b0 = step0 + j * stride + (int64_t)tid * V;
      Raw v[U][V];
#pragma unroll
      for (int u = 0; u < U; ++u) load_items<Raw, V, true>(x, b0 + u * STEP, end, v[u]);
      if constexpr (FUSE) {
        count_record(v, j, (int64_t)tid * V, [](int, int) { return true; });
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) count(v[u]);
      }
    }
  }
  const int64_t last = step0 + nst * stride;
  int tail = nst;
  asm volatile("" : "+v"(tail));
  for (int64_t b0 = last + (int64_t)tid * V; b0 < end; b0 += STEP) {
    Raw v[1][V];
    load_items<Raw, V, false>(x, b0, end, v[0]);
    if constexpr (FUSE) {
      count_record(v, tail, b0 - last, [&](int, int i) { return b0 + i < end; });
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const uint32_t k = KT::key(v[0][i]) ^ flip;
        const bool match = b0 + i < end && (hs >= KT::kBits || (k >> hs) == want);
        if (match) atomicAdd(&h[hc][(k >> (8 * r)) & 0xffu], 1u);
      }
    }
  }
  __syncthreads();
  for (int e = tid; e < 256; e += kTkThreads) {
    uint32_t s = 0;
#pragma unroll
    for (int w = 0; w < NH; ++w) s += h[w][e];
    if (!gate) {
      partial[(size_t)blockIdx.x * 256 + e] = s;
    } else if (s != 0) {
      __hip_atomic_fetch_add(&bins[e], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if constexpr (FUSE) {
    const int64_t tile0 = step0 / TILE, apart = stride / TILE;
    const int ntl = end > step0 ? (int)((end - step0 + stride - 1) / stride) : 0;
    for (int e = tid; e < ntl; e += kTkThreads) {
      const uint32_t am = s_am[e];
      tstat[tile0 + e * apart] = ((uint64_t)(am >> 16) << 32) | (s_sub[e] << 16) | (am & 0xffffu);
    }
    for (int e = tid; e < ntl * kTkListMax; e += kTkThreads)
      tlist[(tile0 + e / kTkListMax * apart) * kTkListMax + e % kTkListMax] = s_list[e / kTkListMax][e % kTkListMax];
  }
  // Behind a gate the last workgroup picks the digit and leaves the bins zero
  // for the next launch.
  if (gate && topk_last_arrival(arrived)) {
    auto sum = [&](int d, int q, int) {
      if (q != 0) return 0u;
      const uint32_t c = __hip_atomic_load(&bins[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&bins[d], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return c;
    };
    topk_pick<kTkThreads>(sum, r, hs >= KT::kBits, k_all, state);
  }
}

// First level of the digit-count sum: workgroup q adds the partials of
// groups [q * per, (q + 1) * per) into psum[q] (64-bit, high half zero), so
// that the pick reads kTkSumGroups rows instead of one per histogram group.
constexpr int kTkSumGroups = 32;
__global__ __launch_bounds__(256) void topk_sum_kernel(const uint64_t* __restrict__ partial, int groups, int per,
                                                       uint64_t* __restrict__ psum) {
  const int d = threadIdx.x;
  const int g0 = blockIdx.x * per;
  const int g1 = g0 + per < groups ? g0 + per : groups;
  uint32_t s = 0;
  int g = g0;
  for (; g + 8 <= g1; g += 8) {  // eight loads in flight
    uint64_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = partial[(size_t)(g + u) * 256 + d];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += (uint32_t)v[u];
  }
  for (; g < g1; ++g) s += (uint32_t)partial[(size_t)g * 256 + d];
  psum[(size_t)blockIdx.x * 256 + d] = s;
}

__global__ __launch_bounds__(kTkPickThreads) void topk_pick_kernel(const uint64_t* __restrict__ partial,
                                                                   int groups, int r, int first, int64_t k,
                                                                   uint64_t* __restrict__ state) {
  auto count = [&](int d, int q, int nq) {
    uint32_t s = 0;
    int g = q;
    for (; g + 7 * nq < groups; g += 8 * nq) {  // eight loads in flight
      uint64_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = partial[(size_t)(g + nq * u) * 256 + d];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += (uint32_t)v[u];
    }
    for (; g < groups; g += nq) s += (uint32_t)partial[(size_t)g * 256 + d];
    return s;
  };
  topk_pick<kTkPickThreads>(count, r, first, k, state);
}

// ---------------------------------------------------------------------------
// Ordered selection: keys above T go to [0, k - need) in input order, the
// first `need` keys equal to T to [k - need, k).  Three launches with no
// look-back: per-tile counts, one scan of them, then placement, in which a
// tile that places nothing (most of them when k is small) exits after
// reading two words.
// ---------------------------------------------------------------------------

// Loads tile `tile` and sets, per lane group, the bits of the keys above T
// (gtb) and equal to T (eqb); FULL: the tile lies wholly inside [0, n).
// A tile holds at most 16384 keys, so a count
// packed as greater << 16 | equal never carries between the halves.
template <int DT, bool FULL>
__device__ __forceinline__ void topk_classify(const typename SortKey<DT>::Raw* __restrict__ x, int64_t n,
                                              uint32_t flip, uint32_t T, uint32_t tile, int wid, int lane,
                                              Packed<typename SortKey<DT>::Raw, kTkG> (&xv)[TopkGeom<DT>::J],
                                              uint32_t (&gtb)[TopkGeom<DT>::J], uint32_t (&eqb)[TopkGeom<DT>::J]) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int G = kTkG, J = TopkGeom<DT>::J;
  constexpr int64_t TILE = TopkGeom<DT>::kTile;
  static_assert(TILE <= 16384, "packed 16-bit tile counts");
  constexpr int64_t GSPAN = (int64_t)kWave * G, WSEG = GSPAN * J;
  const int64_t wbase = (int64_t)tile * TILE + (int64_t)wid * WSEG + (int64_t)lane * G;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int64_t gb = wbase + j * GSPAN;
    load_items<Raw, G, FULL>(x, gb, n, xv[j]);
    uint32_t g = 0, e = 0;
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const uint32_t kk = KT::key(xv[j][i]) ^ flip;
      const bool valid = FULL || gb + i < n;
      g |= (valid && kk > T ? 1u : 0u) << i;
      e |= (valid && kk == T ? 1u : 0u) << i;
    }
    gtb[j] = g;
    eqb[j] = e;
  }
}

template <int DT>
__device__ __forceinline__ void topk_classify_any(const typename SortKey<DT>::Raw* __restrict__ x, int64_t n,
                                                  uint32_t flip, uint32_t T, uint32_t tile, int wid, int lane,
                                                  Packed<typename SortKey<DT>::Raw, kTkG> (&xv)[TopkGeom<DT>::J],
                                                  uint32_t (&gtb)[TopkGeom<DT>::J],
                                                  uint32_t (&eqb)[TopkGeom<DT>::J]) {
  if ((int64_t)(tile + 1) * TopkGeom<DT>::kTile <= n) {
    topk_classify<DT, true>(x, n, flip, T, tile, wid, lane, xv, gtb, eqb);
  } else {
    topk_classify<DT, false>(x, n, flip, T, tile, wid, lane, xv, gtb, eqb);
  }
}

// In place: tcnt[t] = sum of tcnt over the tiles before t, for t in
// [0, tiles]; one workgroup of NT
// threads, 16 NT tiles per round.  Wave w takes the
// round's tiles [w * 1024, (w + 1) * 1024), lane l tiles w * 1024 + 64q + l
// (coalesced loads and stores: 16 consecutive tiles per thread put every
// lane of a load in a different line, 17.8 us per scan of 16384 tiles),
// scanned as 16 wave scans in order.  The packed halves sum without a carry
// (each total is below 2^31).
constexpr int kTkScanThreads = 1024, kTkScanPer = 16;
template <int NT, bool SHARED>
__device__ __forceinline__ void topk_tilescan(uint64_t* tcnt, uint32_t tiles) {
  constexpr int NWV = NT / kWave;
  constexpr int64_t WSPAN = (int64_t)kWave * kTkScanPer;
  constexpr int64_t ROUND = (int64_t)NT * kTkScanPer;
  __shared__ int64_t s_w[NWV];
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  int64_t carry = 0;
  for (int64_t r0 = 0; r0 < tiles; r0 += ROUND) {
    const int64_t wb = r0 + (int64_t)wid * WSPAN + lane;
    int64_t v[kTkScanPer];
#pragma unroll
    for (int q = 0; q < kTkScanPer; ++q) v[q] = wb + q * kWave < tiles ? (int64_t)topk_read<SHARED>(&tcnt[wb + q * kWave]) : 0;
    int64_t run = 0;  // the wave's tiles before row q
#pragma unroll
    for (int q = 0; q < kTkScanPer; ++q) {
      const int64_t incl = wave_incl_scan(v[q]);
      const int64_t row = readlane(incl, kWave - 1);
      v[q] = run + incl - v[q];
      run += row;
    }
    if (lane == 0) s_w[wid] = run;
    __syncthreads();
    int64_t before = carry, total = carry;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const int64_t sw = s_w[w];
      before += w < wid ? sw : 0;
      total += sw;
    }
#pragma unroll
    for (int q = 0; q < kTkScanPer; ++q)
      if (wb + q * kWave < tiles) tcnt[wb + q * kWave] = (uint64_t)(before + v[q]);
    carry = total;
    __syncthreads();  // s_w is rewritten by the next round
  }
  if (tid == 0) tcnt[tiles] = (uint64_t)carry;
}

// tcnt[tile] = (keys above T) << 32 | (keys equal to T) in the tile.  Behind
// a gate, tiles whose sub-chunks all lie below the bound are not read.
template <int DT>
__global__ __launch_bounds__(kTkNW * kWave) void topk_tilecount_kernel(
    const typename SortKey<DT>::Raw* __restrict__ x, int64_t n, uint32_t flip,
    const uint64_t* __restrict__ state, uint64_t* tcnt, uint32_t tiles, const uint32_t* __restrict__ gate,
    uint32_t* __restrict__ arrived, const uint32_t* __restrict__ submax, int sub_shift) {
  constexpr int J = TopkGeom<DT>::J, NW = kTkNW;
  constexpr int64_t TILE = TopkGeom<DT>::kTile;
  if (topk_done(gate)) return;
  __shared__ int s_w[NW];
  const int lane = __lane_id(), wid = threadIdx.x / kWave;
  const uint32_t bound = gate ? gate[1] : 0u;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    if (gate) {
      const int64_t p = (int64_t)tile * TILE + ((int64_t)lane << sub_shift);
      const bool in = ((int64_t)lane << sub_shift) < TILE && p < n;
      if (__ballot(in && submax[in ? p >> sub_shift : 0] >= bound) == 0) {
        if (threadIdx.x == 0) topk_leave(&tcnt[tile], 0, true);
        continue;
      }
    }
    Packed<typename SortKey<DT>::Raw, kTkG> xv[J];
    uint32_t gtb[J], eqb[J];
    topk_classify_any<DT>(x, n, flip, (uint32_t)state[0], tile, wid, lane, xv, gtb, eqb);
    int c = 0;
#pragma unroll
    for (int j = 0; j < J; ++j) c += (__builtin_popcount(gtb[j]) << 16) | __builtin_popcount(eqb[j]);
    c = wave_sum(c);
    __syncthreads();  // s_w of the tile before has been read
    if (lane == 0) s_w[wid] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
      int t = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) t += s_w[w];
      topk_leave(&tcnt[tile], ((uint64_t)((uint32_t)t >> 16) << 32) | ((uint32_t)t & 0xffffu), gate != nullptr);
    }
  }
  // Behind a gate the last workgroup scans the counts.
  if (gate && topk_last_arrival(arrived)) topk_tilescan<kTkNW * kWave, true>(tcnt, tiles);
}

// tcnt[tile] as topk_tilecount_kernel writes it, from the record of the
// last digit round: keys above T are those whose higher digits are above
// T's plus the recorded matching keys whose low byte is above T's, keys
// equal to T the recorded ones with T's low byte.  A tile with more matching
// keys than were recorded is counted from its keys.  One wave per tile.
// Workgroups of 256 threads spread the tiles that are read; behind a gate few
// are, and 1024 threads mean few arrivals and a quick scan.
template <int DT, int NT>
__global__ __launch_bounds__(NT) void topk_tilefix_kernel(const typename SortKey<DT>::Raw* __restrict__ x,
                                                           int64_t n, uint32_t flip,
                                                           const uint64_t* __restrict__ state,
                                                           const uint64_t* __restrict__ tstat,
                                                           const uint8_t* __restrict__ tlist,
                                                           uint64_t* tcnt, uint32_t tiles,
                                                           const uint32_t* __restrict__ gate,
                                                           uint32_t* __restrict__ arrived) {
  if (topk_done(gate)) return;
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int64_t TILE = TopkGeom<DT>::kTile;
  constexpr int V = 16 / (int)sizeof(Raw);
  const int lane = __lane_id();
  const uint32_t tile = blockIdx.x * (NT / kWave) + threadIdx.x / kWave;
  if (tile < tiles) {
    const uint32_t T = (uint32_t)state[0];
    const uint64_t rec = tstat[tile];
    const uint32_t m = (uint32_t)rec & 0xffffu;
    uint32_t g, e;
    if (m <= (uint32_t)kTkListMax) {
      const bool in = lane < (int)m;
      const uint32_t low = in ? (uint32_t)tlist[(size_t)tile * kTkListMax + lane] : 0u;
      g = (uint32_t)(rec >> 32) + (uint32_t)__popcll(__ballot(in && low > (T & 0xffu)));
      e = (uint32_t)__popcll(__ballot(in && low == (T & 0xffu)));
    } else {
      const int64_t t0 = (int64_t)tile * TILE;
      const int64_t t1 = t0 + TILE < n ? t0 + TILE : n;
      uint32_t gl = 0, el = 0;
      auto add = [&](const auto& v, int64_t b) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const uint32_t kk = KT::key(v[i]) ^ flip;
          const bool ok = b + i < t1;
          gl += ok && kk > T ? 1u : 0u;
          el += ok && kk == T ? 1u : 0u;
        }
      };
      // Four loads in flight: a wave reads the tile by itself.
      constexpr int F = 4;
      int64_t b = t0 + (int64_t)lane * V;
      for (; t0 + TILE <= n && b < t1; b += F * kWave * V) {
        Raw v[F][V];
#pragma unroll
        for (int f = 0; f < F; ++f) load_items<Raw, V, true>(x, b + f * (kWave * V), t1, v[f]);
#pragma unroll
        for (int f = 0; f < F; ++f) add(v[f], b + f * (kWave * V));
      }
      for (; b < t1; b += (int64_t)kWave * V) {
        Raw v[V];
        load_items<Raw, V>(x, b, t1, v);
        add(v, b);
      }
      g = (uint32_t)wave_sum((int)gl);
      e = (uint32_t)wave_sum((int)el);
    }
    if (lane == 0) topk_leave(&tcnt[tile], ((uint64_t)g << 32) | e, gate != nullptr);
  }
  // Behind a gate the last workgroup scans the counts.
  if (gate && topk_last_arrival(arrived)) topk_tilescan<NT, true>(tcnt, tiles);
}

__global__ __launch_bounds__(kTkScanThreads) void topk_tilescan_kernel(uint64_t* __restrict__ tcnt,
                                                                       uint32_t tiles) {
  topk_tilescan<kTkScanThreads, false>(tcnt, tiles);
}

// One wave per tile, no workgroup barrier: wave w of the grid takes tiles
// w, w + W, ... (W waves in all), reads the counts of 64 of them at once
// and ballots which place anything; for each such tile it reads the keys
// one 2048-key sub-chunk (four 512-key groups) at a time, only the
// sub-chunks its record marks when there is one (tstat non-null), and
// places them, carrying the tile's running offsets through one wave scan
// per group.  Lane l holds keys 8l..8l+7 of a group, so the wave's (group,
// lane, item) order is input order.  2^28 fp16, k = 2048: about 1,940
// tiles place; reading all of each took 31-39 us of the placement's 45-58
// (scattered 32 KB reads run far below the streaming rate), reading only
// the first 1 KB of each 4-5 us.
// WORDS: the selected keys go to cand_w as rank words (topk_word), else as
// values and positions.
constexpr int kTkPlaceThreads = 256;
__device__ __forceinline__ uint64_t topk_word(uint32_t key, uint32_t pos) { return ((uint64_t)~key << 32) | pos; }
template <int DT, bool WORDS>
__global__ __launch_bounds__(kTkPlaceThreads) void topk_place_kernel(
    const typename SortKey<DT>::Raw* __restrict__ x, int64_t n, uint32_t flip,
    const uint64_t* __restrict__ state, int64_t k, const uint64_t* __restrict__ tcnt,
    const uint64_t* __restrict__ tstat, typename SortKey<DT>::Raw* __restrict__ cand_v,
    int32_t* __restrict__ cand_i, uint64_t* __restrict__ cand_w, uint32_t num_tiles,
    const uint32_t* __restrict__ gate) {
  if (topk_done(gate)) return;
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int G = kTkG;
  constexpr int64_t TILE = TopkGeom<DT>::kTile;
  constexpr int64_t GSPAN = (int64_t)kWave * G;
  constexpr int B = (int)(kTkSubChunk / GSPAN);  // groups per sub-chunk
  constexpr int NS = (int)(TILE / kTkSubChunk);  // sub-chunks per tile
  static_assert(TILE % kTkSubChunk == 0 && kTkSubChunk % GSPAN == 0, "whole sub-chunks of whole groups");
  constexpr uint32_t kAll = (1u << NS) - 1u;
  static_assert(GSPAN < 65536, "packed 16-bit group counts");
  const int64_t need = (int64_t)state[1];
  const int64_t c_gt = k - need;
  const uint32_t T = (uint32_t)state[0];
  const int lane = __lane_id();
  const uint32_t W = gridDim.x * (kTkPlaceThreads / kWave);
  const uint32_t gw = blockIdx.x * (kTkPlaceThreads / kWave) + threadIdx.x / kWave;
  if (gw >= num_tiles) return;
  const uint32_t per = (num_tiles - gw + W - 1) / W;
  for (uint32_t j0 = 0; j0 < per; j0 += kWave) {
    int64_t lgt0 = 0, leq0 = 0;
    uint32_t lsub = kAll;
    bool places = false;
    if (j0 + lane < per) {
      const uint32_t t = gw + (j0 + lane) * W;
      const uint64_t e0 = tcnt[t], e1 = tcnt[t + 1];
      if (tstat) lsub = (uint32_t)(tstat[t] >> 16) & kAll;
      lgt0 = (int64_t)(e0 >> 32);
      leq0 = (int64_t)(e0 & 0xffffffffu);
      const int64_t gth = (int64_t)(e1 >> 32) - lgt0, eqh = (int64_t)(e1 & 0xffffffffu) - leq0;
      places = !(gth == 0 && (eqh == 0 || leq0 >= need));
    }
    uint64_t mask = __ballot(places);
    while (mask != 0) {
      const int b = __builtin_ctzll(mask);
      mask &= mask - 1;
      const uint32_t tile = gw + (j0 + (uint32_t)b) * W;
      int64_t gpos = readlane(lgt0, b), epos = readlane(leq0, b);  // the wave's running offsets
      uint32_t subs = (uint32_t)readlane((int)lsub, b);
      const int64_t t0 = (int64_t)tile * TILE;
      auto batch = [&](int r, auto full_c) {
        constexpr bool FULL = decltype(full_c)::value;
        Packed<Raw, G> xv[B];
#pragma unroll
        for (int q = 0; q < B; ++q) load_items<Raw, G, FULL>(x, t0 + (r + q) * GSPAN + lane * G, n, xv[q]);
#pragma unroll
        for (int q = 0; q < B; ++q) {
          const int64_t gb = t0 + (r + q) * GSPAN + lane * G;
          uint32_t gtb = 0, eqb = 0;
#pragma unroll
          for (int i = 0; i < G; ++i) {
            const uint32_t kk = KT::key(xv[q][i]) ^ flip;
            const bool valid = FULL || gb + i < n;
            gtb |= (valid && kk > T ? 1u : 0u) << i;
            eqb |= (valid && kk == T ? 1u : 0u) << i;
          }
          // Most groups of a placing tile hold no selected key: skip their
          // scan (2^28 fp16, k = 2048: the scan and placement loop of every
          // group made each placing wave a chain of ~5,400 VALU
          // instructions, 53 us per call).
          if (__ballot((gtb | eqb) != 0) == 0) continue;
          const int c = (__builtin_popcount(gtb) << 16) | __builtin_popcount(eqb);
          const int incl = wave_incl_scan(c);
          const int tot = readlane(incl, kWave - 1);
          if ((gtb | eqb) != 0) {
            const int ex = incl - c;
            int64_t gp = gpos + (ex >> 16), ep = epos + (ex & 0xffff);
            auto put = [&](int64_t at, Raw r, int64_t pos) {
              if constexpr (WORDS) {
                cand_w[at] = topk_word(KT::key(r) ^ flip, (uint32_t)pos);
              } else {
                cand_v[at] = r;
                cand_i[at] = (int32_t)pos;
              }
            };
#pragma unroll
            for (int i = 0; i < G; ++i) {
              if ((gtb >> i) & 1u) {
                put(gp, xv[q][i], gb + i);
                ++gp;
              } else if ((eqb >> i) & 1u) {
                if (ep < need) put(c_gt + ep, xv[q][i], gb + i);
                ++ep;
              }
            }
          }
          gpos += tot >> 16;
          epos += tot & 0xffff;
        }
      };
      // Sub-chunks in order; the ones skipped hold no selected key.
      const bool full_tile = t0 + TILE <= n;
      while (subs != 0) {
        const int c = __builtin_ctz(subs);
        subs &= subs - 1;
        if (full_tile) {
          batch(c * B, std::integral_constant<bool, true>{});
        } else if (t0 + c * kTkSubChunk < n) {
          batch(c * B, std::integral_constant<bool, false>{});
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Sampled estimate of the k-th largest fp16 value (one per block).
// ---------------------------------------------------------------------------
constexpr int kPivInner = 8, kPivOuter = 4, kPivIters = 8;

// Descending rank of `key` among the lanes [first, first + count) of its
// wave (ties broken by lane index); lanes outside compare as absent.
__device__ __forceinline__ int rank_desc(uint32_t key, int first, int count) {
  const int lane = __lane_id();
  int r = 0;
  for (int j = 0; j < count; ++j) {
    const uint32_t o = (uint32_t)__shfl((int)key, first + j);
    r += (o > key || (o == key && first + j < lane)) ? 1 : 0;
  }
  return r;
}

__global__ __launch_bounds__(256) void topk_pivot_kernel(const uint16_t* __restrict__ x, int64_t n, int num_samples,
                                                         int64_t tiles_per_block, uint16_t* __restrict__ out) {
  using KT = SortKey<TCS_F16>;
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  const int64_t tile_len = (int64_t)num_samples * 32;
  const int64_t t_begin = (int64_t)blockIdx.x * tiles_per_block;
  __shared__ uint32_t s_gk[64];
  __shared__ uint16_t s_gr[64];
  __shared__ uint32_t s_tk;
  __shared__ uint16_t s_tr;
  uint32_t best_k = 0;
  uint16_t best_r = 0xfc00u;  // -inf
  for (int it = 0; it < kPivIters && it < tiles_per_block; ++it) {
    const int64_t base = (t_begin + it) * tile_len;
    if (base >= n) break;
    // Two groups of 32 per wave, four waves: eight groups per round.
    for (int g0 = wid * 2; g0 < num_samples; g0 += 8) {
      const int g = g0 + (lane >> 5);
      const int64_t p = base + (int64_t)g * 32 + (lane & 31);
      const uint16_t raw = (g < num_samples && p < n) ? x[p] : (uint16_t)0xfc00u;
      const uint32_t key = KT::key(raw);
      const int r = rank_desc(key, lane & 32, 32);
      if (g < num_samples && r == kPivInner - 1) {
        s_gk[g] = key;
        s_gr[g] = raw;
      }
    }
    __syncthreads();
    if (wid == 0) {
      const bool in = lane < num_samples;
      const uint32_t key = in ? s_gk[lane] : 0u;
      const int r = rank_desc(key, 0, num_samples);
      if (in && r == kPivOuter - 1) {
        s_tk = key;
        s_tr = s_gr[lane];
      }
    }
    __syncthreads();
    if (s_tk > best_k || it == 0) {
      best_k = s_tk;
      best_r = s_tr;
    }
    __syncthreads();
  }
  if (tid == 0) out[blockIdx.x] = best_r;
}

// ---------------------------------------------------------------------------
// Maxima path.  A sub-chunk is U vectors of 64 lanes of 16 bytes; wave g of
// the grid takes sub-chunks g, g + groups, ... (at most 64; far apart, so that
// large keys that lie together fall into many groups): submax[s] = the
// sub-chunk's largest order key, gcomp[g] = the group's largest << 32 |
// ~(its first sub-chunk that holds it).  Reads at the streaming rate: seven
// packed instructions map two 16-bit keys and one takes their maximum (2^28
// fp16 keys 82 us, 6.5 TB/s; plain loads measured 12 us slower).
// ---------------------------------------------------------------------------
constexpr int kTkMaxThreads = 256;

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  auto step = [&](uint32_t o) { v = v > o ? v : o; };
  step(dpp_mov<kRowShr1>(v));
  step(dpp_mov<kRowShr2>(v));
  step(dpp_mov<kRowShr4>(v));
  step(dpp_mov<kRowShr8>(v));
  step(dpp_mov<kRowBcast15, 0xa>(v));
  step(dpp_mov<kRowBcast31, 0xc>(v));
  return (uint32_t)readlane((int)v, kWave - 1);
}

template <int DT, int U>
struct TopkSub {
  using Raw = typename SortKey<DT>::Raw;
  static constexpr int V = 16 / (int)sizeof(Raw);
  static constexpr int64_t kKeys = (int64_t)U * kWave * V;
};

template <int DT, int U>
__global__ __launch_bounds__(kTkMaxThreads) void topk_max_kernel(const typename SortKey<DT>::Raw* __restrict__ x,
                                                                 int64_t n, uint32_t flip, uint32_t subs,
                                                                 uint32_t groups, uint32_t* __restrict__ submax,
                                                                 uint64_t* __restrict__ gcomp,
                                                                 uint32_t* __restrict__ state) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int V = TopkSub<DT, U>::V;
  constexpr int64_t SUB = TopkSub<DT, U>::kKeys;
  const int lane = __lane_id();
  // Candidates, counted by the gather kernel, and the gated launches' words.
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) state[0] = state[kTkArrived] = 0;
    static_assert(kTkMaxThreads == 256, "one bin a thread");
    state[kTkBins + threadIdx.x] = 0;
  }
  const uint32_t g = blockIdx.x * (kTkMaxThreads / kWave) + threadIdx.x / kWave;
  if (g >= groups) return;
  uint32_t mine = 0, best = 0, at = g;
  int j = 0;
  for (uint32_t s = g; s < subs; s += groups, ++j) {
    const int64_t b = (int64_t)s * SUB + lane * V;
    uint32_t m = 0;
    if ((int64_t)(s + 1) * SUB <= n) {
      Packed<Raw, V> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const u32x4 q = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x + b + u * (kWave * V)));
#pragma unroll
        for (int c = 0; c < 4; ++c) v[u].w[c] = q[c];
      }
      if constexpr (KT::kBits == 16) {
        u16x2 mp = {0, 0};
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int i = 0; i < V / 2; ++i)
            mp = __builtin_elementwise_max(mp, __builtin_bit_cast(u16x2, KT::pair(v[u].w[i]) ^ (flip * 0x10001u)));
        }
        m = mp[0] > mp[1] ? mp[0] : mp[1];
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int i = 0; i < V; ++i) {
            const uint32_t k = KT::key(v[u][i]) ^ flip;
            m = m > k ? m : k;
          }
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        Raw r[V];
        load_items<Raw, V, false>(x, b + u * (kWave * V), n, r);
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const uint32_t k = b + u * (kWave * V) + i < n ? KT::key(r[i]) ^ flip : 0u;
          m = m > k ? m : k;
        }
      }
    }
    m = wave_max(m);
    if (lane == j) mine = m;
    if (m > best) {
      best = m;
      at = s;
    }
  }
  if (lane < j) submax[g + lane * groups] = mine;
  if (lane == 0) gcomp[g] = ((uint64_t)best << 32) | (uint32_t)~at;
}

// state[1] = T, state[2] = P: at least k keys are above T, or equal to T in a
// sub-chunk up to P.  T is the k-th largest of the groups' maxima, P by
// default the last of the sub-chunks that hold the maxima of the first groups
// at T.  One workgroup, the maxima in LDS; T two bits at a time from the top
// (the counts of maxima at or above three trials by ballots: a histogram's
// atomics would meet in the few bins the maxima fall into).  Short loops on
// purpose: code unrolled over registers took as long to fetch as to run.
constexpr int kTkBoundThreads = 1024;
constexpr uint32_t kTkMaxGroupsM = 16384;
template <int DT, int U>
__global__ __launch_bounds__(kTkBoundThreads) void topk_bound_kernel(const typename SortKey<DT>::Raw* __restrict__ x,
                                                                     int64_t n, uint32_t flip,
                                                                     const uint64_t* __restrict__ gcomp,
                                                                     uint32_t groups,
                                                                     const uint32_t* __restrict__ submax,
                                                                     uint32_t subs, uint32_t k,
                                                                     uint32_t* __restrict__ state) {
  constexpr int bits = SortKey<DT>::kBits;
  __shared__ uint32_t s_key[kTkMaxGroupsM];
  __shared__ uint32_t s_row[kTkMaxGroupsM / kWave];
  __shared__ uint32_t s_cnt[16][3], s_above, s_last, s_p;
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  for (uint32_t g0 = tid; g0 < groups; g0 += 8 * kTkBoundThreads) {  // eight loads in flight
    uint64_t c[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = gcomp[g0 + u * kTkBoundThreads < groups ? g0 + u * kTkBoundThreads : 0];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (g0 + u * kTkBoundThreads < groups) s_key[g0 + u * kTkBoundThreads] = (uint32_t)(c[u] >> 32);
  }
  if (tid < 48) (&s_cnt[0][0])[tid] = 0;
  if (tid == 0) s_above = s_p = 0;
  __syncthreads();
  uint32_t T = 0;
#pragma unroll 1
  for (int b = bits - 2; b >= 0; b -= 2) {
    uint32_t c[3] = {};
#pragma unroll 1
    for (uint32_t g0 = tid; g0 - lane < groups; g0 += 4 * kTkBoundThreads) {
      uint32_t key[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) key[u] = s_key[(g0 + u * kTkBoundThreads) % kTkMaxGroupsM];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = g0 + u * kTkBoundThreads < groups;
#pragma unroll
        for (int e = 0; e < 3; ++e)
          c[e] += (uint32_t)__popcll(__ballot(in && key[u] >= (T | ((uint32_t)(e + 1) << b))));
      }
    }
    if (lane < 3) atomicAdd(&s_cnt[b / 2][lane], lane == 0 ? c[0] : (lane == 1 ? c[1] : c[2]));
    __syncthreads();
    const uint32_t* sc = s_cnt[b / 2];
    T |= (uint32_t)((sc[0] >= k) + (sc[1] >= k) + (sc[2] >= k)) << b;
  }
  // Groups above T, and those at T in every row of 64.
  uint32_t above = 0;
#pragma unroll 1
  for (uint32_t g0 = wid * kWave; g0 < groups; g0 += kTkBoundThreads) {
    const bool in = g0 + lane < groups;
    const uint32_t key = in ? s_key[g0 + lane] : 0u;
    above += (uint32_t)__popcll(__ballot(in && key > T));
    const uint32_t e = (uint32_t)__popcll(__ballot(in && key == T));
    if (lane == 0) s_row[g0 / kWave] = e;
  }
  if (lane == 0) atomicAdd(&s_above, above);
  __syncthreads();
  uint32_t need = k - s_above;  // >= 1: fewer than k maxima lie above T
  // Wave 0: among e (one a lane), the lane that holds the need-th, or 64 with
  // `need` less all of them.
  auto find = [&](uint32_t e) {
    const uint32_t incl = wave_incl_scan(e);
    const uint64_t reach = __ballot(incl >= need);
    if (reach == 0) {
      need -= (uint32_t)readlane((int)incl, kWave - 1);
      return kWave;
    }
    const int l = __builtin_ctzll(reach);
    need -= (uint32_t)readlane((int)(incl - e), l);
    return l;
  };
  if (need <= k / 4) {
    // The row, and in it the group: the need-th at T in order; P covers the
    // groups at T up to it.
    if (wid == 0) {
      const int rows = (int)((groups + kWave - 1) / kWave);
      int row = 0;
#pragma unroll 1
      for (int r0 = 0; r0 < rows; r0 += kWave) {
        const int l = find(r0 + lane < rows ? s_row[r0 + lane] : 0u);
        if (l < kWave) {
          row = r0 + l;
          break;
        }
      }
      const uint32_t g = (uint32_t)row * kWave + lane;
      const int l = find(g < groups && s_key[g] == T ? 1u : 0u);
      if (lane == l) s_last = g;
    }
    __syncthreads();
#pragma unroll 1
    for (uint32_t g = tid; g <= s_last; g += kTkBoundThreads)
      if (s_key[g] == T) atomicMax(&s_p, ~(uint32_t)gcomp[g]);
    __syncthreads();
    if (tid == 0) {
      state[1] = T;
      state[2] = s_p;
    }
    return;
  }
  // Many groups at T (a value that repeats).  The sub-chunks at T in order,
  // the first `need` of them, replace the maxima in LDS ...
  constexpr int V = 16, W = kTkBoundThreads / kWave;
  uint32_t have = 0;
#pragma unroll 1
  for (uint32_t b = 0; b < subs && have < need; b += kTkBoundThreads * V) {
    // Wave w takes 64 V sub-chunks from b + 64 V w, row by row.
    uint32_t m[V], cnt = 0;
    const uint32_t wb = b + (uint32_t)wid * kWave * V + lane;
#pragma unroll
    for (int u = 0; u < V; ++u) m[u] = submax[wb + u * kWave < subs ? wb + u * kWave : 0];
#pragma unroll
    for (int u = 0; u < V; ++u) cnt += (uint32_t)__popcll(__ballot(wb + u * kWave < subs && m[u] == T));
    __syncthreads();  // s_key and s_row were read
    if (lane == 0) s_row[wid] = cnt;
    __syncthreads();
    uint32_t at = have;
    for (int w = 0; w < W; ++w) {
      at += w < wid ? s_row[w] : 0;
      have += s_row[w];
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const bool in = wb + u * kWave < subs && m[u] == T;
      const uint64_t set = __ballot(in);
      const uint32_t q = at + (uint32_t)__popcll(set & ~(~0ull << lane));
      if (in && q < need) s_key[q] = wb + u * kWave;
      at += (uint32_t)__popcll(set);
    }
  }
  // ... and as a sub-chunk may hold many keys at T, those of the first are
  // counted until they suffice, or until the rest, counted as one each, will
  // give candidates that fit.  2^28 fp16 keys of four values: 148 us (763 by
  // the radix select, which too many candidates lead to).
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int KV = TopkSub<DT, U>::V, Q = 4;
  const uint32_t first = need;
  uint32_t done = 0;
#pragma unroll 1
  for (;;) {
    __syncthreads();  // s_key is written, s_row was read
#pragma unroll 1
    for (int q = 0; q < Q; ++q) {
      const uint32_t e = done + wid * Q + q;
      uint32_t c = 0;
      if (e < first) {
        auto count = [&](auto full_c) {
          constexpr bool FULL = decltype(full_c)::value;
          const int64_t b = (int64_t)s_key[e] * TopkSub<DT, U>::kKeys + lane * KV;
          Packed<Raw, KV> r[U];
#pragma unroll
          for (int u = 0; u < U; ++u) load_items<Raw, KV, FULL>(x, b + u * (kWave * KV), n, r[u]);
#pragma unroll
          for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int i = 0; i < KV; ++i)
              c += (FULL || b + u * (kWave * KV) + i < n) && (KT::key(r[u][i]) ^ flip) == T ? 1u : 0u;
          }
        };
        if ((int64_t)(s_key[e] + 1) * TopkSub<DT, U>::kKeys <= n) {
          count(std::integral_constant<bool, true>{});
        } else {
          count(std::integral_constant<bool, false>{});
        }
      }
      c = (uint32_t)wave_sum((int)c);
      if (lane == 0) s_row[wid * Q + q] = c;
    }
    __syncthreads();
    // Every wave finds the same: 64 counts, one a lane.
    const int l = find(s_row[lane]);
    if (l < kWave) {
      if (tid == 0) {
        state[1] = T;
        state[2] = s_key[done + l];
      }
      return;
    }
    done += W * Q;
    const uint32_t keys = first - need, expect = keys + need * (keys / done + 1);
    if (expect + k <= kTkCandMax) break;
  }
  // `need` left, at most the sub-chunks not yet counted.
  if (tid == 0) {
    state[1] = T;
    state[2] = s_key[done + need - 1];
  }
}

// Appends the keys above T, or equal to T in a sub-chunk up to P, as rank
// words.  A wave looks at kTkGatherSubs sub-chunk maxima and reads the
// sub-chunks that reach the bound, one after the other.  Those may lie
// together, at the front where keys repeat, so the ones a wave and a
// workgroup look at lie apart (2^25 random int8 keys, k = 2048: 37 us with
// consecutive ones, 6 so; and 2^28 fp16 keys of four values, k = 4096, gave
// one workgroup more words than its list holds, 800 us with the select behind
// it, 146 so).  A workgroup's words meet in LDS and take their place in cand_w
// with one atomic.  state[0] counts them all, stored or not.
constexpr int kTkGatherThreads = 512, kTkGatherSubs = 32;
template <int DT, int U>
__global__ __launch_bounds__(kTkGatherThreads) void topk_gather_kernel(
    const typename SortKey<DT>::Raw* __restrict__ x, int64_t n, uint32_t flip, uint32_t subs,
    const uint32_t* __restrict__ submax, uint32_t* __restrict__ state, uint64_t* __restrict__ cand_w) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int V = TopkSub<DT, U>::V;
  constexpr int64_t SUB = TopkSub<DT, U>::kKeys;
  constexpr uint32_t kList = 4096;
  __shared__ uint64_t s_list[kList];
  __shared__ uint32_t s_n, s_base;
  const int tid = threadIdx.x, lane = __lane_id(), wid = tid / kWave;
  if (tid == 0) s_n = 0;
  const uint32_t T = state[1], P = state[2];
  __syncthreads();
  // The wave's sub-chunks: first, first + step, ...; consecutive ones belong
  // to different workgroups.
  const uint32_t first = wid * gridDim.x + blockIdx.x, step = gridDim.x * (kTkGatherThreads / kWave);
  const uint32_t s = first + lane * step;
  const bool look = lane < kTkGatherSubs && s < subs;
  const uint32_t m = look ? submax[s] : 0u;
  uint64_t active = __ballot(look && (m > T || (m == T && s <= P)));
  // A workgroup whose list has overflowed has told the fallback enough.
  while (active != 0 && __hip_atomic_load(&s_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= kList) {
    const int l = __builtin_ctzll(active);
    active &= active - 1;
    const uint32_t sub = first + l * step;
    const int64_t b = (int64_t)sub * SUB + lane * V;
    const uint32_t least = sub <= P ? T : T + 1;  // T + 1 wraps only if nothing is above T
    const bool none = sub > P && T == 0xffffffffu;
    auto take = [&](auto full_c) {
      constexpr bool FULL = decltype(full_c)::value;
      Packed<Raw, V> r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) load_items<Raw, V, FULL>(x, b + u * (kWave * V), n, r[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const int64_t p = b + u * (kWave * V) + i;
          const uint32_t key = KT::key(r[u][i]) ^ flip;
          if ((FULL || p < n) && key >= least && !none) {
            const uint32_t q = atomicAdd(&s_n, 1u);
            if (q < kList) s_list[q] = topk_word(key, (uint32_t)p);
          }
        }
      }
    };
    if ((int64_t)(sub + 1) * SUB <= n) {
      take(std::integral_constant<bool, true>{});
    } else {
      take(std::integral_constant<bool, false>{});
    }
  }
  __syncthreads();
  const uint32_t c = s_n;
  if (c == 0) return;
  // More than the list holds: the count alone tells the fallback.
  if (tid == 0) s_base = atomicAdd(&state[0], c <= kList ? c : kTkCandMax + 1);
  __syncthreads();
  if (c > kList) return;
  for (uint32_t q = tid; q < c; q += kTkGatherThreads)
    if (s_base + q < kTkCandMax) cand_w[s_base + q] = s_list[q];
}

// Orders the candidates by counting: a word's rank is the number of smaller
// words (all differ), and those ranked below k go to their place.  Every
// workgroup holds all words in LDS; a wave ranks four at a time.  *count
// words, or k when count is null or has outgrown the candidates (the radix
// select has then placed exactly k).  2400 words 5 us, where a bitonic sort
// in one workgroup took 17.
constexpr int kTkRankThreads = 512, kTkRankBlocks = 256;
constexpr int64_t kTkRankMax = 4096;
template <int DT>
__global__ __launch_bounds__(kTkRankThreads) void topk_rank_kernel(const uint64_t* __restrict__ cand_w,
                                                                   const uint32_t* __restrict__ count,
                                                                   const typename SortKey<DT>::Raw* __restrict__ x,
                                                                   uint32_t k,
                                                                   typename SortKey<DT>::Raw* __restrict__ out_v,
                                                                   int32_t* __restrict__ out_i) {
  constexpr int Q = 4;
  __shared__ uint64_t s_w[kTkCandMax];
  const int tid = threadIdx.x, lane = __lane_id();
  uint32_t m = k;
  if (count && *count <= kTkCandMax) m = *count;
  const uint32_t first = (blockIdx.x * (kTkRankThreads / kWave) + tid / kWave) * Q;
  if (blockIdx.x * (kTkRankThreads / kWave) * Q >= m) return;
  // A whole row of 64 past the end, of words larger than any.
  const uint32_t padded = (m + kWave - 1) / kWave * kWave;
  for (uint32_t j = tid; j < padded; j += kTkRankThreads) s_w[j] = j < m ? cand_w[j] : ~0ull;
  __syncthreads();
  for (uint32_t i = first; i < m; i += kTkRankBlocks * (kTkRankThreads / kWave) * Q) {
    uint64_t w[Q];
    int c[Q] = {};
#pragma unroll
    for (int q = 0; q < Q; ++q) w[q] = s_w[i + q < m ? i + q : m - 1];
    for (uint32_t j = lane; j < padded; j += kWave) {
      const uint64_t o = s_w[j];
#pragma unroll
      for (int q = 0; q < Q; ++q) c[q] += o < w[q] ? 1 : 0;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const uint32_t rank = (uint32_t)wave_sum(c[q]);
      if (lane == 0 && i + q < m && rank < k) {
        const uint32_t pos = (uint32_t)w[q];
        out_v[rank] = x[pos];
        out_i[rank] = (int32_t)pos;
      }
    }
  }
}

// Placement walks the tiles with the resident grid of topk_place_kernel:
// most tiles place nothing when k is small, and each that does costs a few
// dependent round trips to memory, which the resident waves pay in
// parallel.  2^28 fp16, k = 2048: a workgroup of 8 waves per tile (block
// scans between the waves) took 42 us with 2048 workgroups of which about
// 512 fit at once and 52 us with the resident grid.
template <int DT, bool WORDS>
static uint32_t topk_place_grid() {
  static std::atomic<int> cached[kMaxCachedDevices];
  return (uint32_t)device_cached(cached, [](int dev) {
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, topk_place_kernel<DT, WORDS>, kTkPlaceThreads, 0) !=
            hipSuccess ||
        per_cu < 1)
      per_cu = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    return per_cu * cus;
  });
}

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

inline int topk_elem_bytes(int dt) {
  switch (dt) {
    case TCS_I8: return 1;
    case TCS_F16: case TCS_BF16: case TCS_I16: return 2;
    case TCS_F32: case TCS_I32: case TCS_U32: return 4;
    default: return 0;
  }
}

// Sub-chunks of one vector (U = 1) up to 2^17 of them, of four above; 4096
// groups (enough waves for the read) or four times the winners, which leave
// the bound tight, and more where a group would take over 64 sub-chunks.
// Fewer, of equal size, where those are enough for the winners (the bound
// looks at every group: 9e6 fp32 keys, k = 3000, 67 us with 11719 groups, 78
// with 16384).  Otherwise groups differ by one sub-chunk, as many at every
// size: just above a multiple of them equal ones would be half as many, too
// few for the bound (9e6 fp16 keys, k = 3000: 58 us, 88 by the select).  Keys of
// one byte gain nothing there (k = 2048: 53 us either way) and lose where the
// winners lie in one region (87, by the select 57).
constexpr int64_t kTkGroupsPerK = 3;
struct TopkMaxima {
  int U, per;
  uint32_t subs, groups;
};

inline TopkMaxima topk_maxima(int64_t n, int64_t k, int key_bytes) {
  TopkMaxima m{};
  const int64_t vec = kWave * (16 / key_bytes);
  m.U = n > vec << 17 ? 4 : 1;
  m.subs = (uint32_t)((n + m.U * vec - 1) / (m.U * vec));
  int64_t most = 4096;
  while (most < kTkMaxGroupsM && (most < 4 * k || m.subs > most * kWave)) most *= 2;
  m.groups = m.subs < most ? m.subs : (uint32_t)most;
  m.per = m.groups > 0 ? (int)((m.subs + m.groups - 1) / m.groups) : 1;
  const int64_t even = (m.subs + m.per - 1) / m.per;
  if (even >= kTkGroupsPerK * k || key_bytes == 1) m.groups = (uint32_t)even;
  return m;
}

enum class TopkPath { kSort, kMaxima, kSelect };

// The sort while its passes cost less than the maxima path's launches; the
// maxima path where it has groups enough for its bound to be tight (three
// times as many as winners: about 1.2 k candidates); where it has not, the
// sort up to kSortWideMin 16-bit keys, and the radix select beyond.  fp16, k =
// 300: 2^21 keys 31 us sorted, 30 by maxima; k = 3000, 4e6 keys: 45 us sorted,
// the select 114; fp32, k = 300: 5e5 keys 51 us sorted, 1e6 by maxima 44.
inline TopkPath topk_path(const TopkMaxima& m, int64_t n, int64_t k, int key_bytes) {
  if (n <= (key_bytes <= 2 ? (int64_t)1 << 21 : (int64_t)1 << 18)) return TopkPath::kSort;
  if (k <= kTkRankMax && (int64_t)m.groups >= kTkGroupsPerK * k && m.per <= kWave) return TopkPath::kMaxima;
  return n <= (key_bytes <= 2 ? kSortWideMin : kSortWideMin / 2) ? TopkPath::kSort : TopkPath::kSelect;
}

struct TopkLayout {
  size_t state_off, part_off, psum_off, own_total;
  size_t cand_i_off, tcnt_off, tstat_off, tlist_off, sort_scratch_off, scratch, least;
  size_t word_off, submax_off, gcomp_off, mstate_off;  // maxima path and rank words
  int groups;
  int64_t chunk;
  TopkMaxima mx;
  TopkPath path;
  bool words;  // the selected keys are ranked by counting
};

// Scratch of the select with its keys sorted: it does not fall as n or k
// grow, and is the least that tcs_topk takes, so that scratch of the largest
// sizes serves them all.  Where `avail` bytes do not hold the way that the
// sizes take, the select runs.
inline TopkLayout topk_layout(int64_t n, int64_t k, int dt, size_t avail = SIZE_MAX) {
  TopkLayout L{};
  const uint64_t tiles = (uint64_t)((n + kTkTileMin - 1) / kTkTileMin);
  int64_t groups = (n + 65535) / 65536;
  if (groups > kTkMaxGroups) groups = kTkMaxGroups;
  if (groups < 1) groups = 1;
  // Histogram chunks are whole tiles (the last round records per tile).
  const int64_t tile = topk_tile(topk_elem_bytes(dt));
  int64_t chunk = (n + groups - 1) / groups;
  chunk = (chunk + tile - 1) / tile * tile;
  groups = n > 0 ? (n + chunk - 1) / chunk : 1;
  L.groups = (int)groups;
  L.chunk = chunk;
  L.state_off = lookback_ws_bytes(tiles);
  L.part_off = align256(L.state_off + 256);
  L.psum_off = align256(L.part_off + (size_t)groups * 256 * 8);
  L.own_total = align256(L.psum_off + (size_t)kTkSumGroups * 256 * 8);
  L.cand_i_off = align256((size_t)k * topk_elem_bytes(dt));
  L.tcnt_off = align256(L.cand_i_off + (size_t)k * 4);
  L.tstat_off = align256(L.tcnt_off + (size_t)(tiles + 1) * 8);
  L.tlist_off = align256(L.tstat_off + (size_t)tiles * 8);
  L.sort_scratch_off = align256(L.tlist_off + (size_t)tiles * kTkListMax);
  const int kb = topk_elem_bytes(dt);
  L.mx = topk_maxima(n, k, kb);
  L.path = topk_path(L.mx, n, k, kb);
  L.words = k <= kTkRankMax;
  L.word_off = align256(L.sort_scratch_off +
                        (L.path == TopkPath::kSort ? sort_first_scratch_bytes(n, dt) : tcs_sort_scratch_bytes(k, dt)));
  L.submax_off = align256(L.word_off + (size_t)kTkCandMax * 8);
  L.gcomp_off = align256(L.submax_off + (size_t)L.mx.subs * 4);
  L.mstate_off = align256(L.gcomp_off + (size_t)L.mx.groups * 8);
  L.scratch = L.mstate_off + kTkStateWords * sizeof(uint32_t);
  L.least = L.sort_scratch_off + tcs_sort_scratch_bytes(k, dt);
  if (L.scratch > avail) {
    L.path = TopkPath::kSelect;
    L.words = false;
  }
  return L;
}

// The k selected keys of the radix select, by rank words (WORDS) or as
// values and positions; gated as its kernels are.
template <int DT, bool WORDS>
static int topk_select(const typename SortKey<DT>::Raw* xr, int64_t n, int64_t k, uint32_t flip, const TopkLayout& L,
                       char* w, char* sc, uint32_t* gate, hipStream_t st) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  constexpr int P = KT::kBits / 8;
  auto* state = reinterpret_cast<uint64_t*>(w + L.state_off);
  auto* partial = reinterpret_cast<uint64_t*>(w + L.part_off);
  auto* psum = reinterpret_cast<uint64_t*>(w + L.psum_off);
  // Arrivals and digit counts of the gated launches, zeroed with the gate by
  // the maxima pass.
  uint32_t* arrived = gate ? gate + kTkArrived : nullptr;
  uint32_t* bins = gate ? gate + kTkBins : nullptr;
  const auto* submax = reinterpret_cast<const uint32_t*>(sc + L.submax_off);
  const int sub_shift = __builtin_ctz(L.mx.U * kWave * (16 / (int)sizeof(Raw)));
  const int sum_per = (L.groups + kTkSumGroups - 1) / kTkSumGroups;
  const int sum_groups = (L.groups + sum_per - 1) / sum_per;
  constexpr int64_t kTile = TopkGeom<DT>::kTile;
  static_assert(kTile == (int64_t)kTkNW * (sizeof(Raw) <= 2 ? 4 : 2) * kWave * kTkG, "topk_tile");
  const uint32_t tiles = (uint32_t)((n + kTile - 1) / kTile);
  auto* tcnt = reinterpret_cast<uint64_t*>(sc + L.tcnt_off);
  auto* tstat = reinterpret_cast<uint64_t*>(sc + L.tstat_off);
  auto* tlist = reinterpret_cast<uint8_t*>(sc + L.tlist_off);
  constexpr bool kFuse = P > 1;  // keys of one byte: the tile counts read the keys
  // Few arrivals behind a gate, and at most kTkMaxChunkTiles tiles a workgroup.
  const uint32_t most = (tiles + kTkMaxChunkTiles - 1) / kTkMaxChunkTiles;
  const uint32_t few = most > kTkGatedGroups ? most : kTkGatedGroups;
  const uint32_t groups = gate && few < (uint32_t)L.groups ? few : (uint32_t)L.groups;
  for (int r = P - 1; r >= 0; --r) {
    if (kFuse && r == 0) {
      hipLaunchKernelGGL((topk_hist_kernel<DT, kFuse>), dim3(groups), dim3(kTkThreads), 0, st, xr, n, L.chunk,
                         flip, r, k, state, partial, tstat, tlist, gate, arrived, bins, submax, sub_shift);
    } else {
      hipLaunchKernelGGL((topk_hist_kernel<DT, false>), dim3(groups), dim3(kTkThreads), 0, st, xr, n, L.chunk,
                         flip, r, k, state, partial, nullptr, nullptr, gate, arrived, bins, submax, sub_shift);
    }
    TCS_CHECK_LAUNCH();
    if (!gate) {
      hipLaunchKernelGGL(topk_sum_kernel, dim3(sum_groups), dim3(256), 0, st, partial, L.groups, sum_per, psum);
      TCS_CHECK_LAUNCH();
      hipLaunchKernelGGL(topk_pick_kernel, dim3(1), dim3(kTkPickThreads), 0, st, psum, sum_groups, r,
                         r == P - 1 ? 1 : 0, k, state);
      TCS_CHECK_LAUNCH();
    }
  }
  if constexpr (kFuse) {
    if (gate) {
      hipLaunchKernelGGL((topk_tilefix_kernel<DT, 1024>), dim3((tiles + 15) / 16), dim3(1024), 0, st, xr, n, flip, state,
                         tstat, tlist, tcnt, tiles, gate, arrived);
    } else {
      hipLaunchKernelGGL((topk_tilefix_kernel<DT, 256>), dim3((tiles + 3) / 4), dim3(256), 0, st, xr, n, flip, state,
                         tstat, tlist, tcnt, tiles, gate, arrived);
    }
  } else {
    const uint32_t grid = gate && tiles > kTkGatedGroups ? kTkGatedGroups : tiles;
    hipLaunchKernelGGL((topk_tilecount_kernel<DT>), dim3(grid), dim3(kTkNW * kWave), 0, st, xr, n, flip, state, tcnt,
                       tiles, gate, arrived, submax, sub_shift);
  }
  TCS_CHECK_LAUNCH();
  if (!gate) {
    hipLaunchKernelGGL(topk_tilescan_kernel, dim3(1), dim3(kTkScanThreads), 0, st, tcnt, tiles);
    TCS_CHECK_LAUNCH();
  }
  const uint32_t resident = topk_place_grid<DT, WORDS>();
  const uint32_t wave_groups = (tiles + kTkPlaceThreads / kWave - 1) / (kTkPlaceThreads / kWave);  // a wave per tile
  const uint32_t place_grid = wave_groups < resident ? wave_groups : resident;
  hipLaunchKernelGGL((topk_place_kernel<DT, WORDS>), dim3(place_grid), dim3(kTkPlaceThreads), 0, st, xr, n, flip,
                     state, k, tcnt, kFuse ? tstat : nullptr, reinterpret_cast<Raw*>(sc),
                     reinterpret_cast<int32_t*>(sc + L.cand_i_off), reinterpret_cast<uint64_t*>(sc + L.word_off),
                     tiles, gate);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

template <int DT, int U>
static void topk_maxima_launch(const typename SortKey<DT>::Raw* xr, int64_t n, int64_t k, uint32_t flip,
                               const TopkLayout& L, char* sc, uint32_t* mstate, hipStream_t st) {
  auto* submax = reinterpret_cast<uint32_t*>(sc + L.submax_off);
  auto* gcomp = reinterpret_cast<uint64_t*>(sc + L.gcomp_off);
  constexpr uint32_t W = kTkMaxThreads / kWave, W2 = kTkGatherThreads / kWave * kTkGatherSubs;
  hipLaunchKernelGGL((topk_max_kernel<DT, U>), dim3((L.mx.groups + W - 1) / W), dim3(kTkMaxThreads), 0, st, xr, n,
                     flip, L.mx.subs, L.mx.groups, submax, gcomp, mstate);
  hipLaunchKernelGGL((topk_bound_kernel<DT, U>), dim3(1), dim3(kTkBoundThreads), 0, st, xr, n, flip, gcomp,
                     L.mx.groups, submax, L.mx.subs, (uint32_t)k, mstate);
  hipLaunchKernelGGL((topk_gather_kernel<DT, U>), dim3((L.mx.subs + W2 - 1) / W2),
                     dim3(kTkGatherThreads), 0, st, xr, n, flip, L.mx.subs, submax, mstate,
                     reinterpret_cast<uint64_t*>(sc + L.word_off));
}

template <int DT>
static int topk_run(const void* x, int64_t n, int64_t k, bool largest, void* out_v, int32_t* out_i, void* ws,
                    size_t ws_bytes, void* scratch, size_t scratch_bytes, hipStream_t st) {
  using KT = SortKey<DT>;
  using Raw = typename KT::Raw;
  const TopkLayout L = topk_layout(n, k, DT, scratch_bytes);
  char* w = static_cast<char*>(ws);
  char* sc = static_cast<char*>(scratch);
  if (L.path == TopkPath::kSort)
    return sort_first(x, DT, out_v, out_i, n, k, largest, sc + L.sort_scratch_off, st);
  const uint32_t flip = largest ? 0u : (KT::kBits == 32 ? 0xffffffffu : ((1u << KT::kBits) - 1u));
  const Raw* xr = static_cast<const Raw*>(x);
  constexpr int64_t kTile = TopkGeom<DT>::kTile;
  if (L.chunk % kTile != 0 || L.chunk / kTile > kTkMaxChunkTiles) return TCS_ERR_INVALID_ARG;
  if (!L.words) {
    const int rc = topk_select<DT, false>(xr, n, k, flip, L, w, sc, nullptr, st);
    if (rc != TCS_OK) return rc;
    // Largest first (smallest first for !largest), ties in input order.
    return tcs_sort(sc, DT, reinterpret_cast<int32_t*>(sc + L.cand_i_off), out_v, out_i, k, largest ? 1 : 0, ws,
                    ws_bytes, sc + L.sort_scratch_off, scratch_bytes - L.sort_scratch_off, st);
  }
  auto* mstate = reinterpret_cast<uint32_t*>(sc + L.mstate_off);
  uint32_t* gate = nullptr;
  if (L.path == TopkPath::kMaxima) {
    if (L.mx.U == 1) {
      topk_maxima_launch<DT, 1>(xr, n, k, flip, L, sc, mstate, st);
    } else {
      topk_maxima_launch<DT, 4>(xr, n, k, flip, L, sc, mstate, st);
    }
    TCS_CHECK_LAUNCH();
    gate = mstate;
  }
  const int rc = topk_select<DT, true>(xr, n, k, flip, L, w, sc, gate, st);
  if (rc != TCS_OK) return rc;
  hipLaunchKernelGGL((topk_rank_kernel<DT>), dim3(kTkRankBlocks), dim3(kTkRankThreads), 0, st,
                     reinterpret_cast<const uint64_t*>(sc + L.word_off), gate, xr, (uint32_t)k,
                     static_cast<Raw*>(out_v), out_i);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

}  // namespace tcs

extern "C" {

size_t tcs_topk_workspace_bytes(int64_t n, int64_t k, int dtype) {
  using namespace tcs;
  if (n < 0 || k < 0 || topk_elem_bytes(dtype) == 0) return 0;
  const size_t own = topk_layout(n, k, dtype).own_total;
  const size_t srt = tcs_sort_workspace_bytes(k, dtype);
  return own > srt ? own : srt;
}

size_t tcs_topk_scratch_bytes(int64_t n, int64_t k, int dtype) {
  using namespace tcs;
  if (n < 0 || k < 0 || topk_elem_bytes(dtype) == 0) return 0;
  return topk_layout(n, k, dtype).scratch;
}

int tcs_topk(const void* x, int dtype, int64_t n, int64_t k, int largest, void* out_vals, int32_t* out_idx,
             void* workspace, size_t workspace_bytes, void* scratch, size_t scratch_bytes, void* stream) {
  using namespace tcs;
  if (topk_elem_bytes(dtype) == 0) return TCS_ERR_UNSUPPORTED_DTYPE;
  if (n < 0 || k < 0 || k > n || n >= ((int64_t)1 << 31)) return TCS_ERR_INVALID_ARG;
  if (k == 0) return TCS_OK;
  if (!x || !out_vals || !out_idx || !aligned16(x)) return TCS_ERR_INVALID_ARG;
  if (!workspace || workspace_bytes < tcs_topk_workspace_bytes(n, k, dtype)) return TCS_ERR_WORKSPACE;
  if (!scratch || scratch_bytes < topk_layout(n, k, dtype).least) return TCS_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool lg = largest != 0;
  switch (dtype) {
    case TCS_F16: return topk_run<TCS_F16>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
    case TCS_BF16: return topk_run<TCS_BF16>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
    case TCS_F32: return topk_run<TCS_F32>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
    case TCS_I8: return topk_run<TCS_I8>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
    case TCS_I16: return topk_run<TCS_I16>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
    case TCS_I32: return topk_run<TCS_I32>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
    default: return topk_run<TCS_U32>(x, n, k, lg, out_vals, out_idx, workspace, workspace_bytes, scratch, scratch_bytes, st);
  }
}

int64_t tcs_topk_pivot_blocks(int64_t n, int num_samples) {
  if (n <= 0 || num_samples <= 0) return 0;
  const int64_t tile = (int64_t)num_samples * 32;
  const int64_t tiles = (n + tile - 1) / tile;
  return tiles < 64 ? tiles : 64;
}

int tcs_topk_pivot(const void* x, int64_t n, int num_samples, void* out, int64_t out_len, void* stream) {
  using namespace tcs;
  if (n <= 0 || num_samples < kPivOuter || num_samples > 64 || !x || !out) return TCS_ERR_INVALID_ARG;
  const int64_t blocks = tcs_topk_pivot_blocks(n, num_samples);
  if (out_len < blocks) return TCS_ERR_INVALID_ARG;
  const int64_t tile = (int64_t)num_samples * 32;
  const int64_t tiles = (n + tile - 1) / tile;
  const int64_t per_block = (tiles + blocks - 1) / blocks;
  hipLaunchKernelGGL(topk_pivot_kernel, dim3((uint32_t)blocks), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(x), n, num_samples, per_block, static_cast<uint16_t*>(out));
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

}  // extern "C"
