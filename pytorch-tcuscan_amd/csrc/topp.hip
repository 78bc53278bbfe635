// Kept weights of top-p (nucleus) filtering over probabilities already
// sorted largest first, and their inclusive prefix mass: the mask step of
// the reference's top-p recipe (scripts/profiling/profile_tcuscan_ops.py:
// 335-358 and 376-398: `mask = probs_sum - probs_sort > p;
// probs_sort[mask] = 0`), fused into one pass:
//   kept[i] = (mass[i] - x[i] > p) ? 0 : x[i]   (float32 arithmetic)
// with x float16 and mass float32, as torch evaluates that expression.
#include "tcs_common.hpp"
#include "tcs_device.hpp"

namespace tcs {

constexpr int kTopPG = 8, kTopPThreads = 256;

// The kept weights of elements [b, b + kTopPG); 0 past the end.
__device__ __forceinline__ void top_p_kept(const uint16_t* __restrict__ x, const float* __restrict__ mass, float p,
                                           int64_t b, int64_t n, float (&o)[kTopPG]) {
  uint16_t h[kTopPG];
  float m[kTopPG];
  if (b + kTopPG <= n) {
    load_items<uint16_t, kTopPG, true>(x, b, n, h);
    load_items<float, kTopPG, true>(mass, b, n, m);
  } else {
    load_items<uint16_t, kTopPG, false>(x, b, n, h);
    load_items<float, kTopPG, false>(mass, b, n, m);
  }
#pragma unroll
  for (int i = 0; i < kTopPG; ++i) {
    const float v = (float)__builtin_bit_cast(_Float16, h[i]);
    o[i] = b + i >= n || m[i] - v > p ? 0.0f : v;
  }
}

__device__ __forceinline__ void top_p_store(float* __restrict__ kept, int64_t b, int64_t n,
                                            const float (&o)[kTopPG]) {
  if (b + kTopPG <= n) {
    store_items<float, kTopPG, true>(kept, b, n, o);
  } else {
    store_items<float, kTopPG, false>(kept, b, n, o);
  }
}

__global__ __launch_bounds__(kTopPThreads) void top_p_keep_kernel(const uint16_t* __restrict__ x,
                                                                  const float* __restrict__ mass, float p,
                                                                  float* __restrict__ kept, int64_t n) {
  const int64_t b = ((int64_t)blockIdx.x * kTopPThreads + threadIdx.x) * kTopPG;
  if (b >= n) return;
  float o[kTopPG];
  top_p_kept(x, mass, p, b, n, o);
  top_p_store(kept, b, n, o);
}

// Sum of one double per thread, on every thread.
__device__ __forceinline__ double top_p_block_sum(double v) {
  __shared__ double s_w[kTopPThreads / kWave];
  v = wave_sum(v);
  if (__lane_id() == 0) s_w[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = 0;
#pragma unroll
  for (int w = 0; w < kTopPThreads / kWave; ++w) t += s_w[w];
  return t;
}

// Kept weights divided by their sum, in two launches: the sum of each
// workgroup's elements, then every workgroup adds those (in double, so that
// the sum is rounded to float32 once) and divides its own, computed again.
// The elements stay in the caches; bound by the launches (131071 elements,
// the whole filter: 40.0 us with kept weights, their sum and the quotients as
// three operations, 30.2 so).
__global__ __launch_bounds__(kTopPThreads) void top_p_sum_kernel(const uint16_t* __restrict__ x,
                                                                 const float* __restrict__ mass, float p, int64_t n,
                                                                 double* __restrict__ partial) {
  const int64_t b = ((int64_t)blockIdx.x * kTopPThreads + threadIdx.x) * kTopPG;
  double t = 0;
  if (b < n) {
    float o[kTopPG];
    top_p_kept(x, mass, p, b, n, o);
#pragma unroll
    for (int i = 0; i < kTopPG; ++i) t += (double)o[i];
  }
  t = top_p_block_sum(t);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

__global__ __launch_bounds__(kTopPThreads) void top_p_divide_kernel(const uint16_t* __restrict__ x,
                                                                    const float* __restrict__ mass, float p,
                                                                    float* __restrict__ kept, int64_t n,
                                                                    const double* __restrict__ partial) {
  double t = 0;
  for (uint32_t g = threadIdx.x; g < gridDim.x; g += kTopPThreads) t += partial[g];
  const float sum = (float)top_p_block_sum(t);
  const int64_t b = ((int64_t)blockIdx.x * kTopPThreads + threadIdx.x) * kTopPG;
  if (b >= n) return;
  float o[kTopPG];
  top_p_kept(x, mass, p, b, n, o);
#pragma unroll
  for (int i = 0; i < kTopPG; ++i) o[i] /= sum;
  top_p_store(kept, b, n, o);
}

// Elements of a workgroup.
constexpr int64_t kTopPPer = (int64_t)kTopPThreads * kTopPG;

}  // namespace tcs

extern "C" {

int tcs_top_p_keep(const void* sorted_probs, const float* mass, float p, float* kept, int64_t n, void* stream) {
  using namespace tcs;
  if (n < 0) return TCS_ERR_INVALID_ARG;
  if (n == 0) return TCS_OK;
  if (!sorted_probs || !mass || !kept) return TCS_ERR_INVALID_ARG;
  if (!aligned16(sorted_probs) || !aligned16(mass) || !aligned16(kept)) return TCS_ERR_INVALID_ARG;
  const uint64_t blocks = (uint64_t)((n + kTopPPer - 1) / kTopPPer);
  if (blocks > 0x7fffffffull) return TCS_ERR_INVALID_ARG;
  hipLaunchKernelGGL(top_p_keep_kernel, dim3((uint32_t)blocks), dim3(kTopPThreads), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(sorted_probs), mass, p, kept, n);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

size_t tcs_top_p_renorm_workspace_bytes(int64_t n) {
  return n <= 0 ? 0 : (size_t)((n + tcs::kTopPPer - 1) / tcs::kTopPPer) * sizeof(double);
}

int tcs_top_p_renorm(const void* sorted_probs, const float* mass, float p, float* kept, int64_t n, void* workspace,
                     size_t workspace_bytes, void* stream) {
  using namespace tcs;
  if (n < 0) return TCS_ERR_INVALID_ARG;
  if (n == 0) return TCS_OK;
  if (!sorted_probs || !mass || !kept) return TCS_ERR_INVALID_ARG;
  if (!aligned16(sorted_probs) || !aligned16(mass) || !aligned16(kept)) return TCS_ERR_INVALID_ARG;
  if (!workspace || workspace_bytes < tcs_top_p_renorm_workspace_bytes(n)) return TCS_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(workspace) % sizeof(double) != 0) return TCS_ERR_INVALID_ARG;
  const uint64_t blocks = (uint64_t)((n + kTopPPer - 1) / kTopPPer);
  if (blocks > 0x7fffffffull) return TCS_ERR_INVALID_ARG;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const auto* x = static_cast<const uint16_t*>(sorted_probs);
  auto* partial = static_cast<double*>(workspace);
  hipLaunchKernelGGL(top_p_sum_kernel, dim3((uint32_t)blocks), dim3(kTopPThreads), 0, st, x, mass, p, n, partial);
  TCS_CHECK_LAUNCH();
  hipLaunchKernelGGL(top_p_divide_kernel, dim3((uint32_t)blocks), dim3(kTopPThreads), 0, st, x, mass, p, kept, n,
                     partial);
  TCS_CHECK_LAUNCH();
  return TCS_OK;
}

}  // extern "C"
