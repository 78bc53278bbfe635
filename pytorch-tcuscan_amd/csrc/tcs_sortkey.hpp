// Order-preserving unsigned keys of the element types that sort and top-k
// accept: key(a) < key(b) exactly when a sorts before b ascending, with
// -0.0 equal to +0.0 and every NaN after +inf (torch.sort's order).  The
// 16-bit types also map two elements held in one word at once (pair).
#pragma once

#include "tcs_common.hpp"

namespace tcs {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Order keys of two 16-bit floats held in one word, in packed 16-bit
// arithmetic (seven instructions for the two).  INF is the bit pattern of
// +inf.  With k = bits ^ (sign ? 0xffff : 0x8000), -inf maps to 0x7fff - INF
// and the finite values and +inf follow in order, ZERO - 1 being -0.0 and
// ZERO +0.0; k - (0x7fff - INF) moves the NaNs of both signs above +inf,
// where the min makes them one key, and everything above -0.0 then steps
// down by one, which merges the two zeros.
template <uint16_t INF>
__device__ __forceinline__ uint32_t float16_key_pair(uint32_t w) {
  constexpr uint16_t kLow = (uint16_t)(0x7fffu - INF), kNan = (uint16_t)(INF + 0x8000u - kLow + 1u),
                     kNegZero = (uint16_t)(0x7fffu - kLow);
  typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
  const u16x2 r = __builtin_bit_cast(u16x2, w);
  const u16x2 s = __builtin_bit_cast(u16x2, __builtin_bit_cast(i16x2, w) >> (int16_t)15);
  u16x2 t = (r ^ (s | (uint16_t)0x8000u)) - kLow;
  t = __builtin_elementwise_min(t, u16x2{kNan, kNan});
  t = __builtin_elementwise_max(__builtin_elementwise_min(t, u16x2{kNegZero, kNegZero}),
                                __builtin_elementwise_sub_sat(t, u16x2{1, 1}));
  return __builtin_bit_cast(uint32_t, t);
}

template <int DT> struct SortKey;
template <> struct SortKey<TCS_F16> {
  using Raw = uint16_t;
  static constexpr int kBits = 16;
  __device__ static uint32_t pair(uint32_t w) { return float16_key_pair<0x7c00>(w); }
  __device__ static uint32_t key(uint16_t r) { return pair(r) & 0xffffu; }
};
template <> struct SortKey<TCS_BF16> {
  using Raw = uint16_t;
  static constexpr int kBits = 16;
  __device__ static uint32_t pair(uint32_t w) { return float16_key_pair<0x7f80>(w); }
  __device__ static uint32_t key(uint16_t r) { return pair(r) & 0xffffu; }
};
template <> struct SortKey<TCS_F32> {
  using Raw = uint32_t;
  static constexpr int kBits = 32;
  __device__ static uint32_t key(uint32_t r) {
    if ((r & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;
    if (r == 0x80000000u) r = 0;
    return (r & 0x80000000u) ? ~r : (r | 0x80000000u);
  }
};
template <> struct SortKey<TCS_I8> {
  using Raw = uint8_t;
  static constexpr int kBits = 8;
  __device__ static uint32_t key(uint8_t r) { return (uint32_t)(r ^ 0x80u); }
};
template <> struct SortKey<TCS_I16> {
  using Raw = uint16_t;
  static constexpr int kBits = 16;
  __device__ static uint32_t pair(uint32_t w) { return w ^ 0x80008000u; }
  __device__ static uint32_t key(uint16_t r) { return (uint32_t)(r ^ 0x8000u); }
};
template <> struct SortKey<TCS_I32> {
  using Raw = uint32_t;
  static constexpr int kBits = 32;
  __device__ static uint32_t key(uint32_t r) { return r ^ 0x80000000u; }
};
template <> struct SortKey<TCS_U32> {
  using Raw = uint32_t;
  static constexpr int kBits = 32;
  __device__ static uint32_t key(uint32_t r) { return r; }
};

}  // namespace tcs
