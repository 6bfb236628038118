// fp32 operands as three bf16 parts, for products on the half-precision matrix cores.
#pragma once

#include "uv_common.h"

namespace cgtp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// What an operand's elements ask for, or'ed over them.
constexpr unsigned kUvsPlain = 1;       // not to be split
constexpr unsigned kUvsSmall = 2;       // an element of x or W below 2^-50 (and not zero): its products with another such one
constexpr unsigned kUvsLargeY = 4;      // may be subnormal, which shows in the results only next to a y of 16 and more
__device__ __forceinline__ unsigned uvs_asks(float a) {
  const unsigned b = __builtin_bit_cast(unsigned, a) & 0x7fffffffu;
  const unsigned nonzero = b - 1u;      // 0 becomes the largest
  return (b >= (127u + 60) << 23 || nonzero < ((127u - 110) << 23) - 1 ? kUvsPlain : 0) |
         (nonzero < ((127u - 50) << 23) - 1 ? kUvsSmall : 0);
}
__device__ __forceinline__ unsigned uvs_asks_y(float y) {
  return (y - y != 0.f ? kUvsPlain : 0) | (fabsf(y) >= 16.f ? kUvsLargeY : 0);
}
// The smallest magnitude of a, b and m.
__device__ __forceinline__ float uvs_least(float a, float b, float m) {
  asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));
  return m;
}
// The three parts of pairs of elements, one conversion instruction for two (left element by element, each takes its own).
__device__ __forceinline__ unsigned uvs_pair(float a, float b) {
  const floatx2 v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float uvs_low(unsigned pair) { return __builtin_bit_cast(float, pair << 16); }
__device__ __forceinline__ float uvs_high(unsigned pair) { return __builtin_bit_cast(float, pair & 0xffff0000u); }
template <int N>
struct UvsParts {
  unsigned p[3][N / 2];
  float a, b;            // what is left of the pair in work
  // Three, three and five instructions.
  template <int STAGE>
  __device__ __forceinline__ void stage(int j, float x, float y) {
    if constexpr (STAGE == 0) {
      p[0][j] = uvs_pair(x, y);
      a = uvs_low(p[0][j]);
      b = uvs_high(p[0][j]);
    } else if constexpr (STAGE == 1) {
      a = x - a;
      b = y - b;
      p[1][j] = uvs_pair(a, b);
    } else {
      p[2][j] = uvs_pair(a - uvs_low(p[1][j]), b - uvs_high(p[1][j]));
    }
  }
  __device__ __forceinline__ void pair(int j, float x, float y) {
    stage<0>(j, x, y);
    stage<1>(j, x, y);
    stage<2>(j, x, y);
  }
};
__device__ __forceinline__ bf16x8 uvs_frag(const unsigned (&p)[4]) {
  return __builtin_bit_cast(bf16x8, u32x4{p[0], p[1], p[2], p[3]});
}

}  // namespace cgtp
