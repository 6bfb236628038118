// Accumulator-tile helpers of the fully connected products on the matrix cores.
#pragma once

#include "cgtp_device.h"
#include "cgtp_host.h"

namespace cgtp {

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float dot8(const floatx4& g0, const floatx4& g1, const floatx4& z0, const floatx4& z1) {
#pragma clang fp contract(fast)
  float s = g0[0] * z0[0];
  s += g0[1] * z0[1]; s += g0[2] * z0[2]; s += g0[3] * z0[3];
  s += g1[0] * z1[0]; s += g1[1] * z1[1]; s += g1[2] * z1[2]; s += g1[3] * z1[3];
  return s;
}

// gw[i] = sum over the chunks c of part[c * n + i] in a fixed order (uvt_kernels.hip); n a multiple of 4.
int uvt_reduce_chunks(const float* part, float* gw, int64_t n_chunks, int64_t n, hipStream_t stream);

}  // namespace cgtp
