// Device helpers shared by the gate kernels (gate.hip, gate_stage.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "attn_common.h"

namespace oops {

template <typename T>
__device__ __forceinline__ float to_f(T x) {
  return (float)x;
}
// x rounded to T and back (identity for float)
template <typename T>
__device__ __forceinline__ float rnd(float x) {
  return (float)(T)x;
}
// 1 / (1 + 2^(-x log2 e)) on the hardware exp2 and reciprocal
__device__ __forceinline__ float sigmoid_f(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2e));
}

}  // namespace oops
