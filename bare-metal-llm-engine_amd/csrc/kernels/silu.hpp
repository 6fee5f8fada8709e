// silu.hpp -- SwiGLU of one element, shared by every kernel that applies it.
#pragma once

#include <hip/hip_runtime.h>

namespace eng {

// SiLU(g) * u with SiLU(g) = g / (1 + e^-g) (reference src/cpu_ref/swiglu_cpu.cpp:
// 23-25): fp32 exp and a correctly rounded divide; large negative g gives
// g / inf = -0, large positive g gives g.
__device__ __forceinline__ float swiglu_f32(float g, float u) {
  return g / (1.0f + expf(-g)) * u;
}

}  // namespace eng
