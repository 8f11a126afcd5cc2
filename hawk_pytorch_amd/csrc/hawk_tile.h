// What the matrix-core kernels of decode steps and weight gradients share (gfx950).
#pragma once

#include "hawk_device.h"

namespace hawk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// A barrier for what was written to LDS alone: loads from memory stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace hawk
