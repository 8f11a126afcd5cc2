// What the matrix-core kernels of decode steps and weight gradients share (gfx950).
#pragma once

#include "hawk_device.h"

namespace hawk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__host__ __device__ inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// A barrier for what was written to LDS alone: loads from memory stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 16 bytes per lane from memory into LDS, without registers: lane l's bytes land at lds + 16 l (lds the same in
// every lane of the wave).  A lane whose lane_bytes lie past the resource's end writes zeros, which the rows past a
// sum's or a tensor's end depend on (they are added up like the others: tests with ragged rows fail otherwise);
// `bytes` is not part of that check, so lane_bytes in range plus bytes has to be in range.
__device__ __forceinline__ void load_to_lds(rsrc_t r, unsigned char* lds, uint32_t lane_bytes, uint32_t bytes) {
#if __HIP_DEVICE_COMPILE__    // (the host pass has no such builtin)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, lane_bytes, bytes, 0, 0);
#endif
}

// Until at most N of this wave's loads (and stores) are in flight; they finish in order.
template <int N>
__device__ __forceinline__ void wait_vector_memory() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Where 16-byte piece `c` of row `r` of a staged tile of 128-byte rows lies.  The pieces of a row are permuted by the
// row's number, so that the 8 rows one LDS cycle reads the same piece of cover all banks.
constexpr int kPieceRowBytes = 128;
__device__ __forceinline__ int piece_offset(int r, int c) { return r * kPieceRowBytes + ((c ^ (r & 7)) << 4); }

}  // namespace hawk
