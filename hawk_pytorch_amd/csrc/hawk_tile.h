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

// A ring of S tiles in LDS, `steps` of them worked on one after the other, S - 1 loads ahead, one barrier a step.
// load(slot, step) issues LOADS loads into LDS per wave.  Step i: its tile has arrived when at most S - 2 younger ones
// are in flight; behind the barrier everyone's part has, and everyone is done with the tile of step i - 1, whose place
// the tile of step i + S - 1 takes.
template <int S, int LOADS, typename Load, typename Multiply>
__device__ __forceinline__ void staged_steps(int steps, const Load& load, const Multiply& multiply) {
    static_assert(S >= 2 && S <= 4, "the last steps' waits");
#pragma unroll
    for (int d = 0; d < S - 1; ++d)
        if (d < steps) load(d, d);
    int i = 0, slot = 0;
    for (; i + S - 1 < steps; ++i) {
        wait_vector_memory<(S - 2) * LOADS>();
        lds_barrier();
        load(slot == 0 ? S - 1 : slot - 1, i + S - 1);
        multiply(slot);
        slot = slot == S - 1 ? 0 : slot + 1;
    }
    for (; i < steps; ++i) {
        switch (steps - 1 - i) {
            case 0: wait_vector_memory<0>(); break;
            case 1: wait_vector_memory<LOADS>(); break;
            default: wait_vector_memory<2 * LOADS>(); break;       // (no more than S - 2 = 2)
        }
        lds_barrier();
        multiply(slot);
        slot = slot == S - 1 ? 0 : slot + 1;
    }
    lds_barrier();
}

}  // namespace hawk
