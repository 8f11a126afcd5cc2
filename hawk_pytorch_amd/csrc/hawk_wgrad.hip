// Weight gradient of a linear layer in a training pass: dw [N, K] = dy^T x, fp32, for dy [n, N] and
// x [n, K] in bf16 as they lie (the gradient of torch.nn.functional.linear in upstream's modules, which
// autocast rounds to bf16 and casts back).  Both operands have the sum's index as their row, so 8 x 8 blocks
// (8 rows of 16 bytes per lane) are turned in registers with 32 byte permutes on their way into LDS, where
// a matrix operand's lane finds 8 consecutive values of the sum.
//
// A workgroup of four waves owns 128 x 128 results, two workgroups share a compute unit; waves 0 and 1 fetch
// dy, waves 2 and 3 fetch x, two 64-row tiles ahead in registers.  A layer's weights are few tiles
// (1024 x 512: 32 of them), so a layer's four are one launch, the rows are split over workgroups where that still
// leaves some of the chip idle, and a second kernel adds the fp32 partial results in a fixed order.  Four weights of a
// layer of 512 channels over 2048 rows: 33.4 us in one launch, 67.8 in four (with their sums), 94.5 by the library.
// What that spares next to the library's product is the conversion to fp32, and the chip is not left idle by few
// tiles: 2048 rows, 512 x 512 13.9 us (library and conversion 17.8), 4593
// rows, 2048 x 1024 43.3 (50.0), 1024 x 1024 27.8 (38.5).  Between 512 and 4096 rows, where a few steps are split
// and the sums cost a launch, results of more than 32 tiles take up to a fifth longer than the library's (1024
// rows, 2048 x 1024: 21.2 against 17.4).  From 128 tiles on the library is as fast or faster (8192 rows, 2560 x
// 2560: 148 against 123); callers go there.
#include "hawk_scan.h"

#include <stdint.h>

#include "hawk_tile.h"

namespace hawk {
namespace {

constexpr int kThreads = 4 * kWave;
constexpr int kTile = 128, kKT = 64;
constexpr int kRowBytes = kKT * 2;
constexpr int kOperand = kTile * kRowBytes;      // bytes of one operand's tile
constexpr int kMaxSplits = 8;


// 16-byte piece c (8 values along the sum) of row r.  The permutation differs between the 8 rows that one
// LDS cycle reads and between rows 8 apart, which a transposed operand's lanes write together.
__device__ __forceinline__ int piece_offset(int r, int c) {
    return r * kRowBytes + ((c ^ ((r ^ (r >> 3)) & 7)) << 4);
}

// One product of a launch: out [M, N] (or [splits, M, N]) = a^T b for a [K, M] and b [K, N].  Its workgroups start at
// first; the launch's tasks share K and the number of splits.
struct GradTask {
    const bf16_t *a, *b;
    float* out;
    int M, N, ntiles, mtiles;
    unsigned first;
};
struct GradTasks {
    GradTask task[kWeightGradTasks];
    int n, K, splits;
};

__global__ __launch_bounds__(kThreads, 2) void weight_grad_kernel(GradTasks tasks) {
    __shared__ __align__(16) unsigned char smem[4 * kOperand];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wm = wv & 1, wn = wv >> 1;

    int which = 0;
    for (int k = 1; k < tasks.n; ++k)
        if (blockIdx.x >= tasks.task[k].first) which = k;
    const GradTask& task = tasks.task[which];
    const bf16_t* const a = task.a;
    const bf16_t* const b = task.b;
    float* const out = task.out;
    const int M = task.M, N = task.N, K = tasks.K, ntiles = task.ntiles, mtiles = task.mtiles, splits = tasks.splits;

    // row tiles of one column tile sit 8 workgroups apart: on one XCD, at about the same time
    const int blk = (int)(blockIdx.x - task.first);
    const int group = blk / (8 * mtiles), in_group = blk - group * 8 * mtiles;
    const int item = group * 8 + (in_group & 7);
    if (item >= ntiles * splits) return;      // a task's workgroups are padded to whole groups of 8
    const int split = item / ntiles;
    const int m0 = in_group / 8 * kTile, n0 = (item - split * ntiles) * kTile;
    const int all = (K + kKT - 1) / kKT;
    const int step0 = (int)((long long)all * split / splits), step1 = (int)((long long)all * (split + 1) / splits);
    const int steps = step1 - step0;

    // lane -> (8 columns, 8 rows of a step): 8 loads of 16 bytes, one per row; rows past the last read as
    // zeros (range check), columns past the last reach results that are not stored
    const bool second = wv >= 2;
    const int t = tid & 127;
    const uint32_t ld = 2u * (uint32_t)(second ? N : M);
    const size_t start = (size_t)(second ? n0 : m0) * 2u;
    const rsrc_t src = make_rsrc(reinterpret_cast<const unsigned char*>(second ? b : a) + start,
                                 (uint32_t)((size_t)K * ld - start));
    const uint32_t base = (uint32_t)(t / 16) * 8u * ld + (uint32_t)(t & 15) * 16u;

    u32x4 r[2][8];
    auto load = [&](int slot, int step) {
        // (steps past the last repeat it; nothing reads them)
        const uint32_t at = base + (uint32_t)(step0 + min(step, steps - 1)) * kKT * ld;
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            r[slot][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, at + p * ld, 0,
                                                                                         kAuxDefault));
            __builtin_amdgcn_sched_barrier(0);   // one order here and in front of the loop, or the waits merge
        }
    };
    auto stage = [&](int slot, int buf) {
        unsigned char* s = smem + buf * 2 * kOperand + (second ? kOperand : 0);
        const int col = (t & 15) * 8, c = t / 16;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            u32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = __builtin_amdgcn_perm(r[slot][2 * j + 1][e / 2], r[slot][2 * j][e / 2],
                                             e % 2 ? 0x07060302u : 0x05040100u);
            *reinterpret_cast<u32x4*>(s + piece_offset(col + e, c)) = v;
        }
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0.0f;

    const int arow = wm * 64 + (lane & 31), brow = wn * 64 + (lane & 31);
    auto multiply = [&](int buf) {
        const unsigned char* s = smem + buf * 2 * kOperand;
#pragma unroll
        for (int ks = 0; ks < kKT / 16; ++ks) {
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                fa[q] = *reinterpret_cast<const bf16x8*>(s + piece_offset(arow + 32 * q, 2 * ks + (lane >> 5)));
                fb[q] = *reinterpret_cast<const bf16x8*>(s + kOperand + piece_offset(brow + 32 * q, 2 * ks + (lane >> 5)));
            }
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int nb = 0; nb < 2; ++nb)
                    acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[nb], fa[mb], acc[mb][nb], 0, 0, 0);
        }
    };
    load(0, 0);
    load(1, 1);
    stage(0, 0);
    load(0, 2);
    lds_barrier();
    int i = 0;
    for (; i + 2 <= steps; i += 2) {
        stage(1, 1);
        load(1, i + 3);
        multiply(0);
        lds_barrier();
        stage(0, 0);
        load(0, i + 4);
        multiply(1);
        lds_barrier();
    }
    if (i < steps) {
        multiply(0);
        lds_barrier();
    }

    // the tile through LDS, [128 rows][32 pieces of 4 columns], so that it leaves in whole rows
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int row = wm * 64 + mb * 32 + (lane & 31);
                const int c = wn * 16 + nb * 8 + 2 * g + (lane >> 5);
                const f32x4 v = {acc[mb][nb][4 * g], acc[mb][nb][4 * g + 1], acc[mb][nb][4 * g + 2],
                                 acc[mb][nb][4 * g + 3]};
                *reinterpret_cast<f32x4*>(smem + (row * 32 + (c ^ (row & 7))) * 16) = v;
            }
    lds_barrier();
    const int ec = tid & 15, n = n0 + 8 * ec;
#pragma unroll
    for (int row = tid / 16; row < kTile; row += kThreads / 16) {
        const int m = m0 + row;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(smem + (row * 32 + ((2 * ec) ^ (row & 7))) * 16);
        const f32x4 hi = *reinterpret_cast<const f32x4*>(smem + (row * 32 + ((2 * ec + 1) ^ (row & 7))) * 16);
        if (m < M && n < N) {
            float* o = out + ((size_t)split * M + m) * N + n;
            *reinterpret_cast<f32x4*>(o) = lo;
            *reinterpret_cast<f32x4*>(o + 4) = hi;
        }
    }
}

// The partial results of a launch's tasks added up, 1024 values of one task per workgroup.
struct SumTask {
    const float* partial;
    float* out;
    size_t n;
    unsigned first;
};
struct SumTasks {
    SumTask task[kWeightGradTasks];
    int n;
};

template <int S>
__global__ __launch_bounds__(256) void weight_grad_sum_kernel(SumTasks tasks) {
    int which = 0;
    for (int k = 1; k < tasks.n; ++k)
        if (blockIdx.x >= tasks.task[k].first) which = k;
    const SumTask& task = tasks.task[which];
    const size_t n = task.n, at = ((size_t)(blockIdx.x - task.first) * 256 + threadIdx.x) * 4;
    if (at >= n) return;
    f32x4 part[S];
#pragma unroll
    for (int s = 0; s < S; ++s) part[s] = *reinterpret_cast<const f32x4*>(task.partial + s * n + at);
    f32x4 v = part[0];
#pragma unroll
    for (int s = 1; s < S; ++s) v += part[s];
    *reinterpret_cast<f32x4*>(task.out + at) = v;
}

int launched() { return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH; }

// Workgroups along the rows: one per compute unit in all, eight steps or more each.  With two per compute
// unit the partial results cost more than it brings (2048 rows, 2048 x 1024: 29.6 against 26.2 us; 4593
// rows, 1024 x 1024: 32.4 against 27.8), with half of one 28.6 and 34.2.
// Where every workgroup has 24 steps or more left, one split more than fills the chip once is faster: four weights of a
// layer of 512 at 6144 rows 65.7 against 79.2 us, at 4000 49 against 55 (2048 rows, 16 steps: equal).
constexpr int kWorkgroups = 256, kMinSteps = 8, kLongSteps = 24;
int tiles_of(int M, int N) { return ceil_div(M, kTile) * ceil_div(N, kTile); }
int splits_for(int tiles, int K) {
    const int steps = ceil_div(K, kKT), more = ceil_div(kWorkgroups, tiles);
    int s = steps / more >= kLongSteps ? more : kWorkgroups / tiles;
    if (s > steps / kMinSteps) s = steps / kMinSteps;
    if (s > kMaxSplits) s = kMaxSplits;
    return s < 1 ? 1 : s;
}
int splits_for(int n, int rows, const int* N, const int* K) {
    int tiles = 0;
    for (int k = 0; k < n; ++k) tiles += tiles_of(N[k], K[k]);
    return splits_for(tiles, rows);
}

}  // namespace

bool weight_grad_supported(int rows, int N, int K) {
    // byte offsets within an operand stay below 2^31, and those of the rows that fill the last step (range
    // checked, so never read) below 2^32: past that they would come out as other rows'
    return rows >= 1 && N >= 8 && N % 8 == 0 && K >= 8 && K % 8 == 0 && N < (1 << 25) && K < (1 << 25) &&
           (long long)rows * N < (1ll << 30) && (long long)rows * K < (1ll << 30) &&
           (long long)ceil_div(N, kTile) * ceil_div(K, kTile) < (1 << 20);
}
size_t weight_grads_workspace_bytes(int n, int rows, const int* N, const int* K) {
    const int s = splits_for(n, rows, N, K);
    size_t values = 0;
    for (int k = 0; k < n; ++k) values += (size_t)N[k] * K[k];
    return s > 1 ? (size_t)s * values * sizeof(float) : 0;
}
int weight_grads(int n, const void* const* dy, const void* const* x, float* const* dw, int rows, const int* N, const int* K,
                 void* ws, hipStream_t st) {
    GradTasks tasks;
    SumTasks sums;
    tasks.n = sums.n = n;
    tasks.K = rows;
    const int splits = tasks.splits = splits_for(n, rows, N, K);
    unsigned grid = 0, sum_grid = 0;
    float* partial = static_cast<float*>(ws);
    for (int k = 0; k < n; ++k) {
        GradTask& t = tasks.task[k];
        const size_t values = (size_t)N[k] * K[k];
        t = {static_cast<const bf16_t*>(dy[k]), static_cast<const bf16_t*>(x[k]), splits > 1 ? partial : dw[k], N[k], K[k],
             ceil_div(K[k], kTile), ceil_div(N[k], kTile), grid};
        sums.task[k] = {partial, dw[k], values, sum_grid};
        grid += (unsigned)(ceil_div(t.ntiles * splits, 8) * 8 * t.mtiles);
        sum_grid += (unsigned)((values / 4 + 255) / 256);
        if (splits > 1) partial += splits * values;
    }
    hipLaunchKernelGGL(weight_grad_kernel, dim3(grid), dim3(kThreads), 0, st, tasks);
    if (int rc = launched()) return rc;
    switch (splits) {
        case 1: return HAWK_OK;
#define HAWK_SUM(S) \
    case S: hipLaunchKernelGGL((weight_grad_sum_kernel<S>), dim3(sum_grid), dim3(256), 0, st, sums); break;
        HAWK_SUM(2) HAWK_SUM(3) HAWK_SUM(4) HAWK_SUM(5) HAWK_SUM(6) HAWK_SUM(7) HAWK_SUM(8)
#undef HAWK_SUM
        default: return HAWK_ERR_BAD_SHAPE;
    }
    return launched();
}

}  // namespace hawk
