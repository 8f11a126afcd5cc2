// Matrix products of a training pass around the recurrent core (upstream: the Linear modules and their autograd, which
// autocast runs in bf16):
//   * weight gradients dw [N, K] = dy^T x, fp32, for dy [n, N] and x [n, K] as they lie, up to eight in one launch;
//   * layers out [n, N] = x w^T and input gradients dx [n, K] = dy w, bf16, for w [N, K].
// Operands whose rows run along the sum are staged as they lie and turned by the transposing LDS reads; all go from
// memory into LDS without passing through registers, one barrier a step of 64 values.  A workgroup of eight waves
// (2 x 4, 64 x 32 results each) owns 128 x 128 results; layers and input gradients of up to 128 such tiles are cut into
// 64 x 64 (four waves).  Where tiles are too few for a long sum it is split over workgroups, and a second kernel adds the
// fp32 partial results in a fixed order.
//
// What bounds a step is the 32 (16) KiB that have to reach the compute unit: 0.5 us at 128 x 128, so small products want
// small tiles on more compute units, and tiles that share an operand run beside each other on one XCD.  us, in
// parentheses the library's (with its conversion for dw): four weights of a layer of 512 (MLP 1024) over 2048 rows 26.3
// in one launch (97), 62.6 in four; with operands turned in registers by byte permutes 33.4.  2048 x 1024 x 512 6.6 (7.6),
// in tiles of 128 8.1; 2048 x 512 x 512 5.0 (6.3), dx 2048 x 512 over 2048 11.9 (13.7), in tiles of 128 21.2; over
// 32000 94 (201, on 60 workgroups).  6144 x 4096 x 1024 75 (50): callers leave to the library what
// it is faster at, large outputs and weight gradients (hawk_torch.cpp has the lines and both sides' figures).
#include "hawk_scan.h"

#include <stdint.h>

#include <type_traits>

#include "hawk_tile.h"

namespace hawk {
namespace {

constexpr int kTile = 128, kSmallTile = 64;      // results of a workgroup: 128 x 128, or 64 x 64 where those are few
constexpr int kKT = 64;
constexpr int kMaxSplits = 8, kMaxInputSplits = 32;
template <int T, int STAGES>
struct Product {
    static constexpr int kWaves = T / 16, kThreads = kWaves * kWave;
    static constexpr int kOperand = T * kKT * 2;               // bytes of one operand's tile of a step
    static constexpr int kStage = 2 * kOperand;
    static constexpr int kLoads = kOperand / 1024 / kWaves;    // of 1 KiB per wave, operand and step
    static constexpr int kLds = STAGES * kStage > T * T * 4 ? STAGES * kStage : T * T * 4;
};

// An operand whose rows run along the sum ([64 rows][T columns]) is staged as it lies and read with transposing LDS
// reads: 16 lanes read 4 rows of 16 columns (32 bytes each) and every lane gets the four values of one column.  The
// 32-byte pieces of a row are permuted by its number, so that the rows an access covers (4 of them and the 4 that lie 8
// further on) fall on different banks.
template <int T>
__device__ __forceinline__ int sum_row_swizzle(int row) {
    return T == 128 ? (row & 3) | (((row >> 3) & 1) << 2) : ((row >> 1) & 1) | (((row >> 3) & 1) << 1);
}
// Two MFMA operands' worth (16 rows of the sum each) from one operand, or from three of 128 columns.  One block each, with its
// wait: as a builtin the compiler has every such read wait for all loads into LDS that are in flight.
__device__ __forceinline__ uint32_t lds_offset(const unsigned char* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)const_cast<unsigned char*>(p);
}
#define HAWK_TR(OUT, AT, OFF) "ds_read_b64_tr_b16 %" #OUT ", %" #AT " offset:" #OFF "\n\t"
template <int KS, int T>
__device__ __forceinline__ void read_transposed(uint32_t at, u32x2 (&v)[4]) {
#if __HIP_DEVICE_COMPILE__
    static_assert(KS == 0 || KS == 2, "half a step");
    if constexpr (T == 64) {
        if constexpr (KS == 0)
            asm volatile(HAWK_TR(0, 4, 0) HAWK_TR(1, 4, 512) HAWK_TR(2, 4, 2048) HAWK_TR(3, 4, 2560) "s_waitcnt lgkmcnt(0)"
                         : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at) : "memory");
        else
            asm volatile(HAWK_TR(0, 4, 4096) HAWK_TR(1, 4, 4608) HAWK_TR(2, 4, 6144) HAWK_TR(3, 4, 6656) "s_waitcnt lgkmcnt(0)"
                         : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at) : "memory");
    } else if constexpr (KS == 0)
        asm volatile(HAWK_TR(0, 4, 0) HAWK_TR(1, 4, 1024) HAWK_TR(2, 4, 4096) HAWK_TR(3, 4, 5120) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at) : "memory");
    else
        asm volatile(HAWK_TR(0, 4, 8192) HAWK_TR(1, 4, 9216) HAWK_TR(2, 4, 12288) HAWK_TR(3, 4, 13312) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at) : "memory");
#endif
}
template <int KS>
__device__ __forceinline__ void read_transposed(uint32_t at0, uint32_t at1, uint32_t at2, u32x2 (&x)[4], u32x2 (&y)[4], u32x2 (&z)[4]) {
#if __HIP_DEVICE_COMPILE__
    if constexpr (KS == 0)
        asm volatile(HAWK_TR(0, 12, 0) HAWK_TR(1, 12, 1024) HAWK_TR(4, 13, 0) HAWK_TR(5, 13, 1024) HAWK_TR(8, 14, 0)
                         HAWK_TR(9, 14, 1024) HAWK_TR(2, 12, 4096) HAWK_TR(3, 12, 5120) HAWK_TR(6, 13, 4096)
                             HAWK_TR(7, 13, 5120) HAWK_TR(10, 14, 4096) HAWK_TR(11, 14, 5120) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(y[0]), "=&v"(y[1]), "=&v"(y[2]),
                       "=&v"(y[3]), "=&v"(z[0]), "=&v"(z[1]), "=&v"(z[2]), "=&v"(z[3])
                     : "v"(at0), "v"(at1), "v"(at2) : "memory");
    else
        asm volatile(HAWK_TR(0, 12, 8192) HAWK_TR(1, 12, 9216) HAWK_TR(4, 13, 8192) HAWK_TR(5, 13, 9216) HAWK_TR(8, 14, 8192)
                         HAWK_TR(9, 14, 9216) HAWK_TR(2, 12, 12288) HAWK_TR(3, 12, 13312) HAWK_TR(6, 13, 12288)
                             HAWK_TR(7, 13, 13312) HAWK_TR(10, 14, 12288) HAWK_TR(11, 14, 13312) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(y[0]), "=&v"(y[1]), "=&v"(y[2]),
                       "=&v"(y[3]), "=&v"(z[0]), "=&v"(z[1]), "=&v"(z[2]), "=&v"(z[3])
                     : "v"(at0), "v"(at1), "v"(at2) : "memory");
#endif
}
#undef HAWK_TR
// (An operand whose rows are the result's, [T rows][64 values of the sum], is read by piece_offset.)
__device__ __forceinline__ bf16x8 operand(u32x2 lo, u32x2 hi) { return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y}); }
// One product of a launch: out [M, N] (or partial sums [splits, M, N]) = a^T b for a [K, M] and b [K, N], a b for
// a [M, K], a b^T for b [N, K].  Its workgroups start at first; the launch's tasks share K and the number of splits.
struct GradTask {
    const bf16_t *a, *b;
    void* out;
    int M, N, ntiles, mtiles;
    unsigned first;
};
struct GradTasks {
    GradTask task[kWeightGradTasks];
    int n, K, splits;
};

// A_ROWS, B_ROWS: a's rows are the result's, b's its columns ([M, K] and [N, K]; K a multiple of 64); else they run along
// the sum.  Rows past the end of the sum read as zeros (range check), rows and columns past the result repeat others
// and are not stored.  OUT: fp32, or bf16 where the sum is not split.
template <bool A_ROWS, bool B_ROWS, typename OUT, int T, int STAGES>
__global__ __launch_bounds__(T / 16 * kWave, STAGES == 2 ? 4 : 2) void sum_product_kernel(GradTasks tasks) {
    using P = Product<T, STAGES>;
    constexpr int kOperand = P::kOperand, kStage = P::kStage, kWaves = P::kWaves, MB = T / 64;
    __shared__ __align__(16) unsigned char smem[P::kLds];
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
    OUT* const out = static_cast<OUT*>(task.out);
    const int M = task.M, N = task.N, K = tasks.K, ntiles = task.ntiles, mtiles = task.mtiles, splits = tasks.splits;

    // the tiles along the result's shorter side sit 8 workgroups apart: on one XCD, at about the same time, so that the
    // longer side's operand comes to one L2
    const int blk = (int)(blockIdx.x - task.first);
    const bool rows_inside = mtiles < ntiles;
    const int inner = min(mtiles, ntiles), outer = max(mtiles, ntiles);
    const int group = blk / (8 * inner), in_group = blk - group * 8 * inner;
    const int item = group * 8 + (in_group & 7);
    if (item >= outer * splits) return;       // a task's workgroups are padded to whole groups of 8
    const int split = item / outer, ti = in_group / 8, to = item - split * outer;
    const int m0 = (rows_inside ? ti : to) * T, n0 = (rows_inside ? to : ti) * T;
    const int all = (K + kKT - 1) / kKT;
    const int step0 = (int)((long long)all * split / splits), step1 = (int)((long long)all * (split + 1) / splits);
    const int steps = step1 - step0;

    constexpr int L = P::kLoads, S = STAGES;
    const uint32_t lda = 2u * (uint32_t)(A_ROWS ? K : M), ldb = 2u * (uint32_t)(B_ROWS ? K : N);
    const rsrc_t ra = make_rsrc(a, (uint32_t)((size_t)(A_ROWS ? M : K) * lda)),
                 rb = make_rsrc(b, (uint32_t)((size_t)(B_ROWS ? N : K) * ldb));
    // a load brings 1 KiB of an operand: 512 / T rows along the sum, or 8 rows of the result
    auto sum_rows = [&](int l, uint32_t ld, int c0, int columns) {
        constexpr int kLanes = T / 8;       // of a row
        const int row = (kWave / kLanes) * (wv + l * kWaves) + lane / kLanes, p = lane % kLanes;
        const int c = c0 + 8 * ((((p >> 1) ^ sum_row_swizzle<T>(row)) << 1) | (p & 1));
        return (uint32_t)row * ld + 2u * (uint32_t)(c < columns ? c : 0);
    };
    auto result_rows = [&](int l, uint32_t ld, int r0, int rows) {
        const int row = 8 * (wv + l * kWaves) + (lane >> 3);
        return (uint32_t)min(r0 + row, rows - 1) * ld + (uint32_t)(((lane & 7) ^ (lane >> 3)) << 4);
    };
    uint32_t at_a[L], at_b[L];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        at_a[l] = A_ROWS ? result_rows(l, lda, m0, M) : sum_rows(l, lda, m0, M);
        at_b[l] = B_ROWS ? result_rows(l, ldb, n0, N) : sum_rows(l, ldb, n0, N);
    }
    auto load = [&](int slot, int step) {
        const uint32_t k = (uint32_t)(step0 + step) * kKT;
        unsigned char* s = smem + slot * kStage + wv * 1024;
#pragma unroll
        for (int l = 0; l < L; ++l) {
            load_to_lds(ra, s + l * kWaves * 1024, at_a[l] + k * (A_ROWS ? 2u : lda), 0);
            load_to_lds(rb, s + kOperand + l * kWaves * 1024, at_b[l] + k * (B_ROWS ? 2u : ldb), 0);
        }
    };

    f32x16 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][i] = 0.0f;

    // a lane's operand: column lane % 32, eight values of the sum from 8 (lane / 32) on; the transposing reads take the
    // address of row (lane % 16) / 4, columns 4 (lane % 4) of 16
    const int q = lane & 15, row = 8 * (lane >> 5) + (q >> 2);
    auto transposed_at = [&](int c0) {
        return row * 2 * T + ((((c0 >> 4) + ((lane >> 4) & 1)) ^ sum_row_swizzle<T>(row)) << 5) + (q & 3) * 8;
    };
    const int b_at = B_ROWS ? wn * 32 + (lane & 31) : kOperand + transposed_at(wn * 32);
    int a_at[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int r = wm * (T / 2) + mb * 32;
        a_at[mb] = A_ROWS ? r + (lane & 31) : transposed_at(r);
    }
    auto half = [&](auto first, const unsigned char* s) {
        constexpr int KS = decltype(first)::value;
        bf16x8 fa[2][MB], fb[2];
        auto piece = [&](int row, int k) { return piece_offset(row, 2 * (KS + k) + (lane >> 5)); };
        if constexpr (A_ROWS) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) fa[k][mb] = *reinterpret_cast<const bf16x8*>(s + piece(a_at[mb], k));
        }
        if constexpr (B_ROWS) {
            static_assert(A_ROWS, "no product has operands of this kind");
#pragma unroll
            for (int k = 0; k < 2; ++k) fb[k] = *reinterpret_cast<const bf16x8*>(s + kOperand + piece(b_at, k));
        } else {
            u32x2 b4[4], a0[4], a1[4];
            if constexpr (A_ROWS) {
                read_transposed<KS, T>(lds_offset(s + b_at), b4);
            } else {
                static_assert(T == 128, "offsets of the three-operand read");
                read_transposed<KS>(lds_offset(s + b_at), lds_offset(s + a_at[0]), lds_offset(s + a_at[1]), b4, a0, a1);
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                fb[k] = operand(b4[2 * k], b4[2 * k + 1]);
                if constexpr (!A_ROWS) {
                    fa[k][0] = operand(a0[2 * k], a0[2 * k + 1]);
                    fa[k][1] = operand(a1[2 * k], a1[2 * k + 1]);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[k], fa[k][mb], acc[mb], 0, 0, 0);
    };
    auto multiply = [&](int slot) {
        const unsigned char* s = smem + slot * kStage;
        half(std::integral_constant<int, 0>{}, s);
        half(std::integral_constant<int, 2>{}, s);
    };

    // Step i: its tile has arrived when at most S - 2 younger ones are in flight; behind the barrier everyone's part
    // has, and everyone is done with the tile of step i - 1, whose place the tile of step i + S - 1 takes.
#pragma unroll
    for (int d = 0; d < S - 1; ++d)
        if (d < steps) load(d, d);
    int i = 0, slot = 0;
    for (; i + S - 1 < steps; ++i) {
        wait_vector_memory<(S - 2) * 2 * L>();
        lds_barrier();
        load(slot == 0 ? S - 1 : slot - 1, i + S - 1);
        multiply(slot);
        slot = slot == S - 1 ? 0 : slot + 1;
    }
    for (; i < steps; ++i) {
        switch (steps - 1 - i) {
            case 0: wait_vector_memory<0>(); break;
            case 1: wait_vector_memory<2 * L>(); break;
            default: wait_vector_memory<4 * L>(); break;       // (no more than S - 2 = 2)
        }
        lds_barrier();
        multiply(slot);
        slot = slot == S - 1 ? 0 : slot + 1;
    }
    lds_barrier();

    // the tile through LDS, [T rows][T / 4 pieces of 4 columns], so that it leaves in whole rows
    constexpr int PR = T / 4;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int r = wm * (T / 2) + mb * 32 + (lane & 31), c = wn * 8 + 2 * g + (lane >> 5);
            const f32x4 v = {acc[mb][4 * g], acc[mb][4 * g + 1], acc[mb][4 * g + 2], acc[mb][4 * g + 3]};
            *reinterpret_cast<f32x4*>(smem + (r * PR + (c ^ (r & 7))) * 16) = v;
        }
    lds_barrier();
    constexpr int TPR = T / 8;       // threads per row
    const int ec = tid % TPR, n = n0 + 8 * ec;
#pragma unroll
    for (int r = tid / TPR; r < T; r += P::kThreads / TPR) {
        const int m = m0 + r;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(smem + (r * PR + ((2 * ec) ^ (r & 7))) * 16);
        const f32x4 hi = *reinterpret_cast<const f32x4*>(smem + (r * PR + ((2 * ec + 1) ^ (r & 7))) * 16);
        if (m < M && n < N) {
            OUT* o = out + ((size_t)split * M + m) * N + n;
            if constexpr (sizeof(OUT) == 2) {
                *reinterpret_cast<u32x4*>(o) = u32x4{pack_bf16x2(lo.x, lo.y), pack_bf16x2(lo.z, lo.w), pack_bf16x2(hi.x, hi.y),
                                                     pack_bf16x2(hi.z, hi.w)};
            } else {
                *reinterpret_cast<f32x4*>(o) = lo;
                *reinterpret_cast<f32x4*>(o + 4) = hi;
            }
        }
    }
}

// The partial results of a launch's tasks added up, 1024 values of one task per workgroup.
struct SumTask {
    const float* partial;
    void* out;
    size_t n;
    unsigned first;
};
struct SumTasks {
    SumTask task[kWeightGradTasks];
    int n;
};

template <int S, bool TO_BF16>
__global__ __launch_bounds__(256) void sum_partial_kernel(SumTasks tasks) {
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
    if constexpr (TO_BF16) *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(task.out) + at) = u32x2{pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)};
    else *reinterpret_cast<f32x4*>(static_cast<float*>(task.out) + at) = v;
}

int launched() { return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH; }

// Workgroups along the rows: one per compute unit in all, eight steps or more each.  With two per compute
// unit the partial results cost more than it brings (2048 rows, 2048 x 1024: 29.6 against 26.2 us; 4593
// rows, 1024 x 1024: 32.4 against 27.8), with half of one 28.6 and 34.2.
// Where every workgroup has 24 steps or more left, one split more than fills the chip once is faster: four weights of a
// layer of 512 at 6144 rows 65.7 against 79.2 us, at 4000 49 against 55 (2048 rows, 16 steps: equal).
constexpr int kWorkgroups = 256, kMinSteps = 8, kLongSteps = 24;
constexpr int kSmallTiles = 128;     // 1000 x 4096 x 1024, 256 of them: 14.3 us in 128 x 128; 128: 2048 x 1024 x 512 6.6 in 64 x 64, 8.1 in 128 x 128
int tiles_of(int M, int N) { return ceil_div(M, kTile) * ceil_div(N, kTile); }
int splits_for(int tiles, int K) {
    const int steps = ceil_div(K, kKT), more = ceil_div(kWorkgroups, tiles);
    int s = steps / more >= kLongSteps ? more : kWorkgroups / tiles;
    if (s > steps / kMinSteps) s = steps / kMinSteps;
    if (s > kMaxSplits) s = kMaxSplits;
    return s < 1 ? 1 : s;
}
unsigned workgroups_of(const GradTask& t, int splits) {
    const int inner = t.mtiles < t.ntiles ? t.mtiles : t.ntiles, outer = t.mtiles + t.ntiles - inner;
    return (unsigned)(ceil_div(outer * splits, 8) * 8 * inner);
}
template <bool A_ROWS, bool B_ROWS, typename OUT, int T>
int launch_products(const GradTasks& tasks, unsigned grid, hipStream_t st) {
    // four tiles of steps in flight where no compute unit has a second workgroup (of 64 x 64: a third), else two
    if (grid <= (unsigned)kWorkgroups * (T == kTile ? 1 : 2))
        hipLaunchKernelGGL((sum_product_kernel<A_ROWS, B_ROWS, OUT, T, 4>), dim3(grid), dim3(Product<T, 4>::kThreads), 0, st, tasks);
    else
        hipLaunchKernelGGL((sum_product_kernel<A_ROWS, B_ROWS, OUT, T, 2>), dim3(grid), dim3(Product<T, 2>::kThreads), 0, st, tasks);
    return launched();
}
template <bool TO_BF16>
int launch_sums(const SumTasks& sums, int splits, unsigned grid, hipStream_t st) {
    switch (splits) {
#define HAWK_SUM(S) \
    case S: hipLaunchKernelGGL((sum_partial_kernel<S, TO_BF16>), dim3(grid), dim3(256), 0, st, sums); break;
        HAWK_SUM(2) HAWK_SUM(3) HAWK_SUM(4) HAWK_SUM(5) HAWK_SUM(6) HAWK_SUM(7) HAWK_SUM(8) HAWK_SUM(16) HAWK_SUM(32)
#undef HAWK_SUM
        default: return HAWK_ERR_BAD_SHAPE;
    }
    return launched();
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
        grid += workgroups_of(t, splits);
        sum_grid += (unsigned)((values / 4 + 255) / 256);
        if (splits > 1) partial += splits * values;
    }
    if (int rc = launch_products<false, false, float, kTile>(tasks, grid, st)) return rc;
    return splits > 1 ? launch_sums<false>(sums, splits, sum_grid, st) : HAWK_OK;
}


namespace {
// Splits of a linear layer's sum of `steps` steps: one workgroup per compute unit, eight steps or more each; the fixed
// cost of a split product, partial sums and a launch, pays from 64 steps on.
int linear_splits_for(int tiles, int steps) {
    if (steps < 8 * kMinSteps) return 1;
    int s = ceil_div(kWorkgroups, tiles);
    if (s > steps / kMinSteps) s = steps / kMinSteps;
    if (s > 8) s = s >= kMaxInputSplits ? kMaxInputSplits : (s >= 16 ? 16 : 8);
    return s;
}
template <bool B_ROWS>
int linear(const void* a, const void* b, void* out, int M, int N, int K, void* ws, hipStream_t st) {
    const int splits = linear_splits_for(tiles_of(M, N), K / kKT);
    // an unsplit product of few tiles of 128 x 128 is cut finer
    const int tile = splits == 1 && tiles_of(M, N) <= kSmallTiles ? kSmallTile : kTile;
    GradTasks tasks;
    tasks.n = 1, tasks.K = K, tasks.splits = splits;
    GradTask& t = tasks.task[0];
    t = {static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(b), splits > 1 ? ws : out, M, N, ceil_div(N, tile),
         ceil_div(M, tile), 0};
    const unsigned grid = workgroups_of(t, splits);
    if (tile == kSmallTile) return launch_products<true, B_ROWS, bf16_t, kSmallTile>(tasks, grid, st);
    if (splits == 1) return launch_products<true, B_ROWS, bf16_t, kTile>(tasks, grid, st);
    if (int rc = launch_products<true, B_ROWS, float, kTile>(tasks, grid, st)) return rc;
    const size_t values = (size_t)M * N;
    SumTasks sums;
    sums.n = 1;
    sums.task[0] = {static_cast<const float*>(ws), out, values, 0};
    return launch_sums<true>(sums, splits, (unsigned)((values / 4 + 255) / 256), st);
}
}  // namespace

bool linear_supported(int rows, int N, int K) {
    return rows >= 1 && N >= 8 && N % 8 == 0 && K >= kKT && K % kKT == 0 && N < (1 << 25) && K < (1 << 25) &&
           (long long)rows * K < (1ll << 30) && (long long)N * K < (1ll << 30) && (long long)rows * N < (1ll << 31) &&
           (long long)ceil_div(rows, kTile) * ceil_div(N, kTile) < (1 << 20);
}
size_t linear_workspace_bytes(int rows, int N, int K) {
    const int s = linear_splits_for(tiles_of(rows, N), K / kKT);
    return s > 1 ? (size_t)s * rows * N * sizeof(float) : 0;
}
int linear_fwd(const void* x, const void* w, void* out, int rows, int N, int K, void* ws, hipStream_t st) {
    return linear<true>(x, w, out, rows, N, K, ws, st);
}
int linear_input_grad(const void* dy, const void* w, void* dx, int rows, int N, int K, void* ws, hipStream_t st) {
    return linear<false>(dy, w, dx, rows, K, N, ws, st);
}

}  // namespace hawk
