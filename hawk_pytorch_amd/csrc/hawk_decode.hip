// Decode step around the recurrent core: the dense projections of a layer for a handful of rows
// (one new token per sequence), with the norms, residual adds and the gated GELU in the same
// kernels.  Upstream runs them as library GEMMs with eager kernels in between
// (hawk/hawk.py:53-58, :70-86, :163-203, :222-243, :284-303).
//
// With up to 256 rows a projection is a pass over its weights: 2560 x 15360 bf16 weights are
// 79 MB, 14 us at the rate a large copy reaches, and their 20 GFLOP at 256 rows are half of that
// on the matrix cores.  What the kernel must do is keep enough weight bytes in flight and touch
// every byte in as few places as possible:
//   * a workgroup of four waves owns MT rows x 64 output columns; the weights are read once per
//     MT rows, in full 128-byte lines, through registers into LDS;
//   * the waves split K, not the tile: wave w multiplies the w-th 16 of every 64 input channels for
//     the whole tile, so each staged byte is read from LDS exactly once.  With the tile split over
//     the waves instead every weight byte is read by as many waves as there are row blocks;
//   * the four partial tiles meet in LDS at the end and leave in whole rows;
//   * projections with few columns also split K over workgroups and leave fp32 partial sums, which
//     the kernel that follows (residual add + norm) adds up in a fixed order on its way.
// A layer of 2560 channels and an MLP of 7680, next layer's input projection included, takes 44 / 53 / 64 /
// 78 / 83 / 98 us at 1 / 32 / 64 / 128 / 129 / 256 rows with cold weights (157 MB); the library's four products
// alone took 121 us at 256 rows, with the norms, additions, GELU and product around them 149.
// All sums are fp32, in an order that depends on the shape alone, and values are rounded to bf16 where
// the separate operations round them, so both routes differ by the order of the sums only.
#include "hawk_scan.h"

#include <stdint.h>

#include "hawk_tile.h"

namespace hawk {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kNT = 64;          // output columns of a workgroup
constexpr int kKT = 64;          // input channels of a step: 128 bytes of a row
constexpr int kRowBytes = kKT * 2;
static_assert(kRowBytes == kPieceRowBytes, "piece_offset's rows");

enum Epilogue { kStoreBf16 = 0, kStorePartial = 1, kStoreGelu = 2 };

inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// One thread's share of a finished row: 8 adjacent columns a, c, or 4 gate columns a and the up
// columns c beside them.
template <int EPI>
__device__ __forceinline__ void store_columns(void* out, f32x4 a, f32x4 c, int split, int m, int n, int M, int N) {
    if constexpr (EPI == kStorePartial) {
        float* o = static_cast<float*>(out) + ((size_t)split * M + m) * N + n;
        *reinterpret_cast<f32x4*>(o) = a;
        *reinterpret_cast<f32x4*>(o + 4) = c;
    } else if constexpr (EPI == kStoreBf16) {
        const u32x4 r = {pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(c.x, c.y), pack_bf16x2(c.z, c.w)};
        *reinterpret_cast<u32x4*>(static_cast<bf16_t*>(out) + (size_t)m * N + n) = r;
    } else {
        // rounded where the separate operations round: the projection, the GELU, the product
        float g[4], u[4];
        unpack(u32x2{pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w)}, g);
        unpack(u32x2{pack_bf16x2(c.x, c.y), pack_bf16x2(c.z, c.w)}, u);
#pragma unroll
        for (int v = 0; v < 4; ++v) g[v] = gelu_times(g[v], 1.0f);
        unpack(u32x2{pack_bf16x2(g[0], g[1]), pack_bf16x2(g[2], g[3])}, g);
        const u32x2 r = {pack_bf16x2(g[0] * u[0], g[1] * u[1]), pack_bf16x2(g[2] * u[2], g[3] * u[3])};
        *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(out) + (size_t)m * N + n) = r;
    }
}

template <int MT>
struct GemmLds {
    static constexpr int kStage = (MT + kNT) * kRowBytes;
    static constexpr int kSums = kWaves * 32 * kNT * 4;      // the waves' sums of 32 rows
    static constexpr int kBytes = 2 * kStage > kSums ? 2 * kStage : kSums;
};

// out = x w^T for x [M, K] and w [N, K], both bf16 with dense rows; K a multiple of DEPTH * 64, N of 8.
//   kStoreBf16     out [M, N] bf16
//   kStorePartial  out [splits, M, N] fp32, split s over its share of K
//   kStoreGelu     w [2 N, K] holds gate rows, then up rows; out [M, N] bf16 = gelu(gate) * up
// DEPTH: tiles kept in flight in registers.
template <int MT, int DEPTH, int EPI>
__global__ __launch_bounds__(kThreads, 3) void decode_gemm_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int M, int N, int K,
    int ntiles, int mtiles, int splits) {
    constexpr int MB = MT / 32;
    constexpr int XP = MT / 32;               // 16-byte loads per thread and step for x; the weights take two
    static_assert(DEPTH == 2 || DEPTH == 4, "an even number of steps per turn of the loop");
    __shared__ __align__(16) unsigned char smem[GemmLds<MT>::kBytes];

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);

    // The row tiles of one weight tile sit 8 workgroups apart: on the same XCD, at the same time,
    // so the second one finds the weights in that XCD's L2.
    const int b = (int)blockIdx.x;
    const int group = b / (8 * mtiles), in_group = b - group * 8 * mtiles;
    const int mt = in_group / 8;
    const int item = group * 8 + (in_group & 7);
    if (item >= ntiles * splits) return;      // the grid is padded to whole groups of 8
    const int split = item / ntiles;
    const int nt = item - split * ntiles;
    const int m0 = mt * MT, n0 = nt * (EPI == kStoreGelu ? kNT / 2 : kNT);

    // this split's share of K, in turns of DEPTH steps
    const int turns = K / (DEPTH * kKT);
    const int turn0 = (int)((long long)turns * split / splits);
    const int turn1 = (int)((long long)turns * (split + 1) / splits);
    const int steps = (turn1 - turn0) * DEPTH;
    const uint32_t k_bytes0 = (uint32_t)turn0 * DEPTH * kRowBytes;
    const uint32_t row_bytes = (uint32_t)K * 2u;
    // rows past M and weight rows past N read as zeros (range check of the buffer resources)
    const rsrc_t bx = make_rsrc(x + (size_t)m0 * K, (uint32_t)min(MT, M - m0) * row_bytes);
    const int n1 = EPI == kStoreGelu ? N + n0 : n0 + 32;            // first row of the tile's second half
    const int rows0 = min(32, N - n0), rows1 = EPI == kStoreGelu ? rows0 : max(min(32, N - n1), 0);
    const rsrc_t bw0 = make_rsrc(w + (size_t)n0 * K, (uint32_t)rows0 * row_bytes);
    const rsrc_t bw1 = make_rsrc(rows1 > 0 ? w + (size_t)n1 * K : w, (uint32_t)rows1 * row_bytes);

    const int lr = tid / 8, lc = tid & 7;     // a load covers 32 rows of 128 bytes
    const uint32_t lane_bytes = (uint32_t)lr * row_bytes + (uint32_t)lc * 16u;
    const int piece = piece_offset(lr, lc);   // (rows 32 apart have the same permutation)

    u32x4 rx[DEPTH][XP], rw[DEPTH][2];
    auto load = [&](int slot, int step) {
        const uint32_t k = k_bytes0 + (uint32_t)min(step, steps - 1) * kRowBytes;
        // The loads keep this order, here and in front of the loop: the compiler counts them to know
        // which have arrived, and where two orders meet it waits for all of the younger step too.
#pragma unroll
        for (int p = 0; p < XP; ++p) {
            rx[slot][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                        bx, lane_bytes + p * 32u * row_bytes + k, 0, kAuxDefault));
            __builtin_amdgcn_sched_barrier(0);
        }
        rw[slot][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bw0, lane_bytes + k, 0, kAuxDefault));
        __builtin_amdgcn_sched_barrier(0);
        rw[slot][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bw1, lane_bytes + k, 0, kAuxDefault));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](int slot, int buf) {
        unsigned char* s = smem + buf * GemmLds<MT>::kStage;
#pragma unroll
        for (int p = 0; p < XP; ++p) *reinterpret_cast<u32x4*>(s + p * 32 * kRowBytes + piece) = rx[slot][p];
        *reinterpret_cast<u32x4*>(s + MT * kRowBytes + piece) = rw[slot][0];
        *reinterpret_cast<u32x4*>(s + (MT + 32) * kRowBytes + piece) = rw[slot][1];
    };

    f32x16 acc[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nh = 0; nh < 2; ++nh)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mb][nh][i] = 0.0f;

    // operand of this wave: 16 input channels = two 16-byte pieces of every row
    const int op = piece_offset(lane & 31, 2 * wv + (lane >> 5));

#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(d, d);
    stage(0, 0);
    load(0, DEPTH);
    lds_barrier();
    for (int t = 0; t < steps; t += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            // buffer d & 1 holds step t + d; the next step's tile is written beside it, its slot
            // asks for the tile DEPTH steps on, and the products hide both
            const unsigned char* s = smem + (d & 1) * GemmLds<MT>::kStage;
            bf16x8 fw[2], fx[MB];
#pragma unroll
            for (int nh = 0; nh < 2; ++nh)
                fw[nh] = *reinterpret_cast<const bf16x8*>(s + (MT + 32 * nh) * kRowBytes + op);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) fx[mb] = *reinterpret_cast<const bf16x8*>(s + 32 * mb * kRowBytes + op);
            stage((d + 1) % DEPTH, (d + 1) & 1);
            load((d + 1) % DEPTH, t + d + 1 + DEPTH);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int nh = 0; nh < 2; ++nh)
                    acc[mb][nh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[nh], fx[mb], acc[mb][nh], 0, 0, 0);
            lds_barrier();
        }
    }

    // The waves' sums of 32 rows at a time meet in LDS: [wave][row][16 pieces of 4 columns], pieces
    // permuted by the row like the staged tiles; then 8 threads finish one row.
    const int er = tid / 8, ec = tid & 7;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb > 0) lds_barrier();
#pragma unroll
        for (int nh = 0; nh < 2; ++nh)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int r = lane & 31, c = nh * 8 + 2 * g + (lane >> 5);
                const f32x4 v = {acc[mb][nh][4 * g], acc[mb][nh][4 * g + 1], acc[mb][nh][4 * g + 2],
                                 acc[mb][nh][4 * g + 3]};
                *reinterpret_cast<f32x4*>(smem + ((wv * 32 + r) * 16 + (c ^ (r & 7))) * 16) = v;
            }
        lds_barrier();
        const int m = m0 + mb * 32 + er;
        f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f}, c = a;
        // kStoreGelu: 4 gate columns and the up columns beside them; else 8 adjacent columns
        const int pa = EPI == kStoreGelu ? ec : 2 * ec, pc = EPI == kStoreGelu ? 8 + ec : 2 * ec + 1;
#pragma unroll
        for (int q = 0; q < kWaves; ++q) {
            a += *reinterpret_cast<const f32x4*>(smem + ((q * 32 + er) * 16 + (pa ^ (er & 7))) * 16);
            c += *reinterpret_cast<const f32x4*>(smem + ((q * 32 + er) * 16 + (pc ^ (er & 7))) * 16);
        }
        const int n = n0 + (EPI == kStoreGelu ? 4 : 8) * ec;
        if (m < M && n < N) {
            store_columns<EPI>(out, a, c, split, m, n, M, N);
        }
    }
}

// The same products for more than 64 rows, in tiles of 128 rows x NT columns.  What sets the pace is how much a
// compute unit can have in flight: loads return in order and no more than about 32 KB of them are outstanding (more
// in the queue changes nothing: a stream from HBM into one compute unit of 64 stays at 47 bytes per ns, from L2 at
// 123), and since a quarter to a half of a tile's bytes are weights that HBM takes 0.7 us to deliver, all of them
// arrive at that pace.  So the tile is as square as the number of workgroups allows, and tiles go from memory into
// LDS without passing through registers, a few steps ahead, one barrier a step.  Eight waves split the tile
// (2 x 4, or 4 x 2 of 64 columns); each sums all of a workgroup's K in order.  256 x 15360 x 2560 takes 34.7 us (36.6 through registers with four
// waves; 35 without any products, 24 with the weights alone), 256 x 5120 x 2560 17.7 (20.4), 129 x 15360 x 2560 29.3
// (32.7), 65 x 32000 x 512 10.0 (12.2); where each workgroup starts along K makes no difference.
//
// STAGES tiles of a step are held: four where no compute unit has a second workgroup; where there are more workgroups
// than compute units two share one, and the tiles held are what both have room for, three of 64 columns or two of
// 128 (256 x 32000 x 512 in us: 17.6 with four, 15.7 with two; with no second workgroup, 256 x 15360 x 2560, 35.5
// with four, 35.7 with three, 45.5 with two).
template <int NT, int STAGES>
struct WideLds {
    static constexpr int kGroups = (128 + NT) / 8;             // wave loads of 8 rows x 128 bytes per step
    static constexpr int kStage = (128 + NT) * kRowBytes;
    static constexpr int kSums = 128 * NT * 4;                 // the tile on its way out
    static constexpr int kBytes = STAGES * kStage > kSums ? STAGES * kStage : kSums;
};
constexpr int kWideWaves = 8;
constexpr int kWideThreads = kWideWaves * kWave;

template <int NT, int STAGES, int EPI>
__global__ __launch_bounds__(kWideThreads, STAGES == 4 ? 2 : 4) void decode_gemm_wide_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int M, int N, int K,
    int ntiles, int mtiles, int splits) {
    constexpr int MT = 128;
    constexpr int WN = NT / 32, WM = kWideWaves / WN, MB = MT / WM / 32;    // waves side by side, and blocks of 32 rows of one
    constexpr int NC = EPI == kStoreGelu ? NT / 2 : NT;       // output columns of a tile
    using Lds = WideLds<NT, STAGES>;
    constexpr int S = STAGES, L = Lds::kGroups / kWideWaves;
    __shared__ __align__(16) unsigned char smem[Lds::kBytes];

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wm = wv % WM, wn = wv / WM;

    // row tiles of one weight tile 8 workgroups apart, as above
    const int b = (int)blockIdx.x;
    const int group = b / (8 * mtiles), in_group = b - group * 8 * mtiles;
    const int item = group * 8 + (in_group & 7);
    if (item >= ntiles * splits) return;
    const int split = item / ntiles;
    const int nt = item - split * ntiles;
    const int m0 = in_group / 8 * MT, n0 = nt * NC;

    const int pairs = K / (2 * kKT);          // this split's share of K, in pairs of steps
    const int step0 = 2 * (int)((long long)pairs * split / splits);
    const int steps = 2 * (int)((long long)pairs * (split + 1) / splits) - step0;
    const uint32_t row_bytes = (uint32_t)K * 2u;
    const uint32_t k_bytes0 = (uint32_t)step0 * kRowBytes;

    // A load brings 8 rows of 128 bytes, lane by lane one behind the other; the permutation of a row's pieces is
    // in the address a lane reads from.  Rows past the last repeat it: their results are not stored.
    const rsrc_t bx = make_rsrc(x + (size_t)m0 * K, (uint32_t)min(MT, M - m0) * row_bytes);
    const int ncols = min(NC, N - n0);
    const rsrc_t bw = make_rsrc(w + (size_t)n0 * K, (uint32_t)ncols * row_bytes);
    const rsrc_t bup = make_rsrc(EPI == kStoreGelu ? w + (size_t)(N + n0) * K : w, (uint32_t)ncols * row_bytes);
    const uint32_t piece = (uint32_t)(((lane & 7) ^ (lane >> 3)) << 4);
    uint32_t at[L];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        const int g = wv + l * kWideWaves;                    // groups 0..15 are rows of x
        int row = (l < 2 ? g : g - 16) * 8 + (lane >> 3);
        if (EPI == kStoreGelu && row >= NC && l >= 2) row -= NC;
        row = min(row, (l < 2 ? min(MT, M - m0) : ncols) - 1);
        at[l] = (uint32_t)row * row_bytes + piece;
    }
    auto load = [&](int slot, int step) {
        const uint32_t k = k_bytes0 + (uint32_t)step * kRowBytes;
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const int g = wv + l * kWideWaves;
            const bool up = EPI == kStoreGelu && l >= 2 && (g - 16) * 8 >= NC;
            load_to_lds(l < 2 ? bx : (up ? bup : bw), smem + slot * Lds::kStage + g * 1024, at[l], k);
        }
    };

    f32x16 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][i] = 0.0f;

    const int xrow = wm * (MT / WM) + (lane & 31), wrow = MT + wn * 32 + (lane & 31);
    auto multiply = [&](int slot) {
        const unsigned char* s = smem + slot * Lds::kStage;
        bf16x8 fx[kKT / 16][MB], fw[kKT / 16];
#pragma unroll
        for (int ks = 0; ks < kKT / 16; ++ks) {
            const int c = 2 * ks + (lane >> 5);
            fw[ks] = *reinterpret_cast<const bf16x8*>(s + piece_offset(wrow, c));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                fx[ks][mb] = *reinterpret_cast<const bf16x8*>(s + piece_offset(xrow + 32 * mb, c));
        }
#pragma unroll
        for (int ks = 0; ks < kKT / 16; ++ks)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[ks], fx[ks][mb], acc[mb], 0, 0, 0);
    };

    // Step i: its tile has arrived when at most S - 2 younger ones are in flight; behind the barrier everyone's part
    // has, and everyone is done with the tile of step i - 1, whose place the tile of step i + S - 1 takes.
#pragma unroll
    for (int d = 0; d < S - 1; ++d)
        if (d < steps) load(d, d);
    int i = 0, slot = 0;
    for (; i + S - 1 < steps; ++i) {
        wait_vector_memory<(S - 2) * L>();
        lds_barrier();
        load(slot == 0 ? S - 1 : slot - 1, i + S - 1);
        multiply(slot);
        slot = slot == S - 1 ? 0 : slot + 1;
    }
    for (; i < steps; ++i) {
        switch (steps - 1 - i) {
            case 0: wait_vector_memory<0>(); break;
            case 1: wait_vector_memory<L>(); break;
            default: wait_vector_memory<2 * L>(); break;       // (no more than S - 2 = 2)
        }
        lds_barrier();
        multiply(slot);
        slot = slot == S - 1 ? 0 : slot + 1;
    }
    lds_barrier();

    // the tile through LDS, [128 rows][NT / 4 pieces of 4 columns] with the pieces permuted by the row,
    // so that it leaves in whole rows
    constexpr int PR = NT / 4;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int r = wm * (MT / WM) + mb * 32 + (lane & 31);
            const int c = wn * 8 + 2 * g + (lane >> 5);
            const f32x4 v = {acc[mb][4 * g], acc[mb][4 * g + 1], acc[mb][4 * g + 2], acc[mb][4 * g + 3]};
            *reinterpret_cast<f32x4*>(smem + (r * PR + (c ^ (r & 7))) * 16) = v;
        }
    lds_barrier();
    constexpr int CPT = EPI == kStoreGelu ? 4 : 8;            // output columns per thread
    constexpr int TPR = NC / CPT;                             // threads per row
    const int ec = tid % TPR;
    const int n = n0 + CPT * ec;
#pragma unroll
    for (int r = tid / TPR; r < MT; r += kWideThreads / TPR) {
        const int m = m0 + r;
        const int pa = EPI == kStoreGelu ? ec : 2 * ec, pc = EPI == kStoreGelu ? PR / 2 + ec : 2 * ec + 1;
        const f32x4 a = *reinterpret_cast<const f32x4*>(smem + (r * PR + (pa ^ (r & 7))) * 16);
        const f32x4 c = *reinterpret_cast<const f32x4*>(smem + (r * PR + (pc ^ (r & 7))) * 16);
        if (m < M && n < N) store_columns<EPI>(out, a, c, split, m, n, M, N);
    }
}

// out = the sum of S partial sums [S, n], rounded once: the last step of a product split over K whose
// output is read as bf16.
template <int S>
__global__ __launch_bounds__(256) void sum_partial_kernel(const float* __restrict__ partial, bf16_t* __restrict__ out,
                                                          size_t n) {
    const size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (at >= n) return;
    f32x4 part[S][2];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        part[s][0] = *reinterpret_cast<const f32x4*>(partial + s * n + at);
        part[s][1] = *reinterpret_cast<const f32x4*>(partial + s * n + at + 4);
    }
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        v[k] = part[0][k / 4][k % 4];
#pragma unroll
        for (int s = 1; s < S; ++s) v[k] += part[s][k / 4][k % 4];
    }
    u32x4 r;
    pack(v, r);
    *reinterpret_cast<u32x4*>(out + at) = r;
}

int sum_partial(const float* partial, int splits, void* out, size_t n, hipStream_t st) {
    const dim3 grid((unsigned)((n / 8 + 255) / 256));
    bf16_t* o = static_cast<bf16_t*>(out);
    switch (splits) {
#define HAWK_SUM(S) \
    case S: hipLaunchKernelGGL((sum_partial_kernel<S>), grid, dim3(256), 0, st, partial, o, n); break;
        HAWK_SUM(2) HAWK_SUM(3) HAWK_SUM(4) HAWK_SUM(5) HAWK_SUM(6) HAWK_SUM(7) HAWK_SUM(8)
#undef HAWK_SUM
        default: return HAWK_ERR_BAD_SHAPE;
    }
    return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH;
}

// hidden += the sum of S partial sums, then out = hidden / rms(hidden) * weight; the sum, the new hidden
// state and the result are each rounded to bf16 once, as the separate operations round them
// (hawk/hawk.py:53-58, :236-241).  One workgroup per row, 8 channels per thread: latency is all it
// costs, so every load of a thread is in flight before the first is used (S is a template
// parameter for that: with a loop over the partial sums their round trips added up, 7.8 against
// 4.9 us at 128 rows of 2560 and 8 of them).
constexpr int kNormMaxThreads = 1024;

template <int S>
__global__ __launch_bounds__(kNormMaxThreads) void add_norm_kernel(bf16_t* __restrict__ hidden,
                                                                   const float* __restrict__ partial,
                                                                   const bf16_t* __restrict__ weight, float eps,
                                                                   bf16_t* __restrict__ out, int M, int D) {
    __shared__ float s_sum[kNormMaxThreads / kWave];
    const int m = (int)blockIdx.x, c = 8 * (int)threadIdx.x;
    const bool on = c < D;
    const size_t at = (size_t)m * D + (on ? c : 0);
    const u32x4 h = load_raw<bf16_t, 8>(hidden + at);
    const u32x4 wraw = load_raw<bf16_t, 8>(weight + (on ? c : 0));
    f32x4 part[S > 0 ? S : 1][2];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const float* p = partial + (size_t)s * M * D + at;
        part[s][0] = *reinterpret_cast<const f32x4*>(p);
        part[s][1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
    float v[8], sq = 0.0f;
    unpack(h, v);
    if constexpr (S > 0) {
        float add[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            add[k] = part[0][k / 4][k % 4];
#pragma unroll
            for (int s = 1; s < S; ++s) add[k] += part[s][k / 4][k % 4];
        }
        u32x4 r;
        pack(add, r);        // rounded where a separate projection rounds its output
        unpack(r, add);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] += add[k];
        pack(v, r);
        if (on) *reinterpret_cast<u32x4*>(hidden + at) = r;
        unpack(r, v);     // the norm sees the hidden state as it is kept
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) sq = fmaf(v[k], v[k], sq);
    if (!on) sq = 0.0f;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
    if ((threadIdx.x & (kWave - 1)) == 0) s_sum[threadIdx.x / kWave] = sq;
    __syncthreads();
    float total = 0.0f;
    for (int k = 0; k < (int)blockDim.x / kWave; ++k) total += s_sum[k];
    const float scale = 1.0f / sqrtf(total / (float)D + eps);
    float g[8];
    unpack(wraw, g);
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] *= v[k] * scale;
    u32x4 r;
    pack(g, r);
    if (on) *reinterpret_cast<u32x4*>(out + at) = r;
}

int add_norm(void* hidden, const float* partial, int splits, const void* weight, float eps, void* out, int M, int D,
             hipStream_t st) {
    const dim3 grid((unsigned)M), block((unsigned)(ceil_div(D / 8, kWave) * kWave));
    bf16_t* h = static_cast<bf16_t*>(hidden);
    const bf16_t* w = static_cast<const bf16_t*>(weight);
    bf16_t* o = static_cast<bf16_t*>(out);
    switch (splits) {
#define HAWK_NORM(S) \
    case S: hipLaunchKernelGGL((add_norm_kernel<S>), grid, block, 0, st, h, partial, w, eps, o, M, D); break;
        HAWK_NORM(0) HAWK_NORM(1) HAWK_NORM(2) HAWK_NORM(3) HAWK_NORM(4) HAWK_NORM(5) HAWK_NORM(6) HAWK_NORM(7) HAWK_NORM(8)
#undef HAWK_NORM
        default: return HAWK_ERR_BAD_SHAPE;
    }
    return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------------------
// Products for one or two rows, where a launch's duration is a few memory round trips and not its bytes: a wave takes
// C weight rows at a time, a lane 16 bytes of each per 512 input channels, and the sums meet in a butterfly over the
// lanes.  No LDS tile, no loop of staged steps, and the norm in front needs no launch of its own: every workgroup
// repeats residual add and norm of the few rows into its LDS while its first weights are on their way.
//   kNoNorm     x [M, K] bf16
//   kNorm       x = norm(hidden)
//   kAddNorm    x = norm(hidden + delta), delta [M, K] fp32; the first workgroup writes the sum to hidden_out, which
//               is not hidden: the others may still be reading that
// Values are rounded, and squares added up, as in add_norm_kernel.  out as for decode_gemm_kernel, kStorePartial with
// one split.
// A layer's four products and two norms at one row, against the tiles and add_norm_kernel: 13.8 us (21.9) at 512
// channels and an MLP of 1024, 18.6 (29.4) at 1024 and 3072, 45.4 (49.5) at 2560 and 7680 (157 MB, 32 us at the rate
// of a large copy); a product by itself 7.6 us (9.8) for 5120 x 2560, 31.6 (32.2) for 32000 x 2560.
// ---------------------------------------------------------------------------------------
enum Front { kNoNorm = 0, kNorm = 1, kAddNorm = 2 };
constexpr int kRowsMax = 2;
// Two rows' arithmetic (16 multiply-adds beside 8 conversions a load, on the vector units) is no longer hidden behind
// the loads of a large matrix: 5120 x 2560 takes 8.2 us here and 9.9 in tiles, 2560 x 7680 12.8 and 12.4, 32000 x 512
// 9.9 and 8.3.  At four rows already 5120 x 2560 has little left (9.4), a layer of 2560 loses (68 to 50).
constexpr size_t kRowsTwoWeights = 14 << 20;
constexpr int kRowsFourFrom = 4096;
constexpr int kRowsBlocks = 1024;                  // (512 and 2048 measure the same)
constexpr int kChunk = 8 * kWave;                  // input channels a wave's lanes cover with one load each

struct NormArgs {
    const bf16_t* hidden;
    const float* delta;
    const bf16_t* weight;
    float eps;
    bf16_t* hidden_out;
};

template <int MR, int C, int EPI, int FRONT>
__global__ __launch_bounds__(kThreads) void decode_rows_kernel(const bf16_t* __restrict__ x, NormArgs norm,
                                                               const bf16_t* __restrict__ w, void* __restrict__ out,
                                                               int M, int N, int K) {
    // loads of a lane in flight: eight of weights, or twelve with those of x
    constexpr int kUnroll = FRONT != kNoNorm ? 8 / C : 12 / (C + MR);
    constexpr int kOut = EPI == kStoreGelu ? C / 2 : C;   // output columns of a wave
    extern __shared__ __align__(16) unsigned char smem[];  // FRONT: x, bf16 [MR][K]
    __shared__ float s_sq[MR][kNormMaxThreads / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t row_bytes = (uint32_t)K * 2u;
    const int units = (N + kOut - 1) / kOut, stride = (int)gridDim.x * kWaves;
    int unit = (int)blockIdx.x * kWaves + wv;

    u32x4 rw[kUnroll][C], rx[kUnroll][MR];
    // weights of `unit`, and x, from input channel k0 on; zeros past K and past N
    auto load = [&](int u, int k0) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int n = u * kOut + c % kOut;
            const size_t row = EPI == kStoreGelu && c >= kOut ? (size_t)N + n : (size_t)n;
            const rsrc_t r = make_rsrc(w + (n < N ? row : 0) * K, u < units && n < N ? row_bytes : 0u);
#pragma unroll
            for (int q = 0; q < kUnroll; ++q)
                rw[q][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                         r, (uint32_t)(k0 + q * kChunk + 8 * lane) * 2u, 0, kAuxDefault));
        }
        if constexpr (FRONT == kNoNorm) {
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const rsrc_t r = make_rsrc(x + (size_t)min(m, M - 1) * K, row_bytes);
#pragma unroll
                for (int q = 0; q < kUnroll; ++q)
                    rx[q][m] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                             r, (uint32_t)(k0 + q * kChunk + 8 * lane) * 2u, 0, kAuxDefault));
            }
        }
    };
    load(unit, 0);
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (FRONT != kNoNorm) {
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const int row = min(m, M - 1);
            for (int k0 = 0; k0 < K; k0 += 8 * kThreads) {   // (sums per 512 channels, in add_norm_kernel's order)
                const int k = k0 + 8 * tid;
                float sq = 0.0f;
                if (k < K) {
                    const size_t at = (size_t)row * K + k;
                    u32x4 r = load_raw<bf16_t, 8>(norm.hidden + at);
                    float v[8];
                    unpack(r, v);
                    if constexpr (FRONT == kAddNorm) {
                        const f32x4 d0 = *reinterpret_cast<const f32x4*>(norm.delta + at);
                        const f32x4 d1 = *reinterpret_cast<const f32x4*>(norm.delta + at + 4);
                        float add[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
                        pack(add, r);                  // rounded where a separate projection rounds its output
                        unpack(r, add);
#pragma unroll
                        for (int i = 0; i < 8; ++i) v[i] += add[i];
                        pack(v, r);
                        if (blockIdx.x == 0 && m < M) *reinterpret_cast<u32x4*>(norm.hidden_out + at) = r;
                        unpack(r, v);                  // the norm sees the hidden state as it is kept
                    }
                    *reinterpret_cast<u32x4*>(smem + (size_t)m * row_bytes + 2 * k) = r;
#pragma unroll
                    for (int i = 0; i < 8; ++i) sq = fmaf(v[i], v[i], sq);
                }
#pragma unroll
                for (int o = kWave / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
                if (lane == 0) s_sq[m][k0 / kChunk + wv] = sq;
            }
        }
        lds_barrier();
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float total = 0.0f;
            for (int q = 0; q < ceil_div(K, kChunk); ++q) total += s_sq[m][q];
            const float scale = 1.0f / sqrtf(total / (float)K + norm.eps);
            for (int k = 8 * tid; k < K; k += 8 * kThreads) {
                u32x4* p = reinterpret_cast<u32x4*>(smem + (size_t)m * row_bytes + 2 * k);
                float v[8], g[8];
                unpack(*p, v);
                unpack(load_raw<bf16_t, 8>(norm.weight + k), g);
#pragma unroll
                for (int i = 0; i < 8; ++i) g[i] *= v[i] * scale;
                pack(g, *p);
            }
        }
        lds_barrier();
    }

    for (; unit < units; unit += stride) {
        float acc[C][MR];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int m = 0; m < MR; ++m) acc[c][m] = 0.0f;
        for (int k0 = 0; k0 < K; k0 += kUnroll * kChunk) {
            u32x4 cw[kUnroll][C], cx[kUnroll][MR];
#pragma unroll
            for (int q = 0; q < kUnroll; ++q) {
#pragma unroll
                for (int c = 0; c < C; ++c) cw[q][c] = rw[q][c];
#pragma unroll
                for (int m = 0; m < MR; ++m)
                    if constexpr (FRONT == kNoNorm) cx[q][m] = rx[q][m];
            }
            const bool last = k0 + kUnroll * kChunk >= K;
            load(last ? unit + stride : unit, last ? 0 : k0 + kUnroll * kChunk);
#pragma unroll
            for (int q = 0; q < kUnroll; ++q) {
                const int k = k0 + q * kChunk + 8 * lane;
                if (k0 + q * kChunk >= K) break;   // (the same in every lane)
                float xv[MR][8];
#pragma unroll
                for (int m = 0; m < MR; ++m) {
                    if constexpr (FRONT == kNoNorm) {
                        unpack(cx[q][m], xv[m]);
                    } else {
                        u32x4 r = {0u, 0u, 0u, 0u};
                        if (k < K) r = *reinterpret_cast<const u32x4*>(smem + (size_t)m * row_bytes + 2 * k);
                        unpack(r, xv[m]);
                    }
                }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    float wf[8];
                    unpack(cw[q][c], wf);
#pragma unroll
                    for (int m = 0; m < MR; ++m)
#pragma unroll
                        for (int i = 0; i < 8; ++i) acc[c][m] = fmaf(wf[i], xv[m][i], acc[c][m]);
                }
            }
        }
        // lane c MR + m finishes output column c of row m
        float mine = 0.0f, up = 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                float v = acc[c][m];
#pragma unroll
                for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
                if (lane == (c % kOut) * MR + m) {
                    if (c < kOut) mine = v;
                    else up = v;
                }
            }
        const int n = unit * kOut + lane / MR, m = lane % MR;
        if (lane < kOut * MR && n < N && m < M) {
            if constexpr (EPI == kStorePartial) {
                static_cast<float*>(out)[(size_t)m * N + n] = mine;
            } else {
                float r = mine;
                if constexpr (EPI == kStoreGelu) {
                    const uint32_t projected = pack_bf16x2(mine, up);
                    const float g = gelu_times(bf16_lo(projected), 1.0f);
                    r = bf16_lo(pack_bf16x2(g, g)) * bf16_hi(projected);
                }
                const uint32_t b = pack_bf16x2(r, r);
                reinterpret_cast<unsigned short*>(out)[(size_t)m * N + n] = (unsigned short)b;
            }
        }
    }
}

inline bool takes_rows(int M, int N, int K) {
    return M == 1 || (M <= kRowsMax && (size_t)N * K <= kRowsTwoWeights);
}

// Workgroups: a wave per C weight rows, C two where four would leave compute units without a wave each.
template <int EPI, int FRONT>
int rows_product(const void* x, const NormArgs& norm, const void* w, void* out, int M, int N, int K, hipStream_t st) {
    const int cols = EPI == kStoreGelu ? 2 * N : N;
    const bool four = cols > kRowsFourFrom;        // four: a wave per SIMD of the chip
    const int units = ceil_div(cols, four ? 4 : 2);
    int blocks = ceil_div(units, kWaves);
    if (blocks > kRowsBlocks) blocks = kRowsBlocks;
    const size_t lds = FRONT == kNoNorm ? 0 : (size_t)M * K * 2;
    const bf16_t* xp = static_cast<const bf16_t*>(x);
    const bf16_t* wp = static_cast<const bf16_t*>(w);
#define HAWK_ROWS(MR)                                                                                               \
    if (four)                                                                                                       \
        hipLaunchKernelGGL((decode_rows_kernel<MR, 4, EPI, FRONT>), dim3((unsigned)blocks), dim3(kThreads), lds, st, xp, \
                           norm, wp, out, M, N, K);                                                                 \
    else                                                                                                            \
        hipLaunchKernelGGL((decode_rows_kernel<MR, 2, EPI, FRONT>), dim3((unsigned)blocks), dim3(kThreads), lds, st, xp, \
                           norm, wp, out, M, N, K)
    if (M == 1) { HAWK_ROWS(1); }
    else { HAWK_ROWS(2); }
#undef HAWK_ROWS
    return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH;
}

// How a product is cut: rows and columns of a tile, tiles in flight, workgroups along K.
struct Cut {
    int mt, nt, depth, splits;
};
// Workgroups a product that is split over K is cut into: one per compute unit.  A layer of 2560 channels (MLP 7680;
// 240 to 266 are the same cuts there) takes 49 / 53 / 64 / 78 / 83 / 98 us at 3 / 32 / 64 / 128 / 129 / 256 rows, with 320
// workgroups 53 / 60 / 73 / 91 / 93 / 119 (the partial sums of more splits cost more than the second workgroup on a
// compute unit brings), with 160 50 / 56 / 68 / 81 / 88 / 106.  With 240 the 128 tiles of 4096 columns at 129 rows and more,
// and of 8192 at 33 to 128, are not split and half of the chip is idle: a layer of 4096 (MLP 12288) takes 199 and 231 us
// at 129 and 256 rows, in two splits 171 and 190, one of 8192 (MLP 24576) 400 / 436 / 512 at 33 / 64 / 128, in two splits
// 356 / 381 / 452.  From 129 tiles on one split stays: 160 tiles over K = 2560 in two take 2 % more of a layer's time.
constexpr int kComputeUnits = 256;
constexpr int kSplitWorkgroups = kComputeUnits;
// Tiles of 128 x 128 from this many of them on; with fewer, part of the chip would be idle.
constexpr int kMinWideTiles = 200;

Cut cut_for(int M, int N, int K, bool gelu, bool may_split) {
    Cut c;
    c.mt = M <= 32 ? 32 : (M <= 64 ? 64 : 128);
    c.nt = kNT;
    c.depth = K % (4 * kKT) == 0 ? 4 : 2;
    c.splits = 1;
    const int mtiles = ceil_div(M, c.mt), cols = gelu ? 2 * N : N;
    if (c.mt == 128) {
        // (split products keep 64 columns: in 128-wide tiles and as many workgroups 256 x 2560 x 7680 takes 22.0 us
        // instead of 24.5, which twice the partial sums cost the norm behind it, 256 x 2560 x 2560 11.8 instead of
        // 11.1, 256 x 5120 x 2560 15.7 and a launch for its sums instead of 17.4)
        if (!may_split && ceil_div(cols, 128) * mtiles >= kMinWideTiles) c.nt = 128;
        else c.depth = 2;
    }
    if (may_split) {
        const int tiles = ceil_div(cols, c.nt) * mtiles, turns = K / (c.depth * kKT);
        int s = kSplitWorkgroups / tiles;
        if (s > kDecodeMaxSplits) s = kDecodeMaxSplits;
        if (s > turns / 2) s = turns / 2;    // shorter loops are all filling of the pipeline
        c.splits = s < 1 ? 1 : s;
    }
    return c;
}

template <int EPI>
int gemm(const void* x, const void* w, void* out, int M, int N, int K, const Cut& c, hipStream_t st) {
    const int ntiles = ceil_div(N, EPI == kStoreGelu ? c.nt / 2 : c.nt), mtiles = ceil_div(M, c.mt);
    const dim3 grid((unsigned)(ceil_div(ntiles * c.splits, 8) * 8 * mtiles));
    const bf16_t* xp = static_cast<const bf16_t*>(x);
    const bf16_t* wp = static_cast<const bf16_t*>(w);
#define HAWK_GEMM(THREADS, ...)                                                                                \
    hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(THREADS), 0, st, xp, wp, out, M, N, K, ntiles, mtiles, c.splits)
    if (c.mt == 32) {
        if (c.depth == 4) HAWK_GEMM(kThreads, decode_gemm_kernel<32, 4, EPI>);
        else HAWK_GEMM(kThreads, decode_gemm_kernel<32, 2, EPI>);
    } else if (c.mt == 64) {
        if (c.depth == 4) HAWK_GEMM(kThreads, decode_gemm_kernel<64, 4, EPI>);
        else HAWK_GEMM(kThreads, decode_gemm_kernel<64, 2, EPI>);
    } else if (c.nt == 64) {
        if (ntiles * c.splits * mtiles <= kComputeUnits) HAWK_GEMM(kWideThreads, decode_gemm_wide_kernel<64, 4, EPI>);
        else HAWK_GEMM(kWideThreads, decode_gemm_wide_kernel<64, 3, EPI>);
    } else {
        if (ntiles * c.splits * mtiles <= kComputeUnits) HAWK_GEMM(kWideThreads, decode_gemm_wide_kernel<128, 4, EPI>);
        else HAWK_GEMM(kWideThreads, decode_gemm_wide_kernel<128, 2, EPI>);
    }
#undef HAWK_GEMM
    return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH;
}

}  // namespace

bool decode_linear_supported(int M, int N, int K) {
    return M >= 1 && M <= kDecodeMaxRows && N >= 8 && N % 8 == 0 && N <= (1 << 20) && K >= 2 * kKT &&
           K % (2 * kKT) == 0 && K <= 65536;
}
bool decode_norm_supported(int D) { return D >= 8 && D % 8 == 0 && D <= 8 * kNormMaxThreads; }

size_t decode_linear_workspace_bytes(int M, int N, int K) {
    const Cut c = cut_for(M, N, K, false, true);
    return c.splits > 1 ? (size_t)c.splits * M * N * sizeof(float) : 0;
}

// The workspace of a layer: normed rows, the MLP's product, partial sums.
size_t decode_layer_workspace_bytes(int M, int H, int R, int I, int n_next) {
    const size_t a = (size_t)cut_for(M, H, R, false, true).splits * H, b = (size_t)cut_for(M, H, I, false, true).splits * H;
    const size_t sums = (a > b ? a : b) * M * sizeof(float), next = decode_linear_workspace_bytes(M, n_next, H);
    return align256((size_t)M * H * 2) + align256((size_t)M * I * 2) + align256(sums > next ? sums : next);
}

int decode_linear(const void* x, const void* w, void* out, int M, int N, int K, void* ws, hipStream_t st) {
    if (takes_rows(M, N, K)) return rows_product<kStoreBf16, kNoNorm>(x, NormArgs{}, w, out, M, N, K, st);
    const Cut c = cut_for(M, N, K, false, true);
    if (c.splits == 1) return gemm<kStoreBf16>(x, w, out, M, N, K, cut_for(M, N, K, false, false), st);
    if (int rc = gemm<kStorePartial>(x, w, ws, M, N, K, c, st)) return rc;
    return sum_partial(static_cast<const float*>(ws), c.splits, out, (size_t)M * N, st);
}

int decode_norm_linear(void* hidden, const void* norm_w, float eps, const void* w, void* out, int M, int N, int H,
                       void* ws, hipStream_t st) {
    if (takes_rows(M, N, H)) {
        const NormArgs norm{static_cast<const bf16_t*>(hidden), nullptr, static_cast<const bf16_t*>(norm_w), eps, nullptr};
        return rows_product<kStoreBf16, kNorm>(nullptr, norm, w, out, M, N, H, st);
    }
    if (int rc = add_norm(hidden, nullptr, 0, norm_w, eps, ws, M, H, st)) return rc;
    return decode_linear(ws, w, out, M, N, H, static_cast<char*>(ws) + align256((size_t)M * H * 2), st);
}

int decode_layer_tail(const void* gated, const void* w_resid, void* hidden, const void* norm_w, float eps,
                      const void* w_gate_up, const void* w_down, const void* next_norm_w, float next_eps,
                      const void* w_next, void* next_out, int M, int H, int R, int I, int n_next, void* ws,
                      hipStream_t st) {
    char* p = static_cast<char*>(ws);
    void* normed = p;
    void* act = p + align256((size_t)M * H * 2);
    float* partial = reinterpret_cast<float*>(p + align256((size_t)M * H * 2) + align256((size_t)M * I * 2));
    if (takes_rows(M, H, R) && takes_rows(M, 2 * I, H) && takes_rows(M, H, I) && takes_rows(M, n_next, H)) {
        // the hidden state between the two norms lies where the wider step keeps its normed rows
        const NormArgs first{static_cast<const bf16_t*>(hidden), partial, static_cast<const bf16_t*>(norm_w), eps,
                             static_cast<bf16_t*>(normed)};
        const NormArgs second{static_cast<const bf16_t*>(normed), partial, static_cast<const bf16_t*>(next_norm_w),
                              next_eps, static_cast<bf16_t*>(hidden)};
        if (int rc = rows_product<kStorePartial, kNoNorm>(gated, NormArgs{}, w_resid, partial, M, H, R, st)) return rc;
        if (int rc = rows_product<kStoreGelu, kAddNorm>(nullptr, first, w_gate_up, act, M, I, H, st)) return rc;
        if (int rc = rows_product<kStorePartial, kNoNorm>(act, NormArgs{}, w_down, partial, M, H, I, st)) return rc;
        return rows_product<kStoreBf16, kAddNorm>(nullptr, second, w_next, next_out, M, n_next, H, st);
    }
    const Cut resid = cut_for(M, H, R, false, true), down = cut_for(M, H, I, false, true);
    if (int rc = gemm<kStorePartial>(gated, w_resid, partial, M, H, R, resid, st)) return rc;
    if (int rc = add_norm(hidden, partial, resid.splits, norm_w, eps, normed, M, H, st)) return rc;
    if (int rc = gemm<kStoreGelu>(normed, w_gate_up, act, M, I, H, cut_for(M, I, H, true, false), st)) return rc;
    if (int rc = gemm<kStorePartial>(act, w_down, partial, M, H, I, down, st)) return rc;
    if (int rc = add_norm(hidden, partial, down.splits, next_norm_w, next_eps, normed, M, H, st)) return rc;
    return decode_linear(normed, w_next, next_out, M, n_next, H, partial, st);
}

}  // namespace hawk
