// What surrounds the recurrent core and the library GEMMs in a training pass of the model
// (hawk/hawk.py:53-58, :70-86, :222-303 upstream): residual add + RMSNorm, the gated GELU, the
// next-token cross entropy, the embedding's gradient and the conversions of weights and weight gradients,
// each as one pass over its tensors per direction.  Arithmetic is fp32; values are rounded to bf16
// where bf16 autocast rounds them.  Every sum has a fixed order.
#include "hawk_scan.h"

#include <stdint.h>

#include "hawk_device.h"
#include "hawk_reduce.h"

namespace hawk {
namespace {

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------------------
// Conversions of up to kCastSegments arrays in one launch: a layer's four weights to bf16 in front of
// its forward, their gradients to fp32 behind its backward.  Bound by memory; a launch each (4 us with
// the gap) is what it spares: 6.5 us for the 2.4 M weights of a layer of 512 x 1024.
// ---------------------------------------------------------------------------------------
constexpr int kCastThreads = 256;
struct CastTask {
    const void* src[kCastSegments];
    void* dst[kCastSegments];
    unsigned long long first_quad[kCastSegments + 1];   // of four elements
    int n;
};

template <bool TO_BF16>
__global__ __launch_bounds__(kCastThreads) void cast_kernel(CastTask t) {
    const unsigned long long step = (unsigned long long)gridDim.x * kCastThreads;
    for (unsigned long long i = (unsigned long long)blockIdx.x * kCastThreads + threadIdx.x; i < t.first_quad[t.n];
         i += step) {
        int s = 0;
        while (i >= t.first_quad[s + 1]) ++s;
        const unsigned long long q = i - t.first_quad[s];
        if constexpr (TO_BF16) {
            const f32x4 v = reinterpret_cast<const f32x4*>(t.src[s])[q];
            reinterpret_cast<u32x2*>(t.dst[s])[q] = u32x2{pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)};
        } else {
            float v[4];
            unpack(reinterpret_cast<const u32x2*>(t.src[s])[q], v);
            reinterpret_cast<f32x4*>(t.dst[s])[q] = f32x4{v[0], v[1], v[2], v[3]};
        }
    }
}

// ---------------------------------------------------------------------------------------
// Residual add + RMSNorm.  A wave owns a row, so its sum is a few shuffles and rows need no barrier; a lane
// owns Q groups of 8 adjacent channels (16 bytes of bf16).  Memory and, at a few thousand rows,
// latency bound.  2048 rows of 512: forward 5.2 us (add, norm and conversion to bf16 apart 12.8),
// backward 6.2 + 3.0 for the weight's sums (conversion, two norm kernels, weight sums and add apart 25).
// ---------------------------------------------------------------------------------------
constexpr int kNormWaves = 4;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int k = 0; k < 4; ++k) { v[k] = a[k]; v[4 + k] = b[k]; }
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4*>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}

// sum = hidden + delta (stored if delta is there), out = sum rstd weight with rstd = 1 / rms(sum)
template <int Q>
__global__ __launch_bounds__(kNormWaves* kWave) void add_norm_fwd_kernel(
    const float* __restrict__ hidden, const bf16_t* __restrict__ delta, const float* __restrict__ weight, float eps,
    float* __restrict__ sum, bf16_t* __restrict__ out, float* __restrict__ rstd, int rows, int D) {
    const int lane = threadIdx.x & (kWave - 1);
    const int row = (int)blockIdx.x * kNormWaves + (int)(threadIdx.x / kWave);
    if (row >= rows) return;
    const size_t base = (size_t)row * D;
    float x[Q][8], sq = 0.0f;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = 8 * (lane + q * kWave);
        if (c < D) {
            load8(hidden + base + c, x[q]);
            if (delta != nullptr) {
                float d[8];
                unpack(load_raw<bf16_t, 8>(delta + base + c), d);
#pragma unroll
                for (int k = 0; k < 8; ++k) x[q][k] += d[k];
                store8(sum + base + c, x[q]);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) sq = fmaf(x[q][k], x[q][k], sq);
        }
    }
    const float r = 1.0f / sqrtf(wave_sum(sq) / (float)D + eps);
    if (lane == 0) rstd[row] = r;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = 8 * (lane + q * kWave);
        if (c < D) {
            float w[8];
            load8(weight + c, w);
#pragma unroll
            for (int k = 0; k < 8; ++k) w[k] *= x[q][k] * r;
            u32x4 p;
            pack(w, p);
            *reinterpret_cast<u32x4*>(out + base + c) = p;
        }
    }
}

// d_sum = d_direct + rstd (w dy) - x rstd^3 / D sum(w dy x); its bf16 rounding is delta's gradient.
// Each wave takes rows of a fixed stride and keeps its share of dweight = sum(dy x rstd) in registers;
// a workgroup's share goes to part [gridDim.x, D].
template <int Q>
__global__ __launch_bounds__(kNormWaves* kWave) void add_norm_bwd_kernel(
    const bf16_t* __restrict__ dout, const float* __restrict__ x_all, const float* __restrict__ rstd,
    const float* __restrict__ weight, const float* __restrict__ d_direct, float* __restrict__ d_sum,
    bf16_t* __restrict__ d_delta, float* __restrict__ part, int rows, int D) {
    extern __shared__ float s_dw[];   // [kNormWaves][D]
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = threadIdx.x / kWave;
    float w[Q][8], dw[Q][8];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = 8 * (lane + q * kWave);
#pragma unroll
        for (int k = 0; k < 8; ++k) { w[q][k] = 0.0f; dw[q][k] = 0.0f; }
        if (c < D) load8(weight + c, w[q]);
    }
    for (int row = (int)blockIdx.x * kNormWaves + wv; row < rows; row += (int)gridDim.x * kNormWaves) {
        const size_t base = (size_t)row * D;
        const float r = rstd[row];
        float x[Q][8], g[Q][8], dot = 0.0f;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int c = 8 * (lane + q * kWave);
            if (c < D) {
                load8(x_all + base + c, x[q]);
                unpack(load_raw<bf16_t, 8>(dout + base + c), g[q]);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    dw[q][k] = fmaf(g[q][k] * x[q][k], r, dw[q][k]);
                    g[q][k] *= w[q][k];
                    dot = fmaf(g[q][k], x[q][k], dot);
                }
            }
        }
        const float scale = wave_sum(dot) * r * r * r / (float)D;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int c = 8 * (lane + q * kWave);
            if (c < D) {
                float d[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) d[k] = 0.0f;
                if (d_direct != nullptr) load8(d_direct + base + c, d);
#pragma unroll
                for (int k = 0; k < 8; ++k) d[k] += fmaf(g[q][k], r, -x[q][k] * scale);
                store8(d_sum + base + c, d);
                if (d_delta != nullptr) {
                    u32x4 p;
                    pack(d, p);
                    *reinterpret_cast<u32x4*>(d_delta + base + c) = p;
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = 8 * (lane + q * kWave);
        if (c < D) store8(s_dw + wv * D + c, dw[q]);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < D; c += kNormWaves * kWave) {
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < kNormWaves; ++k) v += s_dw[k * D + c];
        part[(size_t)blockIdx.x * D + c] = v;
    }
}

__global__ __launch_bounds__(kColsumThreads) void norm_weight_kernel(ColsumTask t) {
    __shared__ float s[kColsumSlices][kColsumCols];
    colsum_block(t, (int)blockIdx.x, s);
}

// ---------------------------------------------------------------------------------------
// act = gelu(gate) * up on rows [gate, up] of 2 I channels, and its gradient in the same layout, 16 bytes
// per lane and access.  Memory bound: 2048 rows of 2 x 1024 forward 4.8 us (GELU and product apart 13),
// backward 6.3 (two products, GELU gradient and concatenation apart 33).
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gelu_mul_fwd_kernel(const bf16_t* __restrict__ gu, bf16_t* __restrict__ act,
                                                           size_t groups, int per_row) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= groups) return;
    const size_t row = i / per_row;
    const int c = (int)(i - row * per_row) * 8;
    const bf16_t* p = gu + row * 16 * per_row + c;
    float g[8], u[8];
    unpack(load_raw<bf16_t, 8>(p), g);
    unpack(load_raw<bf16_t, 8>(p + 8 * per_row), u);
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] = gelu_times(g[k], 1.0f);
    u32x4 r;
    pack(g, r);          // rounded where the separate GELU rounds
    unpack(r, g);
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] *= u[k];
    pack(g, r);
    *reinterpret_cast<u32x4*>(act + i * 8) = r;
}

__global__ __launch_bounds__(256) void gelu_mul_bwd_kernel(const bf16_t* __restrict__ gu,
                                                           const bf16_t* __restrict__ dact, bf16_t* __restrict__ dgu,
                                                           size_t groups, int per_row) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= groups) return;
    const size_t row = i / per_row;
    const int c = (int)(i - row * per_row) * 8;
    const size_t at = row * 16 * per_row + c;
    float g[8], u[8], d[8], dg[8], ge[8];
    unpack(load_raw<bf16_t, 8>(gu + at), g);
    unpack(load_raw<bf16_t, 8>(gu + at + 8 * per_row), u);
    unpack(load_raw<bf16_t, 8>(dact + i * 8), d);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float cdf, e;
        normal_cdf<true>(g[k], cdf, e);
        ge[k] = g[k] * cdf;
        dg[k] = fmaf(g[k] * kInvSqrt2Pi, e, cdf);
        u[k] *= d[k];    // the GELU's gradient
    }
    u32x4 r;
    pack(ge, r);
    unpack(r, ge);
    pack(u, r);
    unpack(r, u);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        dg[k] *= u[k];
        ge[k] *= d[k];
    }
    pack(dg, r);
    *reinterpret_cast<u32x4*>(dgu + at) = r;
    pack(ge, r);
    *reinterpret_cast<u32x4*>(dgu + at + 8 * per_row) = r;
}

// ---------------------------------------------------------------------------------------
// Next-token cross entropy on bf16 logits [B T, V]: row (b, t) is scored against labels[b, t + 1], the
// last row of a sequence and rows whose label is -100 count for nothing.  The forward reads the logits
// once (running maximum and sum), the backward reads them once more and writes their gradient; as
// fp32 log-probabilities the same rows were written and read six times over in 32 bits.  A workgroup of 512
// threads per row.  2048 rows of 32000: 46 us forward, 43 backward, 550 us before.  The backward streams at
// 6.1 TB/s; the forward is not bound by memory (2.9 TB/s): a row is two rounds of four loads per thread, with
// the exponentials and the merges of maximum and sum behind each, and a reduction over the workgroup.
// ---------------------------------------------------------------------------------------
constexpr int kCeThreads = 512;
constexpr long long kIgnoreIndex = -100;

__device__ __forceinline__ long long label_of(const long long* labels, int row, int T, int V, bool& counted) {
    const bool last = row % T == T - 1;
    const long long l = last ? kIgnoreIndex : labels[row + 1];
    counted = l != kIgnoreIndex;
    return l;
}

__device__ __forceinline__ void merge(float& m, float& s, float m2, float s2) {
    const float top = fmaxf(m, m2);
    if (top == -INFINITY) {   // nothing but -inf so far (a NaN sum stays one)
        s += s2;
        return;
    }
    s = s * expf(m - top) + s2 * expf(m2 - top);
    m = top;
}

__global__ __launch_bounds__(kCeThreads) void cross_entropy_fwd_kernel(const bf16_t* __restrict__ logits,
                                                                       const long long* __restrict__ labels,
                                                                       float* __restrict__ lse_out,
                                                                       float* __restrict__ loss, int T, int V) {
    __shared__ float s_m[kCeThreads / kWave], s_s[kCeThreads / kWave];
    const int row = (int)blockIdx.x;
    bool counted;
    const long long label = label_of(labels, row, T, V, counted);
    if (!counted) {           // (uniform)
        if (threadIdx.x == 0) { lse_out[row] = 0.0f; loss[row] = 0.0f; }
        return;
    }
    const bf16_t* p = logits + (size_t)row * V;
    float m = -INFINITY, s = 0.0f;
    for (int c0 = 8 * (int)threadIdx.x; c0 < V; c0 += 4 * 8 * kCeThreads) {
        u32x4 raw[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = c0 + q * 8 * kCeThreads;
            if (c < V) raw[q] = load_raw<bf16_t, 8>(p + c);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (c0 + q * 8 * kCeThreads >= V) continue;
            float v[8], top = -INFINITY, sum = 0.0f;
            unpack(raw[q], v);
#pragma unroll
            for (int k = 0; k < 8; ++k) top = fmaxf(top, v[k]);
            const float ref = top == -INFINITY ? 0.0f : top;
#pragma unroll
            for (int k = 0; k < 8; ++k) sum += expf(v[k] - ref);
            merge(m, s, top, sum);
        }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) merge(m, s, __shfl_xor(m, o), __shfl_xor(s, o));
    if ((threadIdx.x & (kWave - 1)) == 0) { s_m[threadIdx.x / kWave] = m; s_s[threadIdx.x / kWave] = s; }
    __syncthreads();
    if (threadIdx.x == 0) {
        m = s_m[0];
        s = s_s[0];
        for (int k = 1; k < kCeThreads / kWave; ++k) merge(m, s, s_m[k], s_s[k]);
        const float lse = m + logf(s);
        lse_out[row] = lse;
        // a label outside the vocabulary scores NaN
        float own = __builtin_nanf("");
        if (label >= 0 && label < V) own = bf16_lo((uint32_t)p[label].bits);
        loss[row] = lse - own;
    }
}

// mean[0] = the mean loss of the counted rows, mean[1] = their number.
__global__ __launch_bounds__(1024) void cross_entropy_mean_kernel(const float* __restrict__ loss,
                                                                  const long long* __restrict__ labels,
                                                                  float* __restrict__ mean, int rows, int T, int V) {
    __shared__ float s_l[16], s_n[16];
    float l = 0.0f, n = 0.0f;
    for (int r = threadIdx.x; r < rows; r += 1024) {
        bool counted;
        label_of(labels, r, T, V, counted);
        l += loss[r];
        n += counted ? 1.0f : 0.0f;
    }
    l = wave_sum(l);
    n = wave_sum(n);
    if ((threadIdx.x & (kWave - 1)) == 0) { s_l[threadIdx.x / kWave] = l; s_n[threadIdx.x / kWave] = n; }
    __syncthreads();
    if (threadIdx.x == 0) {
        l = n = 0.0f;
        for (int k = 0; k < 16; ++k) { l += s_l[k]; n += s_n[k]; }
        mean[0] = l / n;
        mean[1] = n;
    }
}

__global__ __launch_bounds__(kCeThreads) void cross_entropy_bwd_kernel(
    const bf16_t* __restrict__ logits, const long long* __restrict__ labels, const float* __restrict__ lse_all,
    const float* __restrict__ mean, const float* __restrict__ dloss, bf16_t* __restrict__ dlogits, int T, int V) {
    const int row = (int)blockIdx.x;
    bool counted;
    const long long label = label_of(labels, row, T, V, counted);
    const bf16_t* p = logits + (size_t)row * V;
    bf16_t* o = dlogits + (size_t)row * V;
    // a label outside the vocabulary has no loss (NaN, as the forward says) and so no gradient either
    const bool known = label >= 0 && label < V;
    const float g = !counted ? 0.0f : known ? dloss[0] / mean[1] : __builtin_nanf("");
    const float lse = lse_all[row];
    for (int c = 8 * (int)threadIdx.x; c < V; c += 8 * kCeThreads) {
        u32x4 r = {0u, 0u, 0u, 0u};
        if (counted) {
            float v[8];
            unpack(load_raw<bf16_t, 8>(p + c), v);
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = g * expf(v[k] - lse) - (c + k == label ? g : 0.0f);
            pack(v, r);
        }
        *reinterpret_cast<u32x4*>(o + c) = r;
    }
}

// ---------------------------------------------------------------------------------------
// Embedding gradient: dweight (zeroed by the caller) [V, D], row id = sum of dout's rows whose token is id.
// One workgroup per position looks through all of them, an eighth per wave and 64 per ballot, and so knows
// every position of its token and which of them it is itself.  The workgroups of a token's n positions take
// its columns in turns, 256 at a time, so that the rows of a frequent token (padding) pass through as many
// compute units as there are columns for: one takes in about 45 bytes per ns.  Of a list of up to eight
// rows a wave adds all; of a longer one each wave adds an eighth, eight rows in flight, and the waves' sums
// are added in order (a sum's order depends on the positions alone).  Looking through the positions is rows^2
// in all and what it costs where tokens repeat little; with the zeros before it, random tokens of 32000 /
// one token throughout, against the library's gradient: 2048 rows of 512 take 22 / 33 us (136 / 208), of 4096
// 102 / 117 (254 / 295); 8192 rows of 512 94 / 102 (100 / 297), of 4096 205 / 237 (402 / 461).  Beyond 8192
// rows the library is as fast.
// ---------------------------------------------------------------------------------------
constexpr int kEmbedWaves = 8, kEmbedCols = 4 * kWave, kEmbedInFlight = 8;

__global__ __launch_bounds__(kEmbedWaves* kWave) void embedding_bwd_kernel(const long long* __restrict__ ids,
                                                                           const float* __restrict__ dout,
                                                                           float* __restrict__ dweight, int rows,
                                                                           int V, int D) {
    __shared__ uint16_t s_list[kEmbeddingMaxRows];        // wave w's hits from position w * share on
    __shared__ int s_count[kEmbedWaves], s_front[kEmbedWaves];
    __shared__ __align__(16) float s_sum[kEmbedWaves][kEmbedCols];
    const int self = (int)blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const long long id = ids[self];
    if (id < 0 || id >= V) return;     // (uniform)
    const int share = ((rows + kEmbedWaves - 1) / kEmbedWaves + kWave - 1) / kWave * kWave;
    {
        int count = 0;
        int in_front = 0;                     // of the token's positions, those in front of this workgroup's
        const int end = min((wv + 1) * share, rows);
#pragma unroll 4
        for (int j0 = wv * share; j0 < end; j0 += kWave) {
            const int j = j0 + lane;
            const unsigned long long hits = __ballot(j < end && ids[j < end ? j : 0] == id);
            const int ahead = self - j0;
            in_front += __builtin_popcountll(ahead >= kWave ? hits : ahead <= 0 ? 0ull : hits & ((1ull << ahead) - 1ull));
            const int before = __builtin_popcountll(hits & ((1ull << lane) - 1ull));
            if ((hits >> lane) & 1ull) s_list[wv * share + count + before] = (uint16_t)j;
            count += __builtin_popcountll(hits);
        }
        if (lane == 0) { s_count[wv] = count; s_front[wv] = in_front; }
    }
    __syncthreads();
    int total = 0, rank = 0;
#pragma unroll
    for (int k = 0; k < kEmbedWaves; ++k) { total += s_count[k]; rank += s_front[k]; }
    const int chunks = (D + kEmbedCols - 1) / kEmbedCols;
    // the sum of the list's entries [from, to) at columns c..c+3
    auto add_rows = [&](int from, int to, int c) {
        f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
        int base = 0;              // entries of the waves in front
        for (int k = 0; k < kEmbedWaves; ++k) {
            const int at = k * share - base, hi = min(to, base + s_count[k]);
            int n = max(from, base);
            for (; n + kEmbedInFlight <= hi; n += kEmbedInFlight) {
                f32x4 v[kEmbedInFlight];
#pragma unroll
                for (int q = 0; q < kEmbedInFlight; ++q)
                    v[q] = *reinterpret_cast<const f32x4*>(dout + (size_t)s_list[at + n + q] * D + c);
#pragma unroll
                for (int q = 0; q < kEmbedInFlight; ++q) sum += v[q];
            }
            for (; n < hi; ++n) sum += *reinterpret_cast<const f32x4*>(dout + (size_t)s_list[at + n] * D + c);
            base += s_count[k];
        }
        return sum;
    };
    if (total <= kEmbedWaves) {        // (uniform)
        for (long long k = wv; rank + k * total < chunks; k += kEmbedWaves) {
            const int c = (int)(rank + k * total) * kEmbedCols + 4 * lane;
            if (c >= D) continue;
            const f32x4 sum = add_rows(0, total, c);
            float* o = dweight + (size_t)id * D + c;     // (on any 4-byte boundary)
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q] = sum[q];
        }
        return;
    }
    const int from = total * wv / kEmbedWaves, to = total * (wv + 1) / kEmbedWaves;
    for (int chunk = rank; chunk < chunks; chunk += total) {
        const int c0 = chunk * kEmbedCols, c = c0 + 4 * lane;
        f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
        if (c < D) sum = add_rows(from, to, c);
        *reinterpret_cast<f32x4*>(&s_sum[wv][4 * lane]) = sum;
        __syncthreads();
        const int oc = threadIdx.x;    // a column per thread of the first four waves
        if (oc < kEmbedCols && c0 + oc < D) {
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < kEmbedWaves; ++k) v += s_sum[k][oc];
            dweight[(size_t)id * D + c0 + oc] = v;
        }
        __syncthreads();
    }
}

int launched() { return hipGetLastError() == hipSuccess ? HAWK_OK : HAWK_ERR_LAUNCH; }

// workgroups of the norm's backward: about two per compute unit, and as many rows of partial sums
int norm_bwd_blocks(int rows) {
    const int need = ceil_div(rows, kNormWaves);
    return need < 512 ? need : 512;
}

}  // namespace

int cast_arrays(const void* const* src, void* const* dst, const unsigned long long* counts, int n, bool to_bf16,
                hipStream_t st) {
    CastTask t = {};
    t.n = n;
    for (int k = 0; k < n; ++k) {
        t.src[k] = src[k];
        t.dst[k] = dst[k];
        t.first_quad[k + 1] = t.first_quad[k] + counts[k] / 4;
    }
    unsigned long long blocks = (t.first_quad[n] + kCastThreads - 1) / kCastThreads;
    if (blocks == 0) return HAWK_OK;
    if (blocks > 4096) blocks = 4096;
    if (to_bf16) hipLaunchKernelGGL((cast_kernel<true>), dim3((unsigned)blocks), dim3(kCastThreads), 0, st, t);
    else hipLaunchKernelGGL((cast_kernel<false>), dim3((unsigned)blocks), dim3(kCastThreads), 0, st, t);
    return launched();
}

bool train_norm_supported(int D) { return D >= 8 && D % 8 == 0 && D <= 4096; }

int add_norm_fwd(const float* hidden, const void* delta, const float* weight, float eps, float* sum, void* out,
                 float* rstd, int rows, int D, hipStream_t st) {
    const dim3 grid((unsigned)ceil_div(rows, kNormWaves)), block(kNormWaves * kWave);
    const bf16_t* dl = static_cast<const bf16_t*>(delta);
    bf16_t* o = static_cast<bf16_t*>(out);
#define HAWK_NORM(Q) \
    hipLaunchKernelGGL((add_norm_fwd_kernel<Q>), grid, block, 0, st, hidden, dl, weight, eps, sum, o, rstd, rows, D)
    if (D <= 512) HAWK_NORM(1);
    else if (D <= 1024) HAWK_NORM(2);
    else if (D <= 2048) HAWK_NORM(4);
    else HAWK_NORM(8);
#undef HAWK_NORM
    return launched();
}

size_t add_norm_bwd_workspace_bytes(int rows, int D) { return (size_t)norm_bwd_blocks(rows) * D * sizeof(float); }

int add_norm_bwd(const void* dout, const float* sum, const float* rstd, const float* weight, const float* d_direct,
                 float* d_sum, void* d_delta, float* dweight, int rows, int D, void* ws, hipStream_t st) {
    const int blocks = norm_bwd_blocks(rows);
    const dim3 grid((unsigned)blocks), block(kNormWaves * kWave);
    const bf16_t* dy = static_cast<const bf16_t*>(dout);
    bf16_t* dd = static_cast<bf16_t*>(d_delta);
    float* part = static_cast<float*>(ws);
    const size_t lds = (size_t)kNormWaves * D * sizeof(float);
#define HAWK_NORM(Q)                                                                                                  \
    hipLaunchKernelGGL((add_norm_bwd_kernel<Q>), grid, block, lds, st, dy, sum, rstd, weight, d_direct, d_sum, dd, part, \
                       rows, D)
    if (D <= 512) HAWK_NORM(1);
    else if (D <= 1024) HAWK_NORM(2);
    else if (D <= 2048) HAWK_NORM(4);
    else HAWK_NORM(8);
#undef HAWK_NORM
    if (int rc = launched()) return rc;
    const ColsumTask reduce{part, dweight, nullptr, nullptr, blocks, D, D};
    hipLaunchKernelGGL(norm_weight_kernel, dim3((unsigned)reduce.blocks()), dim3(kColsumThreads), 0, st, reduce);
    return launched();
}

int gelu_mul_fwd(const void* gu, void* act, long long rows, int I, hipStream_t st) {
    const size_t groups = (size_t)rows * (I / 8);
    hipLaunchKernelGGL(gelu_mul_fwd_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st,
                       static_cast<const bf16_t*>(gu), static_cast<bf16_t*>(act), groups, I / 8);
    return launched();
}

int gelu_mul_bwd(const void* gu, const void* dact, void* dgu, long long rows, int I, hipStream_t st) {
    const size_t groups = (size_t)rows * (I / 8);
    hipLaunchKernelGGL(gelu_mul_bwd_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st,
                       static_cast<const bf16_t*>(gu), static_cast<const bf16_t*>(dact), static_cast<bf16_t*>(dgu),
                       groups, I / 8);
    return launched();
}

int cross_entropy_fwd(const void* logits, const long long* labels, float* lse, float* loss, float* mean, int rows,
                      int T, int V, hipStream_t st) {
    hipLaunchKernelGGL(cross_entropy_fwd_kernel, dim3((unsigned)rows), dim3(kCeThreads), 0, st,
                       static_cast<const bf16_t*>(logits), labels, lse, loss, T, V);
    if (int rc = launched()) return rc;
    hipLaunchKernelGGL(cross_entropy_mean_kernel, dim3(1), dim3(1024), 0, st, loss, labels, mean, rows, T, V);
    return launched();
}

int cross_entropy_bwd(const void* logits, const long long* labels, const float* lse, const float* mean,
                      const float* dloss, void* dlogits, int rows, int T, int V, hipStream_t st) {
    hipLaunchKernelGGL(cross_entropy_bwd_kernel, dim3((unsigned)rows), dim3(kCeThreads), 0, st,
                       static_cast<const bf16_t*>(logits), labels, lse, mean, dloss, static_cast<bf16_t*>(dlogits), T, V);
    return launched();
}

int embedding_bwd(const long long* ids, const float* dout, float* dweight, int rows, int V, int D, hipStream_t st) {
    hipLaunchKernelGGL(embedding_bwd_kernel, dim3((unsigned)rows), dim3(kEmbedWaves * kWave), 0, st, ids, dout, dweight,
                       rows, V, D);
    return launched();
}

}  // namespace hawk
