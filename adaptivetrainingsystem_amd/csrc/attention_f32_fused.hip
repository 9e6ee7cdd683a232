// Float32 attention without materialised scores, forward and backward (head_dim 64 and 128, no dropout, no per-pair mask).
//
// The materialised route (attention_f32.hip between grouped products) costs 20 launches and five [heads, L, Lk] arrays a
// training step; for the sequences that a small float32 model trains on every one of them is too short to fill the chip.
// Here a workgroup owns 16 query rows (forward, dq) or 16 keys (dk, dv) of one head: 16 rows because two sequences of 256
// tokens with 4 heads are then 128 workgroups instead of 16, and the four (eight) waves of a workgroup split the other
// dimension, so that the serial chain is a quarter of the sequence.  All products are v_mfma_f32_16x16x4_f32 with float32
// accumulation.  Operands go from memory (L2: all tiles of a head read the same keys) to registers, never through LDS:
//   S^T = K.Q^T  a lane holds row l % 16 of both operands, 16-byte pieces 4 (l / 16) of every 16 columns (the order of the
//                columns inside a contraction is free, it only has to be the same for both);
//   the result of a lane is keys 4 (l / 16) + r of query l % 16, which is exactly the second operand of
//   O^T += V^T.P^T  when step r contracts over the keys 4 (l / 16) + r; the first operand is a 16-byte piece of those rows
//                of V, whose columns 64 jj + 4 (l % 16) + i belong to the output tile (jj, i).
// The waves' partial results meet in LDS in wave order: nothing depends on timing.
// Values are those of the materialised route: scale, causal fill with -1e4 (Src/Main_Scripts/core/model.py:813-817), the
// additive mask of the keys (819-824), softmax.  The fill is a score like any other: a row whose visible scores all lie near
// or below it gives weight to its future keys, and so does a row before a key whose mask lifts the fill (it is added behind
// it).  The workgroup then walks all keys; it skips future keys only where the largest of their scores, fill plus mask, is so far
// below the row's maximum that its exponential is zero in float32.  (Infinities and NaN in the values of skipped keys, as in the
// bfloat16 kernels, do not reach the row; the materialised product multiplied them by zero, to NaN.)
// Bounds: launches and the serial chain of a tile (32 MFMAs of 32 cycles per product) at short sequences, L1 traffic at long
// ones (every tile is read in both layouts).  Materialised route -> this, microseconds, forward | backward:
//   2 x 54, 4 heads of 128    88 ->    7 |   158 ->   19        1 x 1024, 32 heads of 128   287 ->  127 |   639 ->  458
//   2 x 256, 4 heads of 128   57 ->   12 |   133 ->   39        1 x 2048, 16 heads of  64   480 ->  123 |  1177 ->  435
//   4 x 512, 4 heads of 128   77 ->   32 |   135 ->   92        1 x 4096, 32 heads of 128  6571 -> 1460 | 16260 -> 6104
//   4 x 512, 32 heads of 128 284 ->  153 |   650 ->  562
// Errors against float64 (output, dq, dk, dv), 8 heads x 32: 1.1e-7, 1.9e-7, 2.1e-7, 1.5e-7 -> 1.2e-7, 1.8e-7, 1.8e-7,
// 1.3e-7; 16 heads x 512: 3.4e-7, 4.2e-7, 6.1e-7, 5.9e-7 -> 1.7e-7, 2.2e-7, 2.9e-7, 2.7e-7.
#include <math.h>

#include "ats_common.hpp"
#include "tile_schedule.hpp"

namespace ats {

typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr float kFill = -1e4f;
// Whether a row of this maximum gives weight to keys whose largest score is `fill` (exp(-104) is zero in float32; not a number: yes).
__device__ __forceinline__ bool gives_weight(float fill, float top) { return !(fill - top <= -200.f); }

struct AttnF32Args {
    const float *q, *k, *v, *out, *dout;     // q [B,Hq,L,D], k, v [B,Hkv,Lk,D], out, dout [B,L,Hq*D]
    const float* key_bias;                   // [B,Lk] or null
    float *o, *stats, *delta, *dq, *dk, *dv; // stats [B*Hq,L][2]: row maximum, 1 / sum; delta [B*Hq,L]
    int Hq, Hkv, L, Lk;
    float scale;
};

__device__ __forceinline__ f32x4v mfma_f32(float a, float b, f32x4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4v ldv(const float* p) { return *reinterpret_cast<const f32x4v*>(p); }

// row l % 16 of a 16-row tile, pieces of the lane: columns 16 t + 4 (l / 16) ..
template <int D>
__device__ __forceinline__ void load_rows(f32x4v (&f)[D / 16], const float* row, int g) {
#pragma unroll
    for (int t = 0; t < D / 16; ++t) f[t] = ldv(row + 16 * t + 4 * g);
}
// product of two such tiles over D columns, in four chains: no MFMA waits for the one before it, and the sums are as short
// as those of the materialised route, which cut the columns over four waves
template <int D>
__device__ __forceinline__ f32x4v dot_tiles(const f32x4v (&a)[D / 16], const f32x4v (&b)[D / 16]) {
    f32x4v s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < D / 16; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = mfma_f32(a[t][i], b[t][i], s[i]);
    return (s[0] + s[1]) + (s[2] + s[3]);
}
// acc[jj][i] += rows[4 (l / 16) + r][64 jj + 4 (l % 16) + i] * p[r]
template <int D>
__device__ __forceinline__ void add_outer(f32x4v (&acc)[D / 64][4], const f32x4v (&rows)[4][D / 64], f32x4v p) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[jj][i] = mfma_f32(rows[r][jj][i], p[r], acc[jj][i]);
}
// rows base + min(first + 4 g + r, last), pieces of the lane
template <int D>
__device__ __forceinline__ void load_outer(f32x4v (&f)[4][D / 64], const float* base, int64_t pitch, int first, int last, int g, int c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = first + 4 * g + r;
#pragma unroll
        for (int jj = 0; jj < D / 64; ++jj) f[r][jj] = ldv(base + (int64_t)(row < last ? row : last) * pitch + 64 * jj + 4 * c);
    }
}
// accumulator -> LDS [16][D + 4]; element (jj, i) register r is column 64 jj + 16 g + 4 r + i of row c
template <int D>
__device__ __forceinline__ void put_tile(float* s, const f32x4v (&acc)[D / 64][4], int g, int c, float f) {
#pragma unroll
    for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4v*>(s + c * (D + 4) + 64 * jj + 16 * g + 4 * r) =
                f32x4v{acc[jj][0][r] * f, acc[jj][1][r] * f, acc[jj][2][r] * f, acc[jj][3][r] * f};
}

__device__ __forceinline__ float score(float s, float scale, int key, int last_key, const float* kb, int Lk) {
    float t = key > last_key ? kFill : s * scale;
    if (kb) t += kb[key < Lk ? key : Lk - 1];
    return key < Lk ? t : -INFINITY;
}

// largest of kb[from .. Lk), in every thread of the wave whose workgroup shares the keys out (NaN as infinity)
__device__ __forceinline__ float largest_bias(const float* kb, int from, int Lk) {
    float m = -INFINITY;
    for (int j = from + threadIdx.x; j < Lk; j += blockDim.x) {
        const float b = kb[j];
        m = b <= m ? m : b == b ? b : INFINITY;
    }
#pragma unroll
    for (int s = 1; s < 64; s *= 2) m = fmaxf(m, __shfl_xor(m, s, 64));
    return m;
}

// The tiles of a head on one XCD (consecutive workgroups go to different ones), whose L2 then holds the keys and values of the two or
// three heads that it works on instead of all that run, where the heads divide by the XCDs; same bits.  4 x 512, 32 heads of 128:
// 213 -> 153 us forward, 855 -> 562 backward.
__device__ __forceinline__ void tile_and_head(int& tile, int& head) {
    tile = blockIdx.x;
    head = blockIdx.y;
    if (gridDim.y % kNumXcd == 0) {
        const unsigned id = blockIdx.y * gridDim.x + blockIdx.x, within = id / kNumXcd;
        tile = (int)(within % gridDim.x);
        head = (int)(within / gridDim.x * kNumXcd + id % kNumXcd);
    }
}

template <int D>
__global__ __launch_bounds__(256) void attention_f32_fwd_kernel(AttnF32Args p) {
    constexpr int W = 4;
    __shared__ float s_m[W][16], s_l[W][16], s_b[W];
    __shared__ __align__(16) float s_o[W][16 * (D + 4)];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    int tile, e;
    tile_and_head(tile, e);
    const int b = e / p.Hq, h = e - b * p.Hq;
    const int q0 = ((int)gridDim.x - 1 - tile) * 16;      // the longest rows first
    const int q = q0 + c < p.L ? q0 + c : p.L - 1;
    const int last_key = q + p.Lk - p.L;
    const int64_t kvh = (int64_t)b * p.Hkv + h / (p.Hq / p.Hkv);
    const float* K = p.k + kvh * p.Lk * D;
    const float* V = p.v + kvh * p.Lk * D;
    const float* kb = p.key_bias ? p.key_bias + (int64_t)b * p.Lk : nullptr;
    f32x4v qf[D / 16];
    load_rows<D>(qf, p.q + ((int64_t)e * p.L + q) * D, g);
    f32x4v acc[D / 64][4];
#pragma unroll
    for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[jj][i] = f32x4v{0.f, 0.f, 0.f, 0.f};
    float m = -3.4028235e38f, l = 0.f;
    const int all = (p.Lk + 15) / 16;
    const int past_last = q0 + 16 + p.Lk - p.L;      // keys below it are visible to some row
    const int visible = past_last < p.Lk ? (past_last + 15) / 16 : all;
    auto row_of = [&](int kt) { const int j = 16 * kt + c; return K + (int64_t)(j < p.Lk ? j : p.Lk - 1) * D; };
    auto walk = [&](int from, int to) {
        f32x4v kf[D / 16];
        if (from + wave < to) load_rows<D>(kf, row_of(from + wave), g);
        for (int kt = from + wave; kt < to; kt += W) {
            f32x4v vf[4][D / 64];
            load_outer<D>(vf, V, D, 16 * kt, p.Lk - 1, g, c);
            const f32x4v s = dot_tiles<D>(kf, qf);
            if (kt + W < to) load_rows<D>(kf, row_of(kt + W), g);
            f32x4v t;
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = score(s[r], p.scale, 16 * kt + 4 * g + r, last_key, kb, p.Lk);
            float mx = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            mx = fmaxf(mx, m);
            const float f = expf(m - mx);
            m = mx;
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = expf(t[r] - mx);
            l = l * f + ((t[0] + t[1]) + (t[2] + t[3]));
#pragma unroll
            for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[jj][i] *= f;
            add_outer<D>(acc, vf, t);
        }
    };
    auto exchange = [&]() {
        if (g == 0) s_m[wave][c] = m;
        __syncthreads();
        float mx = s_m[0][c];
#pragma unroll
        for (int w = 1; w < W; ++w) mx = fmaxf(mx, s_m[w][c]);
        return mx;
    };
    if (kb && visible < all) {
        const float b = largest_bias(kb, 16 * visible, p.Lk);
        if (lane == 0) s_b[wave] = b;
    }
    walk(0, visible);
    float top = exchange();
    const float fill = kb && visible < all ? kFill + fmaxf(fmaxf(s_b[0], s_b[1]), fmaxf(s_b[2], s_b[3])) : kFill;
    if (visible < all && __any(gives_weight(fill, top))) {      // the same rows in every wave, hence the same answer
        __syncthreads();
        walk(visible, all);
        top = exchange();
    }
    const float f = expf(m - top);
    l *= f;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) s_l[wave][c] = l;
    put_tile<D>(s_o[wave], acc, g, c, f);
    __syncthreads();
    const int r = threadIdx.x >> 4, part = threadIdx.x & 15;
    if (q0 + r < p.L) {
        const float sum = (s_l[0][r] + s_l[1][r]) + (s_l[2][r] + s_l[3][r]);
        const float inv = 1.0f / sum;
#pragma unroll
        for (int jj = 0; jj < D / 64; ++jj) {
            const int at = r * (D + 4) + 64 * jj + 4 * part;
            const f32x4v o = ((ldv(s_o[0] + at) + ldv(s_o[1] + at)) + (ldv(s_o[2] + at) + ldv(s_o[3] + at))) * inv;
            *reinterpret_cast<f32x4v*>(p.o + (((int64_t)b * p.L + q0 + r) * p.Hq + h) * D + 64 * jj + 4 * part) = o;
        }
    }
    if (p.stats && wave == 0 && g == 0 && q0 + c < p.L) {
        float* st = p.stats + ((int64_t)e * p.L + q0 + c) * 2;
        st[0] = top;
        st[1] = 1.0f / ((s_l[0][c] + s_l[1][c]) + (s_l[2][c] + s_l[3][c]));
    }
}

// dq and delta.  dS = P (dP - delta) scale, dP = dout.V^T; dq = dS.K.  delta = sum_d dout * out, except for rows of few keys,
// where it is taken as sum_j P dP from the dP that it is subtracted from: with one key the difference is then zero and not
// the rounding of two sums, with two keys half of it cancels, .. (8 heads x 32 rows: error of dq 2.4e-7 -> 1.9e-7).
template <int D>
__global__ __launch_bounds__(256) void attention_f32_dq_kernel(AttnF32Args p) {
    constexpr int W = 4;
    __shared__ float s_d[W][16], s_b[W];
    __shared__ __align__(16) float s_o[W][16 * (D + 4)];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    int tile, e;
    tile_and_head(tile, e);
    const int b = e / p.Hq, h = e - b * p.Hq;
    const int q0 = ((int)gridDim.x - 1 - tile) * 16;
    const int q = q0 + c < p.L ? q0 + c : p.L - 1;
    const int last_key = q + p.Lk - p.L;
    const int64_t kvh = (int64_t)b * p.Hkv + h / (p.Hq / p.Hkv);
    const float* K = p.k + kvh * p.Lk * D;
    const float* V = p.v + kvh * p.Lk * D;
    const float* kb = p.key_bias ? p.key_bias + (int64_t)b * p.Lk : nullptr;
    const int64_t orow = (((int64_t)b * p.L + q) * p.Hq + h) * D;
    f32x4v qf[D / 16], df[D / 16];
    load_rows<D>(qf, p.q + ((int64_t)e * p.L + q) * D, g);
    load_rows<D>(df, p.dout + orow, g);
    const float* st = p.stats + ((int64_t)e * p.L + q) * 2;
    const float top = st[0], inv = st[1];
    f32x4v acc[D / 64][4];
#pragma unroll
    for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[jj][i] = f32x4v{0.f, 0.f, 0.f, 0.f};
    const int all = (p.Lk + 15) / 16;
    const int past_last = q0 + 16 + p.Lk - p.L;
    int end = past_last < p.Lk ? (past_last + 15) / 16 : all;
    float fill = kFill;
    if (kb && end < all) {
        const float bias = largest_bias(kb, 16 * end, p.Lk);
        if (lane == 0) s_b[wave] = bias;
        __syncthreads();
        fill += fmaxf(fmaxf(s_b[0], s_b[1]), fmaxf(s_b[2], s_b[3]));
    }
    if (__any(gives_weight(fill, top))) end = all;
    auto weights = [&](int kt, f32x4v& w, f32x4v& dp) {
        const int j = 16 * kt + c < p.Lk ? 16 * kt + c : p.Lk - 1;
        f32x4v kf[D / 16], vf[D / 16];
        load_rows<D>(kf, K + (int64_t)j * D, g);
        load_rows<D>(vf, V + (int64_t)j * D, g);
        const f32x4v s = dot_tiles<D>(kf, qf);
        dp = dot_tiles<D>(vf, df);
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = expf(score(s[r], p.scale, 16 * kt + 4 * g + r, last_key, kb, p.Lk) - top) * inv;
    };
    float delta = 0.f;
    constexpr int KEEP = 2;      // tiles per wave whose weights stay in registers until delta is known
    if (end <= W * KEEP) {       // the same in every wave
        f32x4v w[KEEP], dp[KEEP];
#pragma unroll
        for (int u = 0; u < KEEP; ++u)
            if (wave + u * W < end) {
                weights(wave + u * W, w[u], dp[u]);
                delta += (w[u][0] * dp[u][0] + w[u][1] * dp[u][1]) + (w[u][2] * dp[u][2] + w[u][3] * dp[u][3]);
            }
        delta += __shfl_xor(delta, 16, 64);
        delta += __shfl_xor(delta, 32, 64);
        if (g == 0) s_d[wave][c] = delta;
        __syncthreads();
        delta = (s_d[0][c] + s_d[1][c]) + (s_d[2][c] + s_d[3][c]);
#pragma unroll
        for (int u = 0; u < KEEP; ++u)
            if (wave + u * W < end) {
                f32x4v ko[4][D / 64];
                load_outer<D>(ko, K, D, 16 * (wave + u * W), p.Lk - 1, g, c);
                add_outer<D>(acc, ko, w[u] * (dp[u] - delta) * p.scale);
            }
    } else {
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            const f32x4v x = df[t] * ldv(p.out + orow + 16 * t + 4 * g);
            delta += (x[0] + x[1]) + (x[2] + x[3]);
        }
        delta += __shfl_xor(delta, 16, 64);
        delta += __shfl_xor(delta, 32, 64);
        for (int kt = wave; kt < end; kt += W) {
            f32x4v w, dp, ko[4][D / 64];
            load_outer<D>(ko, K, D, 16 * kt, p.Lk - 1, g, c);
            weights(kt, w, dp);
            add_outer<D>(acc, ko, w * (dp - delta) * p.scale);
        }
    }
    if (wave == 0 && g == 0 && q0 + c < p.L) p.delta[(int64_t)e * p.L + q0 + c] = delta;
    put_tile<D>(s_o[wave], acc, g, c, 1.f);
    __syncthreads();
    const int r = threadIdx.x >> 4, part = threadIdx.x & 15;
    if (q0 + r >= p.L) return;
#pragma unroll
    for (int jj = 0; jj < D / 64; ++jj) {
        const int at = r * (D + 4) + 64 * jj + 4 * part;
        *reinterpret_cast<f32x4v*>(p.dq + ((int64_t)e * p.L + q0 + r) * D + 64 * jj + 4 * part) =
            (ldv(s_o[0] + at) + ldv(s_o[1] + at)) + (ldv(s_o[2] + at) + ldv(s_o[3] + at));
    }
}

// dk = dS^T.Q and dv = P^T.dout of 16 keys, summed over the query heads of their kv head: the waves take (head, query
// tile) pairs in turn.
template <int D>
__global__ __launch_bounds__(512) void attention_f32_dkv_kernel(AttnF32Args p) {
    constexpr int W = 8;
    __shared__ __align__(16) float s_o[W / 2][16 * (D + 4)];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    int tile, kvh;
    tile_and_head(tile, kvh);
    const int b = kvh / p.Hkv, hk = kvh - b * p.Hkv;
    const int k0 = tile * 16;                                    // the first keys have the most rows
    const int key = k0 + c < p.Lk ? k0 + c : p.Lk - 1;
    const int rep = p.Hq / p.Hkv, off = p.Lk - p.L;
    const float* kb = p.key_bias ? p.key_bias + (int64_t)b * p.Lk : nullptr;
    const int64_t e0 = (int64_t)b * p.Hq + hk * rep;             // first query head
    f32x4v kf[D / 16], vf[D / 16];
    load_rows<D>(kf, p.k + ((int64_t)kvh * p.Lk + key) * D, g);
    load_rows<D>(vf, p.v + ((int64_t)kvh * p.Lk + key) * D, g);
    float fill = kFill;                                          // largest score of these keys in the rows before them
    if (kb) {
        const float own = kb[key];
        float bias = own == own ? own : INFINITY;
#pragma unroll
        for (int x = 1; x < 16; x *= 2) bias = fmaxf(bias, __shfl_xor(bias, x, 64));
        fill += bias;
    }
    // query tiles before `first` see none of these keys, unless a row gives weight to its future
    int first = k0 - off > 0 ? (k0 - off) / 16 : 0;
    const int tiles = (p.L + 15) / 16;
    first = first < tiles ? first : tiles;
    bool early = false;
    for (int h = 0; h < rep; ++h)
        for (int i = threadIdx.x; i < first * 16; i += W * 64) early |= gives_weight(fill, p.stats[((e0 + h) * p.L + i) * 2]);
    if (__syncthreads_or(early)) first = 0;
    f32x4v dk[D / 64][4], dv[D / 64][4];
#pragma unroll
    for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
        for (int i = 0; i < 4; ++i) dk[jj][i] = dv[jj][i] = f32x4v{0.f, 0.f, 0.f, 0.f};
    const int per_head = tiles - first;
    for (int it = wave; it < rep * per_head; it += W) {
        const int h = it / per_head, q0 = (first + it - h * per_head) * 16;
        const int64_t e = e0 + h;
        const int q = q0 + c < p.L ? q0 + c : p.L - 1;
        const float* Q = p.q + e * p.L * D;
        const float* dO = p.dout + ((int64_t)b * p.L * p.Hq + hk * rep + h) * D;
        const int64_t pitch = (int64_t)p.Hq * D;
        f32x4v qf[D / 16], df[D / 16], qo[4][D / 64], go[4][D / 64];
        load_rows<D>(qf, Q + (int64_t)q * D, g);
        load_rows<D>(df, dO + q * pitch, g);
        load_outer<D>(go, dO, pitch, q0, p.L - 1, g, c);
        float top[4], inv[4], delta[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = q0 + 4 * g + r < p.L ? q0 + 4 * g + r : p.L - 1;
            top[r] = p.stats[(e * p.L + i) * 2];
            inv[r] = p.stats[(e * p.L + i) * 2 + 1];
            delta[r] = p.delta[e * p.L + i];
        }
        const f32x4v s = dot_tiles<D>(qf, kf), dp = dot_tiles<D>(df, vf);
        load_outer<D>(qo, Q, D, q0, p.L - 1, g, c);
        f32x4v w, ds;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = q0 + 4 * g + r;
            w[r] = i < p.L ? expf(score(s[r], p.scale, key, i + off, kb, p.Lk) - top[r]) * inv[r] : 0.f;
            ds[r] = i < p.L ? w[r] * (dp[r] - delta[r]) * p.scale : 0.f;
        }
        add_outer<D>(dv, go, w);
        add_outer<D>(dk, qo, ds);
    }
    const int r = threadIdx.x >> 4, part = threadIdx.x & 15;     // of the first 256 threads
    auto finish = [&](f32x4v(&acc)[D / 64][4], float* out) {
        if (wave >= W / 2) put_tile<D>(s_o[wave - W / 2], acc, g, c, 1.f);
        __syncthreads();
        if (wave < W / 2) {      // each adds the tile of the wave W / 2 above it
            float* s = s_o[wave];
#pragma unroll
            for (int jj = 0; jj < D / 64; ++jj)
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) {
                    const f32x4v x = ldv(s + c * (D + 4) + 64 * jj + 16 * g + 4 * rr);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[jj][i][rr] += x[i];
                }
            put_tile<D>(s, acc, g, c, 1.f);
        }
        __syncthreads();
        if (threadIdx.x < 256 && k0 + r < p.Lk) {
#pragma unroll
            for (int jj = 0; jj < D / 64; ++jj) {
                const int at = r * (D + 4) + 64 * jj + 4 * part;
                *reinterpret_cast<f32x4v*>(out + ((int64_t)kvh * p.Lk + k0 + r) * D + 64 * jj + 4 * part) =
                    (ldv(s_o[0] + at) + ldv(s_o[1] + at)) + (ldv(s_o[2] + at) + ldv(s_o[3] + at));
            }
        }
        __syncthreads();
    };
    finish(dv, p.dv);
    finish(dk, p.dk);
}

static int check_attn_f32(const char* name, int B, int Hq, int Hkv, int L, int Lk, int D, float scale) {
    ATS_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && L >= 0 && Lk >= L && (D == 64 || D == 128) && scale > 0.f,
                ATS_ERR_INVALID_ARG, "%s: B=%d Hq=%d Hkv=%d L=%d Lk=%d D=%d scale=%g", name, B, Hq, Hkv, L, Lk, D, scale);
    ATS_REQUIRE((int64_t)B * Hq <= 65535, ATS_ERR_UNSUPPORTED, "%s: %lld (batch, head) pairs", name, (long long)B * Hq);
    return ATS_OK;
}

}  // namespace ats

extern "C" int ats_attention_f32_fwd(const float* q, const float* k, const float* v, float* out, float* stats, int B, int Hq,
                                     int Hkv, int L, int Lk, int D, float scale, const float* key_bias, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_attention_f32_fwd";
    const int rc = check_attn_f32(name, B, Hq, Hkv, L, Lk, D, scale);
    if (rc != ATS_OK) return rc;
    if (B == 0 || L == 0) return ATS_OK;
    ATS_REQUIRE(q && k && v && out && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), ATS_ERR_INVALID_ARG,
                "%s: null or misaligned pointer", name);
    AttnF32Args a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.o = out;
    a.stats = stats;
    a.key_bias = key_bias;
    a.Hq = Hq;
    a.Hkv = Hkv;
    a.L = L;
    a.Lk = Lk;
    a.scale = scale;
    const dim3 grid((L + 15) / 16, B * Hq);
    if (D == 64) hipLaunchKernelGGL(attention_f32_fwd_kernel<64>, grid, dim3(256), 0, as_stream(stream), a);
    else hipLaunchKernelGGL(attention_f32_fwd_kernel<128>, grid, dim3(256), 0, as_stream(stream), a);
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_attention_f32_bwd(const float* q, const float* k, const float* v, const float* out, const float* stats,
                                     const float* dout, float* delta, float* dq, float* dk, float* dv, int B, int Hq, int Hkv,
                                     int L, int Lk, int D, float scale, const float* key_bias, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_attention_f32_bwd";
    const int rc = check_attn_f32(name, B, Hq, Hkv, L, Lk, D, scale);
    if (rc != ATS_OK) return rc;
    if (B == 0 || L == 0) return ATS_OK;
    for (const void* x : {(const void*)q, (const void*)k, (const void*)v, (const void*)out, (const void*)dout, (const void*)dq,
                          (const void*)dk, (const void*)dv})
        ATS_REQUIRE(x && aligned16(x), ATS_ERR_INVALID_ARG, "%s: null or misaligned pointer", name);
    ATS_REQUIRE(stats && delta, ATS_ERR_INVALID_ARG, "%s: null pointer", name);
    AttnF32Args a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.dout = dout;
    a.stats = const_cast<float*>(stats);
    a.delta = delta;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.key_bias = key_bias;
    a.Hq = Hq;
    a.Hkv = Hkv;
    a.L = L;
    a.Lk = Lk;
    a.scale = scale;
    const dim3 grid_q((L + 15) / 16, B * Hq), grid_k((Lk + 15) / 16, B * Hkv);
    hipStream_t s = as_stream(stream);
    if (D == 64) {
        hipLaunchKernelGGL(attention_f32_dq_kernel<64>, grid_q, dim3(256), 0, s, a);
        hipLaunchKernelGGL(attention_f32_dkv_kernel<64>, grid_k, dim3(512), 0, s, a);
    } else {
        hipLaunchKernelGGL(attention_f32_dq_kernel<128>, grid_q, dim3(256), 0, s, a);
        hipLaunchKernelGGL(attention_f32_dkv_kernel<128>, grid_k, dim3(512), 0, s, a);
    }
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}
