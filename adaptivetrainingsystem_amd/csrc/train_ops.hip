// Training-step ops next to the sparse layer (gfx950, HBM-bound):
//   fused cross-entropy + accuracy (forward and the gradient w.r.t. the logits),
//   multi-tensor gradient norm + clipping.
// They replace fused_cross_entropy_accuracy_launcher (Src/Main_Scripts/training/fused_loss.cu:179-214)
// and fused_grad_clip_launcher (Src/Main_Scripts/training/fused_grad_clip.cu:117-175).  Differences by
// design: every sum runs in a fixed order (per-token / per-chunk partials and an ordered second pass
// instead of float atomics), nothing synchronises, bf16 logits and gradients are accepted, and the
// logits gradient exists (the reference's fused loss returns a value without a graph).
#include <math.h>

#include "ats_common.hpp"

namespace ats {

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// exp(x) for x <= 0 or NaN (differences to a maximum) through the hardware exp2 (about 1 ulp): x log2(e) in two parts, so
// that the rounding of the product, |x| 2^-24 of the result, is put back.  Below -104 the float32 result is zero; the
// bound also keeps -inf out of the second part.
__device__ __forceinline__ float exp_split(float x) {
    x = x < -104.f ? -104.f : x;
    const float h = x * 1.44269502162933349609375f;
    float e = fmaf(x, 1.44269502162933349609375f, -h);
    e = fmaf(x, 1.92596299112661746887e-8f, e);
    const float p = __builtin_amdgcn_exp2f(h);
    return fmaf(p * e, 0.693147182464599609375f, p);
}

// exp(x - ref), x and ref of one row, x <= ref.  Float32 rows through exp_split.  bfloat16 rows have twice the elements per
// byte, and with eight operations each the forward pass was bound by them (16376 x 32000: 262 us, 185 with these two): one
// rounding of (x - ref) log2(e), and the product with a ref common to the whole row.  Near the end of the type's range (a
// mask of the lowest value) that product overflows; there x - ref is 0 or so far below it that exp2 without the factor gives
// the same 1 or 0.
template <typename T>
struct RowExp {
    float scale, ref;
    __device__ __forceinline__ explicit RowExp(float r)
        : scale(fabsf(r) > 1e38f ? 1.f : 1.4426950408889634f), ref(sizeof(T) == 2 ? r * scale : r) {}
    __device__ __forceinline__ float operator()(float x) const {
        if (sizeof(T) == 2) return __builtin_amdgcn_exp2f(fmaf(x, scale, -ref));
        return exp_split(x - ref);
    }
};

// A row of V elements as a head up to the next 16-byte boundary, whole vectors, and a tail.  Rows of a vocabulary that
// is no multiple of 8 start at every alignment (50257 columns took an element-wise route: loss and gradient of 16376
// bfloat16 rows 3593 us, now 969; 4095 float32 rows 990, now 501).
struct RowSplit {
    int head, nv, tail0;
};
template <typename T>
__device__ __forceinline__ RowSplit split_row(const T* row, int V) {
    constexpr int VW = Elem<T>::kVec;
    RowSplit r;
    r.head = (int)((16 - (reinterpret_cast<uintptr_t>(row) & 15u)) & 15u) / (int)sizeof(T);
    r.head = r.head < V ? r.head : V;
    r.nv = (V - r.head) / VW;
    r.tail0 = r.head + r.nv * VW;
    return r;
}

// ---------------------------------------------------------------- cross entropy
struct MaxSum {
    float m, s;   // running maximum and sum of exp(x - m)
};
__device__ __forceinline__ MaxSum ms_merge(MaxSum a, MaxSum b) {
    if (b.m > a.m) {
        MaxSum t = a;
        a = b;
        b = t;
    }
    if (b.m == -INFINITY) return a;
    a.s += b.s * expf(b.m - a.m);
    return a;
}
// One block (256 threads) per token: one pass over the row in tiles of 16 vectors per thread, whose loads are all in
// flight together (64 KiB a block); per tile the maximum, then one exp per element against the maximum so far; then a
// block reduction.  HBM-bound: 16376 x 32000 bfloat16 185 us (5.7 TB/s); float32 rows of that length, which took one
// exponential and one branch per element one load at a time, 1452 -> 1152 us with the backward.  Marking these loads as not
// to be kept gains 10 us here and costs the backward 25.
// Outputs per token: loss (0 for ignored tokens), lse = max + log(sum exp), correct (1.0 when the arg-max equals the
// label), valid (1.0 / 0.0).  A token is ignored when its label equals pad_id or lies outside [0, V)
// (fused_loss.cu:83-84).
template <typename T>
__global__ __launch_bounds__(256) void cross_entropy_fwd_kernel(const T* __restrict__ logits,
                                                                const int64_t* __restrict__ labels, int64_t pad_id,
                                                                float* __restrict__ loss, float* __restrict__ lse,
                                                                float* __restrict__ correct, float* __restrict__ valid,
                                                                int V) {
    constexpr int VW = Elem<T>::kVec;
    __shared__ MaxSum s_ms[4];
    __shared__ int s_lower;
    const int64_t t = blockIdx.x;
    const int64_t label = labels[t];
    if (label == pad_id || label < 0 || label >= V) {
        if (threadIdx.x == 0) {
            loss[t] = 0.f;
            lse[t] = 0.f;
            correct[t] = 0.f;
            valid[t] = 0.f;
        }
        return;
    }
    const T* row = logits + t * V;
    MaxSum ms{-INFINITY, 0.f};
    const float x_label = Elem<T>::load(row + label);
    const RowSplit rs = split_row(row, V);
    bool nan = false;        // a NaN among elements that are all -inf otherwise (else the sum has it)
    // element e of the head and the tail (fewer than 2 * VW): thread e's
    auto edge = [&](int i) {
        const float x = Elem<T>::load(row + i);
        if (x > ms.m) ms = MaxSum{x, ms.s * exp_split(ms.m - x) + 1.f};
        else if (ms.m != -INFINITY) ms.s += exp_split(x - ms.m);
        else nan = nan || x != x;
    };
    if ((int)threadIdx.x < rs.head) edge(threadIdx.x);
    constexpr int kTileVecs = 16;
    const u32x4_t* body = reinterpret_cast<const u32x4_t*>(row + rs.head);
    for (int v0 = 0; v0 < rs.nv; v0 += 256 * kTileVecs) {
        u32x4_t raw[kTileVecs];
#pragma unroll
        for (int q = 0; q < kTileVecs; ++q) {
            const int v = v0 + threadIdx.x + q * 256;
            if (v < rs.nv) raw[q] = body[v];
        }
        float mx = -INFINITY;
#pragma unroll
        for (int q = 0; q < kTileVecs; ++q) {
            const int v = v0 + threadIdx.x + q * 256;
            if (v < rs.nv) {
                float f[VW];
                Elem<T>::unpack(make_uint4(raw[q][0], raw[q][1], raw[q][2], raw[q][3]), f);
#pragma unroll
                for (int j = 0; j < VW; ++j) mx = fmaxf(mx, f[j]);
            }
        }
        const float m = mx > ms.m ? mx : ms.m;
        if (m == -INFINITY) {                // nothing but masked elements so far
#pragma unroll
            for (int q = 0; q < kTileVecs; ++q) {
                float f[VW];
                Elem<T>::unpack(make_uint4(raw[q][0], raw[q][1], raw[q][2], raw[q][3]), f);
#pragma unroll
                for (int j = 0; j < VW; ++j) nan = nan || (v0 + (int)threadIdx.x + q * 256 < rs.nv && f[j] != f[j]);
            }
            continue;
        }
        const RowExp<T> ex(m);
        float sum = ms.m == -INFINITY ? 0.f : ms.s * exp_split(ms.m - m);
#pragma unroll
        for (int q = 0; q < kTileVecs; ++q) {
            const int v = v0 + threadIdx.x + q * 256;
            if (v < rs.nv) {
                float f[VW];
                Elem<T>::unpack(make_uint4(raw[q][0], raw[q][1], raw[q][2], raw[q][3]), f);
#pragma unroll
                for (int j = 0; j < VW; ++j) sum += ex(f[j]);
            }
        }
        ms = MaxSum{m, sum};
    }
    if (rs.tail0 + (int)threadIdx.x < V) edge(rs.tail0 + threadIdx.x);
    if (nan) ms = MaxSum{ms.m == -INFINITY ? -3.402823466e38f : ms.m, NAN};
    // wave reduction (fixed butterfly order), then the 4 waves in order
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        MaxSum o{__shfl_xor(ms.m, off, 64), __shfl_xor(ms.s, off, 64)};
        ms = ms_merge(ms, o);
    }
    const int wave = threadIdx.x >> 6;
    if (lane_id() == 0) s_ms[wave] = ms;
    if (threadIdx.x == 0) s_lower = 0;
    __syncthreads();
    MaxSum a = s_ms[0];
    for (int w = 1; w < 4; ++w) a = ms_merge(a, s_ms[w]);
    // The label is the arg-max when it has the maximum and no lower index has it too.  Only rows whose label has the
    // maximum look for one (in the caches), instead of every element carrying its index through the pass above.
    bool hit = a.m > -INFINITY && x_label == a.m;
    if (hit) {
        bool lower = false;
        for (int i = threadIdx.x; i < (int)label; i += 256) lower = lower || Elem<T>::load(row + i) == a.m;
        if (lower) s_lower = 1;
        __syncthreads();
        hit = s_lower == 0;
    }
    if (threadIdx.x == 0) {
        const float l = a.m + logf(a.s);
        float tok = l - x_label;
        if (isnan(tok) || isinf(tok)) tok = 10.0f;   // fused_loss.cu:121-124
        loss[t] = tok;
        lse[t] = l;
        correct[t] = hit ? 1.f : 0.f;
        valid[t] = 1.f;
    }
}

// sums[0] = sum w*loss, sums[1] = sum w (valid tokens), sums[2] = sum loss, sums[3] = sum correct,
// sums[4] = number of valid tokens; w = weights[t] (1 when weights == NULL).  Single block, fixed order; four tokens of
// a thread are loaded together (16376 tokens: 14.2 -> 7.5 us).  With loss / stats given it also forms what the
// training loop reports: loss = sums[0] / max(sums[1], 1e-8); stats = unweighted mean loss, perplexity (of the mean
// clamped to [0, 15]; inf without valid tokens), number of valid tokens, accuracy: each was two to four launches.
__global__ __launch_bounds__(1024) void cross_entropy_sums_kernel(const float* __restrict__ loss,
                                                                 const float* __restrict__ correct,
                                                                 const float* __restrict__ valid,
                                                                 const float* __restrict__ weights, int64_t Tn,
                                                                 float* __restrict__ sums, float* __restrict__ mean,
                                                                 float* __restrict__ stats) {
    __shared__ float part[5][1024];
    float a[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;
    for (int64_t t0 = threadIdx.x; t0 < Tn; t0 += 1024 * U) {
        float v[U], w[U], l[U], c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t t = t0 + u * 1024;
            const bool in = t < Tn;
            v[u] = in ? valid[t] : 0.f;
            w[u] = in && weights ? weights[t] : 1.f;
            l[u] = in ? loss[t] : 0.f;
            c[u] = in ? correct[t] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float wv = weights ? w[u] * v[u] : v[u];
            a[0] += wv * l[u];
            a[1] += wv;
            a[2] += l[u];
            a[3] += c[u];
            a[4] += v[u];
        }
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) part[q][threadIdx.x] = a[q];
    __syncthreads();
    for (int stride = 512; stride > 0; stride >>= 1) {
        if ((int)threadIdx.x < stride) {
#pragma unroll
            for (int q = 0; q < 5; ++q) part[q][threadIdx.x] += part[q][threadIdx.x + stride];
        }
        __syncthreads();
    }
    if (threadIdx.x < 5) sums[threadIdx.x] = part[threadIdx.x][0];
    if (threadIdx.x == 0 && mean) mean[0] = part[0][0] / (part[1][0] < 1e-8f ? 1e-8f : part[1][0]);
    if (threadIdx.x == 0 && stats) {
        const float n = part[4][0], denom = n < 1.f ? 1.f : n;
        const float raw = part[2][0] / denom;
        const float cl = raw < 0.f ? 0.f : (raw > 15.f ? 15.f : raw);      // (NaN stays)
        stats[0] = raw;
        stats[1] = n > 0.f ? expf(cl) : INFINITY;
        stats[2] = n;
        stats[3] = part[3][0] / denom;
    }
}

// dlogits[t, v] = g_t * (exp(z - lse_t) - [v == label_t]),  g_t = scale[0] * w_t * valid_t / max(sums[1], 1e-8)
// (gradient of  sum_t w_t loss_t / sum_t w_t; scale[0] = upstream gradient of that mean).  HBM-bound: one read and one
// write; eight vectors of a thread are loaded together and, as nobody reads the gradient before it has left the caches,
// stored past them.  16376 x 32000 bfloat16: 384 -> 364 us (5.8 TB/s).
template <typename T>
__global__ __launch_bounds__(256) void cross_entropy_bwd_kernel(const T* __restrict__ logits,
                                                                const int64_t* __restrict__ labels,
                                                                const float* __restrict__ lse,
                                                                const float* __restrict__ valid,
                                                                const float* __restrict__ weights,
                                                                const float* __restrict__ sums,
                                                                const float* __restrict__ scale,
                                                                T* __restrict__ dlogits, int V, bool same_split) {
    constexpr int VW = Elem<T>::kVec;
    const int64_t t = blockIdx.x;
    const T* row = logits + t * V;
    T* out = dlogits + t * V;
    const float v = valid[t];
    const float g = v == 0.f ? 0.f : scale[0] * (weights ? weights[t] : 1.f) / fmaxf(sums[1], 1e-8f);
    const float l = lse[t];
    const int label = v == 0.f ? -1 : (int)labels[t];
    auto edge = [&](int i) {
        const float p = g == 0.f ? 0.f : exp_split(Elem<T>::load(row + i) - l);
        Elem<T>::store(out + i, g * (p - (i == label ? 1.f : 0.f)));
    };
    if (same_split) {
        const RowSplit rs = split_row(row, V);
        if ((int)threadIdx.x < rs.head) edge(threadIdx.x);
        const u32x4_t* src = reinterpret_cast<const u32x4_t*>(row + rs.head);
        u32x4_t* dst = reinterpret_cast<u32x4_t*>(out + rs.head);
        constexpr int kTileVecs = 8;
        const RowExp<T> ex(l);
        const int label_vec = label >= rs.head ? (label - rs.head) / VW : -1;
        for (int v0 = 0; v0 < rs.nv; v0 += 256 * kTileVecs) {
            u32x4_t raw[kTileVecs];
#pragma unroll
            for (int q = 0; q < kTileVecs; ++q) {
                const int v = v0 + threadIdx.x + q * 256;
                if (v < rs.nv) raw[q] = __builtin_nontemporal_load(src + v);
            }
#pragma unroll
            for (int q = 0; q < kTileVecs; ++q) {
                const int v = v0 + threadIdx.x + q * 256;
                if (v < rs.nv) {
                    float f[VW];
                    Elem<T>::unpack(make_uint4(raw[q][0], raw[q][1], raw[q][2], raw[q][3]), f);
#pragma unroll
                    for (int j = 0; j < VW; ++j) f[j] = g == 0.f ? 0.f : ex(f[j]);
                    if (v == label_vec) {
#pragma unroll
                        for (int j = 0; j < VW; ++j) f[j] -= rs.head + v * VW + j == label ? 1.f : 0.f;
                    }
#pragma unroll
                    for (int j = 0; j < VW; ++j) f[j] *= g;
                    const uint4 r = Elem<T>::pack(f);
                    __builtin_nontemporal_store(u32x4_t{r.x, r.y, r.z, r.w}, dst + v);
                }
            }
        }
        if (rs.tail0 + (int)threadIdx.x < V) edge(rs.tail0 + threadIdx.x);
    } else {
        for (int i = threadIdx.x; i < V; i += blockDim.x) edge(i);
    }
}

// ---------------------------------------------------------------- gradient norm and clipping
// The tensors are cut into chunks of kClipChunk elements; chunk c belongs to the tensor whose
// chunk_start[] range contains c (chunk_start has n_tensors + 1 entries, built on the host).
constexpr int kClipChunk = 262144;

__device__ __forceinline__ int find_tensor(const int32_t* __restrict__ chunk_start, int n, int c) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (chunk_start[mid] <= c) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// HBM-bound: eight vectors of a thread are loaded together and not kept in the caches.  1409318912 bfloat16
// elements: 498 -> 407 us (6.9 TB/s).
template <typename T>
__global__ __launch_bounds__(256) void grad_sumsq_kernel(const void* const* __restrict__ ptrs,
                                                         const int64_t* __restrict__ sizes,
                                                         const int32_t* __restrict__ chunk_start, int n_tensors,
                                                         float* __restrict__ partial) {
    __shared__ float s_part[4];
    const int c = blockIdx.x;
    const int ti = find_tensor(chunk_start, n_tensors, c);
    const T* g = static_cast<const T*>(ptrs[ti]);
    const int64_t begin = (int64_t)(c - chunk_start[ti]) * kClipChunk;
    const int64_t end = begin + kClipChunk < sizes[ti] ? begin + kClipChunk : sizes[ti];
    float acc = 0.f;
    constexpr int VW = Elem<T>::kVec;
    if ((reinterpret_cast<uintptr_t>(g) & 15u) == 0) {
        const int64_t nv = (end - begin) / VW;
        const u32x4_t* gv = reinterpret_cast<const u32x4_t*>(g + begin);
        constexpr int U = 8;
        for (int64_t i0 = threadIdx.x; i0 < nv; i0 += 256 * U) {
            u32x4_t raw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) raw[u] = i0 + u * 256 < nv ? __builtin_nontemporal_load(gv + i0 + u * 256) : u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float f[VW];
                Elem<T>::unpack(make_uint4(raw[u][0], raw[u][1], raw[u][2], raw[u][3]), f);
#pragma unroll
                for (int j = 0; j < VW; ++j) acc += f[j] * f[j];
            }
        }
        for (int64_t i = begin + nv * VW + threadIdx.x; i < end; i += 256) {
            const float f = Elem<T>::load(g + i);
            acc += f * f;
        }
    } else {
        for (int64_t i = begin + threadIdx.x; i < end; i += 256) {
            const float f = Elem<T>::load(g + i);
            acc += f * f;
        }
    }
    acc = wave_sum(acc);
    if (lane_id() == 0) s_part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[c] = ((s_part[0] + s_part[1]) + s_part[2]) + s_part[3];
}

// norm_out[0] = sqrt(extra_sumsq + sum of the partials, in index order); norm_out[1] = that sum of squares.
__global__ __launch_bounds__(256) void grad_norm_finish_kernel(const float* __restrict__ partial, int n,
                                                               const float* __restrict__ extra_sumsq,
                                                               float* __restrict__ norm_out) {
    __shared__ float s[256];
    float acc = 0.f;
#pragma unroll 8
    for (int i = threadIdx.x; i < n; i += 256) acc += partial[i];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int stride = 128; stride > 0; stride >>= 1) {
        if ((int)threadIdx.x < stride) s[threadIdx.x] += s[threadIdx.x + stride];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const float total = s[0] + (extra_sumsq ? extra_sumsq[0] : 0.f);
        norm_out[1] = total;
        norm_out[0] = sqrtf(total);
    }
}

// grads *= max_norm / (norm + 1e-6) when that factor is below 1 (fused_grad_clip.cu:66-91).
template <typename T>
__global__ __launch_bounds__(256) void grad_scale_kernel(void* const* __restrict__ ptrs,
                                                         const int64_t* __restrict__ sizes,
                                                         const int32_t* __restrict__ chunk_start, int n_tensors,
                                                         const float* __restrict__ norm, float max_norm) {
    const float coef = max_norm / (norm[0] + 1e-6f);
    if (!(coef < 1.0f)) return;
    const int c = blockIdx.x;
    const int ti = find_tensor(chunk_start, n_tensors, c);
    T* g = static_cast<T*>(ptrs[ti]);
    const int64_t begin = (int64_t)(c - chunk_start[ti]) * kClipChunk;
    const int64_t end = begin + kClipChunk < sizes[ti] ? begin + kClipChunk : sizes[ti];
    constexpr int VW = Elem<T>::kVec;
    if ((reinterpret_cast<uintptr_t>(g) & 15u) == 0) {
        const int64_t nv = (end - begin) / VW;
        uint4* gv = reinterpret_cast<uint4*>(g + begin);
        for (int64_t i = threadIdx.x; i < nv; i += 256) {
            float f[VW];
            Elem<T>::unpack(gv[i], f);
#pragma unroll
            for (int j = 0; j < VW; ++j) f[j] *= coef;
            gv[i] = Elem<T>::pack(f);
        }
        for (int64_t i = begin + nv * VW + threadIdx.x; i < end; i += 256) Elem<T>::store(g + i, Elem<T>::load(g + i) * coef);
    } else {
        for (int64_t i = begin + threadIdx.x; i < end; i += 256) Elem<T>::store(g + i, Elem<T>::load(g + i) * coef);
    }
}

}  // namespace ats

extern "C" int ats_cross_entropy_fwd(const void* logits, const int64_t* labels, int64_t pad_id, const float* weights,
                                     float* loss_tok, float* lse, float* correct, float* valid, float* sums, int64_t T,
                                     int V, int dtype, ats_stream_t stream) {
    return ats_cross_entropy_fwd_stats(logits, labels, pad_id, weights, loss_tok, lse, correct, valid, sums, nullptr, nullptr,
                                       T, V, dtype, stream);
}

extern "C" int ats_cross_entropy_fwd_stats(const void* logits, const int64_t* labels, int64_t pad_id, const float* weights,
                                           float* loss_tok, float* lse, float* correct, float* valid, float* sums,
                                           float* loss, float* stats, int64_t T, int V, int dtype, ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(T >= 0 && T <= 0x7fffffffLL && V > 0, ATS_ERR_INVALID_ARG, "ats_cross_entropy_fwd: T=%lld V=%d", (long long)T, V);
    ATS_REQUIRE(dtype == ATS_F32 || dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "ats_cross_entropy_fwd: dtype tag %d", dtype);
    ATS_REQUIRE(sums && (T == 0 || (logits && labels && loss_tok && lse && correct && valid)), ATS_ERR_INVALID_ARG,
                "ats_cross_entropy_fwd: null pointer");
    hipStream_t s = as_stream(stream);
    if (T > 0) {
        if (dtype == ATS_F32)
            hipLaunchKernelGGL((cross_entropy_fwd_kernel<float>), dim3((unsigned)T), dim3(256), 0, s,
                               static_cast<const float*>(logits), labels, pad_id, loss_tok, lse, correct, valid, V);
        else
            hipLaunchKernelGGL((cross_entropy_fwd_kernel<bf16_t>), dim3((unsigned)T), dim3(256), 0, s,
                               static_cast<const bf16_t*>(logits), labels, pad_id, loss_tok, lse, correct, valid, V);
    }
    hipLaunchKernelGGL(cross_entropy_sums_kernel, dim3(1), dim3(1024), 0, s, loss_tok, correct, valid, weights, T, sums, loss, stats);
    ATS_CHECK_LAUNCH("ats_cross_entropy_fwd");
    return ATS_OK;
}

extern "C" int ats_cross_entropy_bwd(const void* logits, const int64_t* labels, const float* lse, const float* valid,
                                     const float* weights, const float* sums, const float* scale, void* dlogits,
                                     int64_t T, int V, int dtype, ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(T >= 0 && T <= 0x7fffffffLL && V > 0, ATS_ERR_INVALID_ARG, "ats_cross_entropy_bwd: T=%lld V=%d", (long long)T, V);
    ATS_REQUIRE(dtype == ATS_F32 || dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "ats_cross_entropy_bwd: dtype tag %d", dtype);
    if (T == 0) return ATS_OK;
    ATS_REQUIRE(logits && labels && lse && valid && sums && scale && dlogits, ATS_ERR_INVALID_ARG,
                "ats_cross_entropy_bwd: null pointer");
    // the same alignment on both sides: one split into head, vectors and tail serves both
    const bool vec = ((reinterpret_cast<uintptr_t>(logits) ^ reinterpret_cast<uintptr_t>(dlogits)) & 15u) == 0;
    if (dtype == ATS_F32)
        hipLaunchKernelGGL((cross_entropy_bwd_kernel<float>), dim3((unsigned)T), dim3(256), 0, as_stream(stream),
                           static_cast<const float*>(logits), labels, lse, valid, weights, sums, scale,
                           static_cast<float*>(dlogits), V, vec);
    else
        hipLaunchKernelGGL((cross_entropy_bwd_kernel<bf16_t>), dim3((unsigned)T), dim3(256), 0, as_stream(stream),
                           static_cast<const bf16_t*>(logits), labels, lse, valid, weights, sums, scale,
                           static_cast<bf16_t*>(dlogits), V, vec);
    ATS_CHECK_LAUNCH("ats_cross_entropy_bwd");
    return ATS_OK;
}

extern "C" int ats_grad_clip_chunk_elems(void) { return ats::kClipChunk; }

extern "C" int ats_grad_norm_clip(void* const* grad_ptrs, const int64_t* sizes, const int32_t* chunk_start,
                                  int n_tensors, int n_chunks, int dtype, const float* extra_sumsq, float* partial,
                                  float* norm_out, float max_norm, int do_clip, ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(n_tensors >= 0 && n_chunks >= 0, ATS_ERR_INVALID_ARG, "ats_grad_norm_clip: n_tensors=%d n_chunks=%d",
                n_tensors, n_chunks);
    ATS_REQUIRE(dtype == ATS_F32 || dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "ats_grad_norm_clip: dtype tag %d", dtype);
    ATS_REQUIRE(norm_out && (n_chunks == 0 || (grad_ptrs && sizes && chunk_start && partial)), ATS_ERR_INVALID_ARG,
                "ats_grad_norm_clip: null pointer");
    hipStream_t s = as_stream(stream);
    if (do_clip == 2) {   // scale only: norm_out already holds the norm over all groups
        if (n_chunks > 0) {
            if (dtype == ATS_F32)
                hipLaunchKernelGGL((grad_scale_kernel<float>), dim3((unsigned)n_chunks), dim3(256), 0, s, grad_ptrs, sizes,
                                   chunk_start, n_tensors, norm_out, max_norm);
            else
                hipLaunchKernelGGL((grad_scale_kernel<bf16_t>), dim3((unsigned)n_chunks), dim3(256), 0, s, grad_ptrs, sizes,
                                   chunk_start, n_tensors, norm_out, max_norm);
        }
        ATS_CHECK_LAUNCH("ats_grad_norm_clip");
        return ATS_OK;
    }
    if (n_chunks > 0) {
        if (dtype == ATS_F32)
            hipLaunchKernelGGL((grad_sumsq_kernel<float>), dim3((unsigned)n_chunks), dim3(256), 0, s,
                               reinterpret_cast<const void* const*>(grad_ptrs), sizes, chunk_start, n_tensors, partial);
        else
            hipLaunchKernelGGL((grad_sumsq_kernel<bf16_t>), dim3((unsigned)n_chunks), dim3(256), 0, s,
                               reinterpret_cast<const void* const*>(grad_ptrs), sizes, chunk_start, n_tensors, partial);
    }
    hipLaunchKernelGGL(grad_norm_finish_kernel, dim3(1), dim3(256), 0, s, partial, n_chunks, extra_sumsq, norm_out);
    if (do_clip == 1 && n_chunks > 0) {
        if (dtype == ATS_F32)
            hipLaunchKernelGGL((grad_scale_kernel<float>), dim3((unsigned)n_chunks), dim3(256), 0, s, grad_ptrs, sizes,
                               chunk_start, n_tensors, norm_out, max_norm);
        else
            hipLaunchKernelGGL((grad_scale_kernel<bf16_t>), dim3((unsigned)n_chunks), dim3(256), 0, s, grad_ptrs, sizes,
                               chunk_start, n_tensors, norm_out, max_norm);
    }
    ATS_CHECK_LAUNCH("ats_grad_norm_clip");
    return ATS_OK;
}
